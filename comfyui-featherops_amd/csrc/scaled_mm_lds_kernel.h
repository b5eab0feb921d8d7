// Large-M fp16 x fp8 GEMM on gfx950: LDS-DMA multi-stage pipeline (the kernel template and its
// launcher; scaled_mm_lds.hip and scaled_mm_mid.hip instantiate its tiles).
//
// Same contract as the reference kernel (kernel/hip/hip_kernel.cu:133-420:
// fp32 accumulation, scale on the accumulator, rounding to the output type,
// bias added in the output type) for K % 64 == 0, and with kTail for any K % 16.
//
// How it works:
//   * global -> LDS copies use gfx950's global_load_lds_dwordx4: each wave
//     instruction moves 64 x 16 bytes straight into a contiguous 1 KB of LDS,
//     with no VGPR staging and no ds_write. Addresses are a wave-uniform SGPR
//     base (advanced per stage with scalar adds) plus a fixed 32-bit per-lane
//     offset;
//   * A rows are 128 bytes in LDS; chunk c of row r is stored at c ^ swz(r).
//     The swizzle is applied on the global side: the lane that fills LDS chunk
//     p of row r fetches logical chunk p ^ swz(r);
//   * three LDS stage buffers with two stages of copies in flight behind the
//     one being multiplied (the split-K tiles: four or five buffers, all but
//     one in flight); each barrier is preceded by an explicit vmcnt
//     wait that leaves the younger stages' copies in flight;
//   * K groups (the split-K tiles): those tiles have one workgroup per CU, and
//     with four waves, one per SIMD, nothing ran while a wave waited at a stage
//     barrier or for its operands (M=2048 N=2048 on 64-row tiles: copies alone
//     0.28 us a stage pair, MFMAs and operand reads alone 0.49, both 0.48-0.53).
//     Two groups of four waves now share a stage of 128 K, each multiplying its
//     own 64 for the whole tile, so that every SIMD has two waves and there is one
//     barrier per 128 K; the groups' sums meet once, through LDS, after the
//     last stage. One group on a five- or six-stage ring -> two, back to back with
//     the weights in the MALL: M=154 N=10240 K=4096 21.3 -> 17.3 us, M=333 N=K=3072
//     15.7 -> 13.2, M=256 N=K=3072 11.7 -> 9.9, M=512 N=3072 K=12288 47.7 -> 42.4,
//     M=128 N=K=5120 14.5 -> 13.3, M=77 N=K=4096 11.5 -> 9.6, M=64 N=13824 K=5120
//     22.1 -> 20.6. With the weights from HBM the gain is smaller or none: M=600
//     N=1024 K=3072 11.3 -> 9.6, M=260 N=K=3072 11.9 -> 11.1, M=130 N=7168 K=4096 17.7 ->
//     17.0, but M=154 N=10240 K=4096 20.5 -> 21.4 and M=128 N=7296 K=4416 17.0 -> 17.4.
//     An unsplit K up to 1024 stays on one group (launch_short). Four groups on
//     64 x 64 (16 waves): 10.6 at M=256 N=K=3072 in the MALL; 2 x 4 waves instead of two
//     groups: 64 x 128 18.1 at M=154, and more LDS reads per MFMA;
//   * per stage, the K halves are processed one after the other (all M
//     repeats of K half 0, then of K half 1), so only half of the widened B
//     operands are live at a time;
//   * default schedule: the barrier sits early in each stage's second half,
//     after which the next stage's operands can be read while the current
//     stage's remaining MFMAs run (measured on the M=32768 K=5120 N=13824
//     shape: ~5% faster than barrier-at-the-top, which is kept as
//     FEATHEROPS_LDS_PIPE=0). The source asks for A one K half ahead and the
//     copies spread between MFMA groups; the compiler's scheduler keeps the
//     kernel at 255 VGPRs by reading A about one M repeat ahead instead and
//     issues each stage's copies together before the barrier (pinning the
//     source order with scheduling barriers spills, and the other scheduler
//     strategies measured 0-2.5% slower);
//   * rows past M / columns past N are clamped to the last valid row/column
//     (their results are computed and dropped), so every copy is in bounds;
//   * optional rank-R update in the epilogue (kLora, the unmerged LoRA side
//     path of the reference's comfy_feather/lora.py:4-35): after the weight
//     scale, acc += T(M x R) . U(N x R)^T on the fp16 or bf16 MFMA, before
//     the rounding to the output type; the tile's rows of T and U go through
//     the free stage buffers 64 ranks at a time (LDS-DMA, one round trip per
//     64 ranks). The separate pass that would re-read and re-write C
//     disappears.
#pragma once

#include <type_traits>

#include "feather_common.h"
#include "lds_dma.h"
#include "scaled_mm_dispatch.h"

namespace feather {
namespace {

// f(std::integral_constant<int, i>{}) for i = 0 .. N-1, in order
template <int N, int I = 0, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<N, I + 1>(f);
    }
}

constexpr int kBK = 64;


// kLora: 0 = none, 1 = fp16 factors, 2 = bf16 factors (T is M x R, U is N x R,
// both row-major with R % 32 == 0 and 16-byte aligned rows), 3 = either, by
// lora_flags: bit 0 = bf16 factors, bit 1 = the term is rounded to the factors'
// type and to the output type and added to the finished result in the output
// type (a separate pass's arithmetic) instead of joining the fp32 accumulator
// kGroups: 1, or 2 = two groups of WAVES_M x WAVES_N waves share a stage of 2 x
// 64 K, each multiplying its own 64 of it for the whole tile (see the K groups
// paragraph in the file header). kTail: K need not be a multiple of the stage
template <int BM, int BN, int WAVES_M, int WAVES_N, int kPipe, bool kBf16, bool kE4m3, int kLora, int kStages,
          int kGroups, bool kTail>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N * kGroups) void scaled_mm_lds_kernel(
    const uint16_t* __restrict__ A, const uint8_t* __restrict__ Bp, const float* __restrict__ scale,
    const uint16_t* __restrict__ bias, uint16_t* __restrict__ C, int M, int N, int K, int has_scale, int has_bias,
    int tiles_m, int tiles_n, int group_m, int ksplit, float* __restrict__ partials, uint32_t* __restrict__ counters,
    const uint16_t* __restrict__ lora_t, const uint16_t* __restrict__ lora_u, int lora_rank, int lora_flags,
    int c_nontemporal) {
    constexpr int kGroupWaves = WAVES_M * WAVES_N;
    constexpr int kWaves = kGroupWaves * kGroups;
    constexpr int WTM = BM / WAVES_M;
    constexpr int WTN = BN / WAVES_N;
    constexpr int RM = WTM / 16;
    constexpr int RN = WTN / 16;
    static_assert(WTM % 16 == 0 && WTN % 16 == 0, "wave tile must be a multiple of 16");
    constexpr int kSK = kBK * kGroups;  // K per stage
    // the 32-bit copy offsets a_off and b_off below (see kMaxK, kMaxN)
    static_assert(int64_t{BM} * kMaxK * 2 <= int64_t{1} << 31 && int64_t{kSK / 16} * kMaxN * 16 <= int64_t{1} << 32,
                  "copy offsets fit 32 bits");
    constexpr int kASub = BM * kBK * 2;  // one group's share of a stage
    constexpr int kBSub = BN * kBK;
    constexpr int kAStage = kASub * kGroups;
    constexpr int kBStage = kBSub * kGroups;
    constexpr int kStage = kAStage + kBStage;
    constexpr int kAInst = kAStage / 1024;  // 1 KB wave copies per stage
    constexpr int kBInst = kBStage / 1024;
    // A and B copies are rounded up to a whole number per wave; the surplus
    // slots repeat the last copy (same bytes to the same LDS address), so every
    // wave issues, and waits for, the same number of copies per stage.
    constexpr int kAPerWave = (kAInst + kWaves - 1) / kWaves;
    constexpr int kBPerWave = (kBInst + kWaves - 1) / kWaves;
    constexpr int kLoadsPerStage = kAPerWave + kBPerWave;
    static_assert(BN % 64 == 0, "a B copy must stay inside one K group");
    // One LDS object per stage buffer for the first three (the main loop is
    // unrolled by the stage count); deeper rings add buffers behind them.
    static_assert(kStages == 3 || (kPipe == 1 && kStages >= 4 && kStages <= 8), "stage ring depth");
    __shared__ __attribute__((aligned(1024))) uint8_t sbuf0[kStage];
    __shared__ __attribute__((aligned(1024))) uint8_t sbuf1[kStage];
    __shared__ __attribute__((aligned(1024))) uint8_t sbuf2[kStage];
    __shared__ __attribute__((aligned(1024))) uint8_t sbufx[kStages > 3 ? (kStages - 3) * kStage : 1024];

    // ---- tile index: XCD-contiguous grouped raster; the K splits of a tile
    // are consecutive in that order (so mostly on one XCD) ----
    const int total = tiles_m * tiles_n * ksplit;
    const int pid = blockIdx.x;
    const int xcd = pid % kNumXcd;
    const int per = total / kNumXcd;
    const int rem = total % kNumXcd;
    const int vlin = xcd * per + (xcd < rem ? xcd : rem) + pid / kNumXcd;
    const int lin = vlin / ksplit;
    const int q = vlin - lin * ksplit;
    const int group_size = group_m * tiles_n;
    const int gid = lin / group_size;
    const int first_m = gid * group_m;
    const int gm = (tiles_m - first_m) < group_m ? (tiles_m - first_m) : group_m;
    const int in_group = lin - gid * group_size;
    const int tm = first_m + in_group % gm;
    const int tn = in_group / gm;
    const int m0 = tm * BM;
    const int n0 = tn * BN;

    // The scale, loaded before anything else by a vector load with no branch
    // around it (an absent scale reads A's first bytes and is not used) and
    // selected in the epilogue: it is in long before the epilogue needs it
    // (read there, the scalar load's round trip came before the staging), and
    // as the oldest load it never holds up the stage waits below, which leave
    // only younger copies in flight.
    const uint32_t scale_raw = __builtin_amdgcn_raw_buffer_load_b32(
        __builtin_amdgcn_make_buffer_rsrc(
            const_cast<void*>(has_scale ? static_cast<const void*>(scale) : static_cast<const void*>(A)), 0, 4,
            0x00020000),
        0, 0, 0);
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int group = wave / kGroupWaves;
    const int wave_m = wave % WAVES_M;
    const int wave_n = (wave / WAVES_M) % WAVES_N;
    const int lr = lane & 15;
    const int lg = lane >> 4;
    // K split q covers stages [kt0, kt0 + nk); the host picks ksplit so none is empty
    const int nk_all = (K + kSK - 1) / kSK;
    const int per_split = (nk_all + ksplit - 1) / ksplit;
    const int kt0 = q * per_split;
    const int nk = (nk_all - kt0) < per_split ? (nk_all - kt0) : per_split;

    // K % kSK != 0: the last stage is the window [K - kSK, K) instead of one that
    // would reach past K, so its copies need no bounds; the K it shares with the
    // stage before is zeroed in LDS, in both operands, once it has landed
    // (zero_tail). K < kSK: the one stage starts at 0, chunks past K copy chunk 0
    // and are zeroed.
    int k_last = (kt0 + nk - 1) * kSK;
    if constexpr (kTail)
        if (k_last >= K - kSK) k_last = K > kSK ? K - kSK : 0;
    const bool tail = kTail && kt0 + nk == nk_all && K % kSK != 0;

    // ---- per-lane copy offsets (fixed), per-stage SGPR bases ----
    // A copy a of a stage (BM / 8 per 64 K) fills 8 rows of 64 K.
    constexpr int kAGroupInst = BM / 8;
    auto a_copy = [&](int j) { return (j * kWaves + wave) < kAInst ? (j * kWaves + wave) : kAInst - 1; };
    // this lane's row of A copy j, and the byte offset of its 16-byte chunk in the stage's K
    auto a_row = [&](int j) { return (a_copy(j) % kAGroupInst) * 8 + (lane >> 3); };
    auto a_kbyte = [&](int j) { return (a_copy(j) / kAGroupInst) * (kBK * 2) + (((lane & 7) ^ swz(a_row(j))) << 4); };
    uint32_t a_off[kAPerWave];
#pragma unroll
    for (int j = 0; j < kAPerWave; ++j) {
        const int row = a_row(j);
        const int kb = !kTail || a_kbyte(j) < 2 * K ? a_kbyte(j) : 0;
        const int lrow = (m0 + row < M ? m0 + row : M - 1) - m0;
        a_off[j] = static_cast<uint32_t>(lrow * K * 2 + kb);
    }
    // B copy j covers chunks [base, base+64) of the (4 * kGroups x BN) stage, base = b_copy(j) * 64.
    auto b_copy = [&](int j) { return (j * kWaves + wave) < kBInst ? (j * kWaves + wave) : kBInst - 1; };
    uint32_t b_off[kBPerWave];
#pragma unroll
    for (int j = 0; j < kBPerWave; ++j) {
        const int chunk = b_copy(j) * 64 + lane;
        const int kb = !kTail || (chunk / BN) * 16 < K ? chunk / BN : 0;
        const int lcol = (n0 + chunk % BN < N ? n0 + chunk % BN : N - 1) - n0;
        b_off[j] = (static_cast<uint32_t>(kb) * static_cast<uint32_t>(N) + static_cast<uint32_t>(lcol)) * 16u;
    }
    const uint8_t* a_base = reinterpret_cast<const uint8_t*>(A) + static_cast<int64_t>(m0) * K * 2;
    const uint8_t* b_base = Bp + static_cast<int64_t>(n0) * 16;
    // first K of stage kt; past the end (deep rings), and for a shifted last
    // stage, that of the last stage. kInside: kt is known to lie before the last
    auto stage_k = [&](int kt, auto inside) -> int {
        const int k = (kt0 + kt) * kSK;
        if constexpr (decltype(inside)::value || (!kTail && kStages == 3)) return k;
        else return k < k_last ? k : k_last;
    };

    auto stage_buf = [&](auto tag) -> uint8_t* {
        constexpr int b = decltype(tag)::value;
        if constexpr (b == 0) return sbuf0;
        else if constexpr (b == 1) return sbuf1;
        else if constexpr (b == 2) return sbuf2;
        else return sbufx + (b - 3) * kStage;
    };
    // LDS byte address of stage buffer `tag` (a constant)
    auto stage_lds = [&](auto tag) -> uint32_t { return lds_addr_of(stage_buf(tag)); };
    // copy i (A copies first, then B copies) of the stage starting at K = k into
    // buffer `tag` (16 K of the weights are N x 16 bytes)
    auto issue_one = [&](auto tag, int k, int i) {
        const uint32_t la = stage_lds(tag);
        if (i < kAPerWave) {
            dma16_lds(a_base + k * 2, a_off[i], la + a_copy(i) * 1024);
        } else {
            const int j = i - kAPerWave;
            dma16_lds(b_base + static_cast<int64_t>(k) * N, b_off[j], la + kAStage + b_copy(j) * 1024);
        }
    };
    auto issue_stage = [&](auto tag, int k) {
#pragma unroll
        for (int i = 0; i < kLoadsPerStage; ++i) issue_one(tag, k, i);
    };
    // Zeroes, in the landed last stage in buffer `tag`, the chunks this wave copied
    // itself whose K is not the stage's own (a chunk that several waves copy is
    // zeroed by each after its own copy has landed, so zero is the last write).
    auto zero_tail = [&](auto tag) {
        const int lo = K > kSK ? nk_all * kSK - K : 0, hi = K > kSK ? kSK : K;
        const uint32_t la = stage_lds(tag);
        using v4 = uint32_t __attribute__((ext_vector_type(4)));
        auto clear = [&](uint32_t addr, int kk) {
            if (kk < lo || kk >= hi)
                *reinterpret_cast<__attribute__((address_space(3))) v4*>(static_cast<uintptr_t>(addr)) = v4{0u, 0u, 0u, 0u};
        };
#pragma unroll
        for (int j = 0; j < kAPerWave; ++j) clear(la + a_copy(j) * 1024 + lane * 16, a_kbyte(j) >> 1);
#pragma unroll
        for (int j = 0; j < kBPerWave; ++j)
            clear(la + kAStage + b_copy(j) * 1024 + lane * 16, ((b_copy(j) * 64 + lane) / BN) * 16);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    };
    // LDS byte offset of this lane's A operand for M repeat rm, K half kh
    auto a_lds = [&](int rm, int kh) -> int {
        const int row = wave_m * WTM + rm * 16 + lr;
        return row * 128 + (((2 * lg + kh) ^ swz(row)) << 4);
    };
    // operand reads as LDS byte addresses: a constant per buffer (and M / N
    // repeat) plus one per-lane offset, so the constants can sit in the
    // ds_read offset field instead of in extra address registers
    auto lds_ld16 = [](uint32_t addr) -> uint4 {
        using v4 = uint32_t __attribute__((ext_vector_type(4)));
        const v4 v = *reinterpret_cast<const __attribute__((address_space(3))) v4*>(static_cast<uintptr_t>(addr));
        return make_uint4(v.x, v.y, v.z, v.w);
    };
    const uint32_t b_lane = static_cast<uint32_t>((lg * BN + wave_n * WTN + lr) * 16 + group * kBSub);
    const uint32_t a_lane0 = static_cast<uint32_t>(a_lds(0, 0) + group * kASub);
    const uint32_t a_lane1 = static_cast<uint32_t>(a_lds(0, 1) + group * kASub);
    auto read_b = [&](auto cur, uint4 (&braw)[RN]) {
        const uint32_t sb = stage_lds(cur) + kAStage + b_lane;
#pragma unroll
        for (int rn = 0; rn < RN; ++rn) braw[rn] = lds_ld16(sb + rn * 256);
    };

    f32x4 acc[RM][RN];
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int j = 0; j < RN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    using S2 = std::integral_constant<int, 2>;
    using Near = std::false_type;  // stage_k: the stage may be the last one

    // A fragments of one K half of a stage, for every M repeat
    // (the A swizzle depends on row & 15 only, so M repeat rm adds rm * 16 rows)
    auto read_a = [&](auto tag, int kh, uint4 (&dst)[RM]) {
        const uint32_t sa = stage_lds(tag) + (kh ? a_lane1 : a_lane0);
#pragma unroll
        for (int rm = 0; rm < RM; ++rm) dst[rm] = lds_ld16(sa + rm * 16 * 128);
    };
    // MFMAs of one K half: widen this half of the B operands, then run every
    // M repeat; `hook(rm)` runs before the MFMAs of repeat rm. The widened
    // weights are the MFMA's first operand and the activations its second, so
    // each 16x16 result is C^T: lane (lr, lg) element i is C[row lr][col
    // 4*lg + i] of the tile. Measured 1.8% faster than the other operand order
    // on M=32768 N=13824 K=5120 (the kernel is power-bound with random data).
    // Changing the activation operand costs more than changing the weight
    // operand (an e5m2 byte widens to an fp16 with a zero low byte): running the M
    // repeats innermost measured 4% slower.
    // Pinned schedule (default schedule, wave tiles of at least 64 x 64):
    // each weight column is widened just before it is first needed, in
    // program order with the MFMAs (both inline asm, so neither moves), instead
    // of a whole K half's columns in one burst ahead of its first MFMA; the
    // MFMAs run in a serpentine over the columns, and the next K half's first
    // two columns are widened during this half's last repeat once they are
    // free. Medians of alternating runs on MI355X, the same bits: M=32768
    // N=13824 K=5120 (256 x 256, 4 x 2 waves) 3.268 vs 3.315 ms, 8192^3 0.765
    // vs 0.774 ms; M=4096 N=3072 K=3072 (128 x 384) 56.2 vs 57.8 us, K=12288
    // 209.8 vs 213.7 us (256 x 192 on 4 x 2 waves: 210.3 vs 217.1 us on 2 x 4);
    // M=2048 N=K=4096: 128 x 256 52.0 vs 52.8 us, 256 x 128 53.3 vs 54.9 us,
    // 128 x 128 62.9 vs 63.6 us; e4m3fn weights at M=32768 N=13824 K=5120
    // 3.225 vs 3.251 ms (4 x 2 pinned vs 2 x 4 compiler-scheduled). Ordering
    // rules the asm keeps by construction (the compiler's hazard tracking does
    // not see inside asm): a widened column is written at least two MFMAs
    // before an MFMA reads it (the register of one an MFMA has read may be
    // rewritten right after it, as the compiler's own code for builtin MFMAs
    // does), the MFMAs accumulate in place with nothing else touching the
    // accumulators in the loop, and other instructions read the accumulators
    // only after the wait states that follow the main loop (all checked on the
    // compiled code by tests/test_pinned_codegen.py).
    constexpr bool kPinned = kPipe == 1 && RM % 2 == 0 && RM >= 4 && RN >= 4;
    // widen_fp8x8's instructions as asm (e5m2: byte shuffles; e4m3fn: the
    // hardware fp8 -> fp16 conversion with scale 1, low then high word)
    auto widen_pinned = [](uint32_t lo, uint32_t hi) -> half8_t {
        uint32_t w0, w1, w2, w3;
        if constexpr (!kE4m3) {
            asm volatile(
                "v_perm_b32 %0, 0, %4, %6\n\t"
                "v_perm_b32 %1, 0, %4, %7\n\t"
                "v_perm_b32 %2, 0, %5, %6\n\t"
                "v_perm_b32 %3, 0, %5, %7"
                : "=&v"(w0), "=&v"(w1), "=&v"(w2), "=&v"(w3)
                : "v"(lo), "v"(hi), "s"(0x010c000cu), "s"(0x030c020cu));
        } else {
            asm volatile(
                "v_cvt_scalef32_pk_f16_fp8 %0, %4, 1.0\n\t"
                "v_cvt_scalef32_pk_f16_fp8 %1, %4, 1.0 op_sel:[1,0,0]\n\t"
                "v_cvt_scalef32_pk_f16_fp8 %2, %5, 1.0\n\t"
                "v_cvt_scalef32_pk_f16_fp8 %3, %5, 1.0 op_sel:[1,0,0]"
                : "=&v"(w0), "=&v"(w1), "=&v"(w2), "=&v"(w3)
                : "v"(lo), "v"(hi));
        }
        return __builtin_bit_cast(half8_t, make_uint4(w0, w1, w2, w3));
    };
    half8_t bqp[RN];  // pinned schedule: the current K half's widened columns
    auto mm_half = [&](int kh, const uint4 (&araw)[RM], const uint4 (&braw)[RN], auto hook, bool pre = false) {
        if constexpr (kPinned) {
            // MFMA j of repeat rm uses column col(kh, rm, j): forward or
            // reversed by repeat, K half 1 starting reversed, so the columns the
            // next half needs first are the ones this half's last repeat uses
            // first. pre: widen the next half's first two columns here (braw
            // holds the next stage's weights by then when kh == 1).
            auto col = [](int h, int rm, int j) { return (((rm & 1) ^ h) != 0) ? RN - 1 - j : j; };
            auto wd = [&](int rn, int h) {
                bqp[rn] = h == 0 ? widen_pinned(braw[rn].x, braw[rn].y) : widen_pinned(braw[rn].z, braw[rn].w);
            };
            constexpr int kPre = RN >= 6 ? RN / 2 : 2;
#pragma unroll
            for (int rm = 0; rm < RM; ++rm) {
                hook(rm);
                const half8_t a = a_frag<false>(araw[rm]);
#pragma unroll
                for (int j = 0; j < RN; ++j) {
                    if (rm == 0 && j + 2 < RN) wd(col(kh, 0, j + 2), kh);
                    if (rm == RM - 1 && pre && (j == kPre || j == kPre + 1)) wd(col(kh ^ 1, 0, j - kPre), kh ^ 1);
                    const int rn = col(kh, rm, j);
                    f32x4 t = acc[rm][rn];
                    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(t) : "v"(bqp[rn]), "v"(a));
                    acc[rm][rn] = t;
                }
            }
            return;
        }
        half8_t bq[RN];
#pragma unroll
        for (int rn = 0; rn < RN; ++rn)
            bq[rn] = kh == 0 ? widen_fp8x8<kE4m3>(braw[rn].x, braw[rn].y) : widen_fp8x8<kE4m3>(braw[rn].z, braw[rn].w);
#pragma unroll
        for (int rm = 0; rm < RM; ++rm) {
            hook(rm);
            const half8_t a = a_frag<false>(araw[rm]);
#pragma unroll
            for (int j = 0; j < RN; ++j) {
                // serpentine over the N repeats: consecutive MFMAs change only
                // one operand (0.6-1.5% faster on M=32768 N=13824 K=5120 than
                // restarting at rn = 0; again a power effect)
                const int rn = (rm & 1) ? RN - 1 - j : j;
                acc[rm][rn] = mfma16x16x32(bq[rn], a, acc[rm][rn]);
            }
        }
    };

    if constexpr (kPipe == 1) {
        // Operands one K half ahead (as written; see the file header for what
        // the scheduler makes of it). Register set araw[kh] holds the A
        // fragments of K half kh of the current stage: the second half's are
        // requested at the start of the first half's MFMAs. Stage kt + 2's
        // copies are placed between the first half's M repeats. Early in the
        // second half -- once every wave has all of stage kt in registers --
        // a barrier publishes stage kt + 1 (its copies were waited for just
        // before) and frees stage kt's buffer, and stage kt + 1's first-half
        // operands are requested while the remaining repeats run.
        constexpr int kBarrierRm = RM / 4;
        uint4 araw[2][RM];
        uint4 braw[RN];
        // Deeper rings (kStages > 3) always keep kStages - 1 stages of copies
        // issued: a stage past the end copies stage nk - 1 again into its
        // (never read) buffer, so every wait count is a constant and no
        // branch surrounds a copy; the main loop waits for those copies
        // before the epilogue reuses the buffers.
        issue_stage(S0{}, stage_k(0, Near{}));
        if constexpr (kStages == 3) {
            if (nk > 1) {
                issue_stage(S1{}, stage_k(1, Near{}));
                wait_vmcnt<kLoadsPerStage>();
            } else {
                wait_vmcnt<0>();
            }
        } else {
            static_for<kStages - 2>([&](auto i) {
                constexpr int st = decltype(i)::value + 1;
                issue_stage(std::integral_constant<int, st>{}, stage_k(st, Near{}));
            });
            wait_vmcnt<(kStages - 2) * kLoadsPerStage>();
        }
        if constexpr (kTail)
            if (tail && nk == 1) zero_tail(S0{});
        stage_barrier();
        read_b(S0{}, braw);
        read_a(S0{}, 0, araw[0]);
        if constexpr (kPinned) {
            // K half 0 of stage 0 starts forward: columns 0 and 1
            static_assert(RM / 4 >= 1, "the next stage's weights arrive after repeat 0");
            bqp[0] = widen_pinned(braw[0].x, braw[0].y);
            bqp[1] = widen_pinned(braw[1].x, braw[1].y);
        }
        // kFull (three-stage ring): stages kt + 1 and kt + 2 exist, and neither is
        // a shifted last stage (no bounds checks, so the steady-state loop body
        // has no branches around the copies; a checked copy of the loop runs the
        // last three to six stages). Deeper rings run every stage unchecked,
        // the copies of stages past the end clamped to the last one.
        auto run_stage = [&](auto cur, auto full, int kt) {
            constexpr int c = decltype(cur)::value;
            constexpr bool kFull = decltype(full)::value;
            using Next = std::integral_constant<int, (c + 1) % kStages>;
            // stage kt + kStages - 1's buffer (stage kt - 1's, freed by its barrier)
            using Free = std::integral_constant<int, (c + kStages - 1) % kStages>;
            const bool has2 = kStages > 3 || kFull || kt + 2 < nk;
            const bool has1 = kStages > 3 || kFull || kt + 1 < nk;
            const int k_free = stage_k(kt + kStages - 1, std::bool_constant<kStages == 3 && kFull>{});
            mm_half(0, araw[0], braw, [&](int rm) {
                if (rm == 0) read_a(cur, 1, araw[1]);
#pragma unroll
                for (int i = 0; i < kLoadsPerStage; ++i)
                    if (rm == (i * RM) / kLoadsPerStage && has2) issue_one(Free{}, k_free, i);
            }, true);
            // mm_half widens braw before the first hook, so the hook may
            // overwrite braw with the next stage's operands
            mm_half(1, araw[1], braw, [&](int rm) {
                if (rm == kBarrierRm && has1) {
                    // this wave's reads of stage kt have returned, stage kt + 1 has landed
                    if (has2) wait_vmcnt_lgkm0<(kStages - 2) * kLoadsPerStage>();
                    else wait_vmcnt_lgkm0<0>();
                    if constexpr (kTail && (kStages > 3 || !kFull))
                        if (tail && kt + 2 == nk) zero_tail(Next{});
                    stage_barrier();
                    read_b(Next{}, braw);
                    read_a(Next{}, 0, araw[0]);
                }
            }, has1);
        };
        using Full = std::true_type;
        using Tail = std::false_type;
        int kt = 0;
        if constexpr (kStages == 3) {
            for (; kt + (tail ? 6 : 5) <= nk; kt += 3) {
                run_stage(S0{}, Full{}, kt);
                run_stage(S1{}, Full{}, kt + 1);
                run_stage(S2{}, Full{}, kt + 2);
            }
            for (; kt < nk; kt += 3) {
                run_stage(S0{}, Tail{}, kt);
                if (kt + 1 < nk) run_stage(S1{}, Tail{}, kt + 1);
                if (kt + 2 < nk) run_stage(S2{}, Tail{}, kt + 2);
            }
        } else {
            for (; kt + kStages <= nk; kt += kStages)
                static_for<kStages>([&](auto c) { run_stage(c, Full{}, kt + decltype(c)::value); });
            static_for<kStages>([&](auto c) {
                if (kt + decltype(c)::value < nk) run_stage(c, Full{}, kt + decltype(c)::value);
            });
            wait_vmcnt<0>();  // the repeated copies past the end
        }
    } else {
        // Plain schedule: at the top of stage kt wait for its copies (issued
        // two stages earlier), barrier, issue stage kt + 2's copies into the
        // buffer stage kt - 1 used, then read and multiply both K halves.
        static_assert(!kTail, "the plain schedule has no shifted last stage");
        auto no_hook = [](int) {};
        auto run_stage = [&](auto cur, int kt) {
            constexpr int c = decltype(cur)::value;
            using Free = std::integral_constant<int, (c + 2) % 3>;
            if (kt + 1 < nk) wait_vmcnt<kLoadsPerStage>();
            else wait_vmcnt<0>();
            stage_barrier();
            if (kt + 2 < nk) issue_stage(Free{}, stage_k(kt + 2, Near{}));
            uint4 braw[RN];
            read_b(cur, braw);
            uint4 araw[RM];
            read_a(cur, 0, araw);
            mm_half(0, araw, braw, no_hook);
            read_a(cur, 1, araw);
            mm_half(1, araw, braw, no_hook);
        };
        issue_stage(S0{}, stage_k(0, Near{}));
        if (nk > 1) issue_stage(S1{}, stage_k(1, Near{}));
        for (int kt = 0; kt < nk; kt += 3) {
            run_stage(S0{}, kt);
            if (kt + 1 < nk) run_stage(S1{}, kt + 1);
            if (kt + 2 < nk) run_stage(S2{}, kt + 2);
        }
    }

    // pinned schedule: wait states between the last asm MFMA and any other
    // instruction that reads its accumulator
    if constexpr (kPinned) asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
    // the scale into a scalar register here, where the main loop has already
    // waited for every load (the memory clobber keeps the epilogue's bias load
    // from being issued before this wait, so the bias still lands behind the
    // staging writes)
    uint32_t scale_s;
    asm volatile("v_readfirstlane_b32 %0, %1" : "=s"(scale_s) : "v"(scale_raw) : "memory");
    float s = has_scale ? __uint_as_float(scale_s) : 1.0f;
    // ---- K groups: the two groups hold partial sums of the same tile. Each keeps
    // half of its M repeats (group 0 the first half), writes the other half to
    // the (now free) stage buffers for the other group, and adds what that one
    // wrote; from here on a wave's results are acc[0 .. RME), rows from erow0. ----
    constexpr int RME = RM / kGroups;
    const int erow0 = wave_m * WTM + group * (RME * 16);
    if constexpr (kGroups == 2) {
        constexpr int kPart = RME * RN * 1024;
        static_assert(RM % 2 == 0 && kGroupWaves * kPart <= kStage, "one group's half must fit a stage buffer");
        const int w = wave % kGroupWaves;
        uint8_t* const mine = (group ? sbuf1 : sbuf0) + w * kPart + lane * 16;
        const uint8_t* const theirs = (group ? sbuf0 : sbuf1) + w * kPart + lane * 16;
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wave's last operand reads are done
        stage_barrier();
#pragma unroll
        for (int rm = 0; rm < RME; ++rm)
#pragma unroll
            for (int rn = 0; rn < RN; ++rn) {
                const f32x4 give = group ? acc[rm][rn] : acc[rm + RME][rn];
                if (group) acc[rm][rn] = acc[rm + RME][rn];
                *reinterpret_cast<f32x4*>(mine + (rm * RN + rn) * 1024) = give;
            }
        __builtin_amdgcn_s_waitcnt(0xC07F);
        stage_barrier();
#pragma unroll
        for (int rm = 0; rm < RME; ++rm)
#pragma unroll
            for (int rn = 0; rn < RN; ++rn)
                acc[rm][rn] += *reinterpret_cast<const f32x4*>(theirs + (rm * RN + rn) * 1024);
    }
    // (K split: only the tiles with two K groups are ever launched with ksplit > 1)
    if constexpr (kGroups == 2) if (ksplit > 1) {
        // ---- K split: each workgroup writes its fp32 accumulators to the
        // workspace in fragment order (lane-contiguous 16-byte pieces) and
        // bumps the tile's arrival counter; the workgroup that arrives last
        // adds the ksplit partials in split order (deterministic; its own from
        // its registers), then runs the normal epilogue and re-zeroes the counter.
        // Ordering: the partials are only ever written and read with agent-scope
        // (sc1) accesses -- the instructions the AMDGPU memory model uses for
        // relaxed agent-scope atomic stores and loads on gfx942/gfx950 -- so
        // they are coherent across XCDs without any L2 write-back or
        // invalidate. A store is acknowledged (vmcnt) only once it is visible
        // at agent scope; every wave waits for that before the barrier, and
        // the arrival RMW is issued after the barrier, so it follows every
        // partial of this workgroup. The last arrival's loads are issued after
        // the RMW has returned (they depend on last_flag through LDS and a
        // barrier) and read the coherence point directly. An agent-scope
        // release/acquire pair instead costs an L2 write-back and invalidate
        // per workgroup (measured: M=64 N=13824 K=5120 25 -> 38 us).
        constexpr int kTileBytes = BM * BN * 4;
        const __amdgpu_buffer_rsrc_t prs = __builtin_amdgcn_make_buffer_rsrc(
            partials + static_cast<int64_t>(lin) * ksplit * (kTileBytes / 4), 0, ksplit * kTileBytes, 0x00020000);
        auto frag_off = [&](int rm, int rn) { return (((wave * RME + rm) * RN + rn) * 64 + lane) * 16; };
        constexpr int kCoherent = 16;  // sc1
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
#pragma unroll
        for (int rm = 0; rm < RME; ++rm)
#pragma unroll
            for (int rn = 0; rn < RN; ++rn)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[rm][rn]), prs,
                                                       q * kTileBytes + frag_off(rm, rn), 0, kCoherent);
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's partial stores are acknowledged
        __shared__ int last_flag;
        __syncthreads();
        if (tid == 0)
            last_flag = __hip_atomic_fetch_add(&counters[lin], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
                        static_cast<uint32_t>(ksplit - 1);
        __syncthreads();
        if (!last_flag) return;
        // the other splits' partials are read in split order, kQ splits' loads in flight at a time
        constexpr int kQ = RME * RN <= 4 ? 4 : 2;
        f32x4 sum[RME][RN];
#pragma unroll
        for (int rm = 0; rm < RME; ++rm)
#pragma unroll
            for (int rn = 0; rn < RN; ++rn) sum[rm][rn] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int q0 = 0; q0 < ksplit; q0 += kQ) {
            f32x4 t[kQ][RME][RN];
#pragma unroll
            for (int j = 0; j < kQ; ++j)
#pragma unroll
                for (int rm = 0; rm < RME; ++rm)
#pragma unroll
                    for (int rn = 0; rn < RN; ++rn)
                        t[j][rm][rn] = q0 + j < ksplit && q0 + j != q
                                           ? __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                                           prs, (q0 + j) * kTileBytes + frag_off(rm, rn),
                                                                           0, kCoherent))
                                           : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < kQ; ++j)
#pragma unroll
                for (int rm = 0; rm < RME; ++rm)
#pragma unroll
                    for (int rn = 0; rn < RN; ++rn) sum[rm][rn] += q0 + j == q ? acc[rm][rn] : t[j][rm][rn];
        }
#pragma unroll
        for (int rm = 0; rm < RME; ++rm)
#pragma unroll
            for (int rn = 0; rn < RN; ++rn) acc[rm][rn] = sum[rm][rn];
        if (tid == 0)  // ready for the next call on this stream
            __hip_atomic_store(&counters[lin], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    // ---- rank-R term T . U^T (fp32, one MFMA K step per 32 ranks; weights' role
    // for U, activations' role for T, so the accumulator layout is the main
    // loop's), added to dst ----
    auto add_term = [&](f32x4 (&dst)[RM][RN], auto factors_bf16) {
        static_assert(kStage >= BM * 128 && kStage >= BN * 128, "a 64-rank chunk of T or U must fit a stage buffer");
        // 64 ranks at a time, the tile's T rows and U rows are copied into the
        // (now free) stage buffers with the A operand's layout (128-byte rows,
        // chunk c at c ^ swz(row)), one round trip for the whole tile, and the
        // MFMA steps read their fragments from LDS. Step kh covers ranks
        // [32 kh, 32 kh + 32): lane group lg reads chunk lg + 4 kh of T and U.
        // A 32-rank tail copies ranks [0, 32) only and runs step 0.
        // kSlots chunks are in flight at a time where the ring has room (both factors in one
        // stage buffer, or in two): their round trips would otherwise follow one another (us, one
        // in flight -> kSlots, rank 1024: M=154 N=K=3072 23.8 -> 20.7, M=1000 41.6 -> 37.9, M=8
        // N=2048 K=12288 23.6 -> 20.9, rank 512 18.1 -> 17.3; up to 64 ranks the same; as many as
        // the ring has stages, six there: 21.5).
        constexpr bool kOneBuf = kStage >= (BM + BN) * 128;
        constexpr int kSlots = kOneBuf ? 3 : kStages >= 4 ? 2 : 1;
        auto slot_t = [&](int slot) -> uint32_t {
            if constexpr (kOneBuf) return slot == 0 ? lds_addr_of(sbuf0) : slot == 1 ? lds_addr_of(sbuf1) : lds_addr_of(sbuf2);
            else return slot == 0 ? lds_addr_of(sbuf0) : lds_addr_of(sbuf2);
        };
        auto slot_u = [&](int slot) -> uint32_t {
            if constexpr (kOneBuf) return slot_t(slot) + BM * 128;
            else return slot == 0 ? lds_addr_of(sbuf1) : lds_addr_of(sbufx);
        };
        constexpr int kTInst = BM / 8;  // 1 KB copies: 8 rows of 64 ranks
        constexpr int kUInst = BN / 8;
        // the same number for every wave, so that the wait counts are constants: surplus
        // ones repeat the last copy
        constexpr int kPerWave = (kTInst + kUInst + kWaves - 1) / kWaves;
        const int chunks = (lora_rank + 63) / 64;
        auto issue_chunk = [&](int ch, int slot) {
            const int r0 = ch * 64;
            const bool rtail = lora_rank - r0 < 64;
#pragma unroll
            for (int i = 0; i < kPerWave; ++i) {
                const int j = i * kWaves + wave < kTInst + kUInst ? i * kWaves + wave : kTInst + kUInst - 1;
                const bool is_t = j < kTInst;
                const int jj = is_t ? j : j - kTInst;
                const int row = jj * 8 + (lane >> 3);
                int c = (lane & 7) ^ swz(row);
                if (rtail && c >= 4) c -= 4;  // past the rank: a valid chunk, never read
                const int grow = is_t ? (m0 + row < M ? m0 + row : M - 1) : (n0 + row < N ? n0 + row : N - 1);
                dma16_lds(is_t ? lora_t : lora_u, static_cast<uint32_t>((grow * lora_rank + r0 + 8 * c) * 2),
                          (is_t ? slot_t(slot) : slot_u(slot)) + jj * 1024);
            }
        };
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wave's reads of the buffers are done
        stage_barrier();                      // and every other wave's
#pragma unroll
        for (int i = 0; i < kSlots; ++i)
            if (i < chunks) issue_chunk(i, i);
        int slot = 0;
        for (int ch = 0; ch < chunks; ++ch) {
            // chunk ch has landed once only the kSlots - 1 after it are outstanding
            if (ch + kSlots <= chunks) wait_vmcnt<(kSlots - 1) * kPerWave>();
            else wait_vmcnt<0>();
            stage_barrier();
            const uint32_t lt = slot_t(slot), lu = slot_u(slot);
            for (int kh = 0; kh < (lora_rank - ch * 64 < 64 ? 1 : 2); ++kh) {
                uint4 tf[RME], uf[RN];
#pragma unroll
                for (int rm = 0; rm < RME; ++rm) {
                    const int row = erow0 + rm * 16 + lr;
                    tf[rm] = lds_ld16(lt + row * 128 + (((lg + 4 * kh) ^ swz(row)) << 4));
                }
#pragma unroll
                for (int rn = 0; rn < RN; ++rn) {
                    const int row = wave_n * WTN + rn * 16 + lr;
                    uf[rn] = lds_ld16(lu + row * 128 + (((lg + 4 * kh) ^ swz(row)) << 4));
                }
#pragma unroll
                for (int rm = 0; rm < RME; ++rm)
#pragma unroll
                    for (int rn = 0; rn < RN; ++rn) {
                        if constexpr (!decltype(factors_bf16)::value)
                            dst[rm][rn] = mfma16x16x32(as_half8(uf[rn]), as_half8(tf[rm]), dst[rm][rn]);
                        else
                            dst[rm][rn] = mfma16x16x32_bf16(uf[rn], tf[rm], dst[rm][rn]);
                    }
            }
            if (ch + kSlots < chunks) {
                __builtin_amdgcn_s_waitcnt(0xC07F);  // the slot's readers are done
                stage_barrier();
                issue_chunk(ch + kSlots, slot);
            }
            slot = slot + 1 < kSlots ? slot + 1 : 0;
        }
    };
    if constexpr (kLora == 1 || kLora == 2) {
        // the weight scale applies to the fp8 product only: scale first, then add the term
#pragma unroll
        for (int rm = 0; rm < RM; ++rm)
#pragma unroll
            for (int rn = 0; rn < RN; ++rn)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    acc[rm][rn][i] = opaque_f32(acc[rm][rn][i] * s);
        s = 1.0f;
        add_term(acc, std::bool_constant<kLora == 2>{});
    }
    [[maybe_unused]] f32x4 term[kLora == 3 ? RM : 1][RN];
    [[maybe_unused]] const bool term_bf16 = (lora_flags & 1) != 0, term_after = (lora_flags & 2) != 0;
    if constexpr (kLora == 3) {
#pragma unroll
        for (int rm = 0; rm < RM; ++rm)
#pragma unroll
            for (int rn = 0; rn < RN; ++rn) term[rm][rn] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (term_after) {
            if (term_bf16) add_term(term, std::true_type{});
            else add_term(term, std::false_type{});
        } else {
#pragma unroll
            for (int rm = 0; rm < RME; ++rm)
#pragma unroll
                for (int rn = 0; rn < RN; ++rn)
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[rm][rn][i] = opaque_f32(acc[rm][rn][i] * s);
            s = 1.0f;
            if (term_bf16) add_term(acc, std::true_type{});
            else add_term(acc, std::false_type{});
        }
    }

    // ---- epilogue: each wave stages its whole output tile (RME x RN 16 x 16 tiles) in LDS
    // (the stage buffers, free once every wave is past its last stage) with
    // one wait, then stores rows of WTN * 2 contiguous bytes ----
    const int out_col0 = n0 + wave_n * WTN;
    constexpr int kCPR = WTN / 8;                // 16-byte chunks per staged row
    constexpr int kRowBytes = WTN * 2;
    constexpr int kRowsPerStore = 64 / kCPR;     // rows one store instruction covers
    constexpr int kLanesUsed = kRowsPerStore * kCPR;
    constexpr int kWaveRows = RME * 16;
    constexpr int kWaveBytes = kWaveRows * kRowBytes;
    constexpr int kWavesPerBuf = kStage / kWaveBytes;
    static_assert(3 * kWavesPerBuf >= kWaves, "epilogue staging must fit the stage buffers");
    const int cc = lane % kCPR;  // this lane's chunk of every row it stores
    const int rsub = lane / kCPR;
    const int gcol = out_col0 + cc * 8;
    // the bias chunk is issued before the barrier and waited for after the
    // staging writes, so its latency overlaps them
    const uint4 b8 = has_bias && lane < kLanesUsed && gcol < N ? load_bias8(bias + gcol) : make_uint4(0u, 0u, 0u, 0u);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wave's last operand reads are done
    stage_barrier();
    auto staging = [&](int buf) -> uint8_t* {
        uint8_t* const b = buf == 0 ? sbuf0 : buf == 1 ? sbuf1 : buf == 2 ? sbuf2 : sbufx + (buf - 3) * kStage;
        return b + (wave % kWavesPerBuf) * kWaveBytes;
    };
    uint8_t* sc = staging(wave / kWavesPerBuf);
    // a separately added term is staged like the result, in the buffers behind it
    constexpr int kResultBufs = (kWaves + kWavesPerBuf - 1) / kWavesPerBuf;
    static_assert(kLora != 3 || 2 * kResultBufs <= kStages, "result and term must fit the stage buffers");
    [[maybe_unused]] uint8_t* const st_term = staging(wave / kWavesPerBuf + (kLora == 3 ? kResultBufs : 0));
    if constexpr (kLora == 3) {
        if (term_after) {
#pragma unroll
            for (int rm = 0; rm < RME; ++rm)
#pragma unroll
                for (int rn = 0; rn < RN; ++rn) {
                    const int row = rm * 16 + lr;
                    const int chunk = (2 * rn + (lg >> 1) + row) % kCPR;
                    const f32x4 v = term[rm][rn];
                    *reinterpret_cast<uint2*>(st_term + row * kRowBytes + chunk * 16 + (lg & 1) * 8) =
                        make_uint2(round_via<kBf16>(v[0], v[1], term_bf16), round_via<kBf16>(v[2], v[3], term_bf16));
                }
        }
    }
    // chunk c of staged row r sits at (c + r) % kCPR (spreads the rows of one
    // write over the LDS banks). bf16 outputs are converted without NaN
    // canonicalisation first; a wave that produced a NaN stages again with
    // torch's canonical NaN (the per-pair canonicalisation in staging and in
    // the bias add cost ~0.7 us per tile: M=4096 N=3072 K=3072 57.9 -> 56.5 us).
    uint32_t nan_track = 0u;
    auto stage = [&](auto canonical) {
        constexpr bool kCanon = decltype(canonical)::value;
#pragma unroll
        for (int rm = 0; rm < RME; ++rm) {
            const int row = rm * 16 + lr;
#pragma unroll
            for (int rn = 0; rn < RN; ++rn) {
                float v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    v[i] = kLora == 1 || kLora == 2 ? acc[rm][rn][i] : opaque_f32(acc[rm][rn][i] * s);
                // row lr, columns 4*lg .. 4*lg+3 of this 16x16 tile: one 8-byte write
                const int chunk = (2 * rn + (lg >> 1) + row) % kCPR;
                uint32_t w0, w1;
                if constexpr (kBf16 && !kCanon) {
                    w0 = f32x2_to_bf16x2_raw(v[0], v[1]);
                    w1 = f32x2_to_bf16x2_raw(v[2], v[3]);
                    nan_track = bf16x2_nan_track(bf16x2_nan_track(nan_track, w0), w1);
                } else {
                    w0 = f32x2_to_out_bits<kBf16>(v[0], v[1]);
                    w1 = f32x2_to_out_bits<kBf16>(v[2], v[3]);
                }
                *reinterpret_cast<uint2*>(sc + row * kRowBytes + chunk * 16 + (lg & 1) * 8) = make_uint2(w0, w1);
            }
        }
    };
    stage(std::false_type{});
    if constexpr (kBf16)
        if (__builtin_amdgcn_ballot_w64(bf16x2_nan_seen(nan_track))) stage(std::true_type{});
    // staging writes and the bias load complete: one wait, then no vmcnt wait
    // between the stores (vmcnt counts stores too)
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
    wave_lds_sync();                     // each wave reads only its own region
    const int out_row0 = m0 + erow0;
#pragma unroll
    for (int p = 0; p < (kWaveRows + kRowsPerStore - 1) / kRowsPerStore; ++p) {
        const int r = p * kRowsPerStore + rsub;
        const int grow = out_row0 + r;
        if (lane < kLanesUsed && r < kWaveRows && grow < M && gcol < N) {
            uint4 v = *reinterpret_cast<const uint4*>(sc + r * kRowBytes + ((cc + r) % kCPR) * 16);
            if (has_bias) {
                if constexpr (kBf16) {
                    uint4 vb = v;
                    uint32_t nt = 0u;
                    add_bias8<true, false>(vb, b8, &nt);
                    if (__builtin_amdgcn_ballot_w64(bf16x2_nan_seen(nt))) add_bias8<true>(v, b8);
                    else v = vb;
                } else {
                    add_bias8<false>(v, b8);
                }
            }
            if constexpr (kLora == 3)
                if (term_after)
                    add_bias8<kBf16>(v, *reinterpret_cast<const uint4*>(st_term + r * kRowBytes + ((cc + r) % kCPR) * 16));
            uint4* dst = reinterpret_cast<uint4*>(C + static_cast<int64_t>(grow) * N + gcol);
            if (c_nontemporal) {
                typedef uint32_t u32x4_nt __attribute__((ext_vector_type(4)));
                __builtin_nontemporal_store(u32x4_nt{v.x, v.y, v.z, v.w}, reinterpret_cast<u32x4_nt*>(dst));
            } else {
                *dst = v;
            }
        }
    }
}

// Whether the epilogue can stage a separately added term beside the result (see
// kResultBufs) and hold 64 ranks of T and U in a stage buffer each.
template <int BM, int BN, int WAVES, int GROUPS, int STAGES>
constexpr bool term_fits() {
    constexpr int kStage = GROUPS * (BM * 128 + BN * 64), kPerBuf = kStage / (BM * BN * 2 / WAVES);
    return 2 * ((WAVES + kPerBuf - 1) / kPerBuf) <= STAGES && kStage >= BM * 128 && kStage >= BN * 128;
}

template <int BM, int BN, int WAVES_M, int WAVES_N, int PIPE, int STAGES = 3, int GROUPS = 1, bool TAIL = false>
bool launch_lds(const MmArgs& p, hipStream_t stream, int ksplit = 1, float* partials = nullptr,
                uint32_t* counters = nullptr) {
    const int tiles_m = (p.M + BM - 1) / BM;
    const int tiles_n = (p.N + BN - 1) / BN;
    const int group_m = p.group_m > 0 ? p.group_m : 4;
    // Outputs larger than the 256 MB MALL are written with nontemporal stores:
    // they are never re-read here and cannot stay cached for the next layer
    // anyway (M=32768 N=13824 K=5120 3.096 -> 3.081 ms on MI355X). Smaller
    // outputs keep ordinary stores: nontemporal ones measured ~2% faster for an
    // isolated one-wave M=4096 N=3072 GEMM, but a chained FFN (M=4096,
    // 3072 -> 12288 -> 3072) took 414 us with ordinary stores and 419 us with
    // the 100 MB intermediate written nontemporally.
    const int c_nt = p.M * p.N * 2 > (int64_t(256) << 20) ? 1 : 0;
    const dim3 grid(static_cast<uint32_t>(tiles_m * tiles_n * ksplit));
    const dim3 block(64 * WAVES_M * WAVES_N * GROUPS);
#define FEATHER_LDS_LAUNCH_L(BF, E4, LORA)                                                                            \
    hipLaunchKernelGGL((scaled_mm_lds_kernel<BM, BN, WAVES_M, WAVES_N, PIPE, BF, E4, LORA, STAGES, GROUPS, TAIL>),     \
                       grid, block, 0, stream, p.a, p.b, p.scale, p.bias, p.c, static_cast<int>(p.M),                 \
                       static_cast<int>(p.N), static_cast<int>(p.K), p.has_scale, p.has_bias, tiles_m, tiles_n,       \
                       group_m, ksplit, partials, counters, p.lora_t, p.lora_u, static_cast<int>(p.lora_rank),         \
                       (p.lora_dtype == 2 ? 1 : 0) | (p.lora_after ? 2 : 0), c_nt)
#define FEATHER_LDS_LAUNCH(BF, E4) FEATHER_LDS_LAUNCH_L(BF, E4, 0)
    if (p.lora_dtype != 0) {
        // rank-R epilogue with the factors' type and the place of the rounding as
        // arguments: the planned tiles (fp16 activations, e5m2 weights, with or without a K split)
        if constexpr (TAIL && term_fits<BM, BN, WAVES_M * WAVES_N * GROUPS, GROUPS, STAGES>()) {
            if (p.a_bf16 || p.b_e4m3) return false;
            if (p.out_bf16) FEATHER_LDS_LAUNCH_L(true, false, 3);
            else FEATHER_LDS_LAUNCH_L(false, false, 3);
            return true;
        }
        // rank-R epilogue: the default schedule's large tiles, fp16 activations,
        // e5m2 weights, no K split
        // (the T and U chunks must fit a stage buffer: not the 128 x 384 tile)
        if constexpr (PIPE == 1 && !TAIL && BM >= 128 && BM * 128 + BN * 64 >= (BM > BN ? BM : BN) * 128) {
            if (p.a_bf16 || p.b_e4m3 || ksplit != 1) return false;
            if (p.lora_dtype == 1) {
                if (p.out_bf16) FEATHER_LDS_LAUNCH_L(true, false, 1);
                else FEATHER_LDS_LAUNCH_L(false, false, 1);
            } else {
                if (p.out_bf16) FEATHER_LDS_LAUNCH_L(true, false, 2);
                else FEATHER_LDS_LAUNCH_L(false, false, 2);
            }
            return true;
        }
        return false;
    }
    // bf16 activations: none of these tiles; the caller rounds A to fp16 first.
    // Converting each A fragment as it is read costs more than a separate cast
    // pass on every tile here, because each fragment is read by 2-4 waves and
    // feeds only 1-6 MFMAs (graph-replayed, bf16 out, M=512 N=3072 K=12288 on
    // the 64 x 64 split-K tiles: 102 us converted in the kernel vs 60 us cast
    // first, fp16 A 54 us; M=4096 N=3072 K=3072 on the 128 x 384 tile: 68 vs
    // 66 us; M=32768 N=13824 K=5120 on the 256 x 256 tile: 4.44 vs 3.68 ms). On the
    // tiles with two K groups, each wave rounding the A chunks it copied itself in LDS
    // before the barrier that publishes them: M=154 N=10240 K=4096 27.9 us (64 x
    // 128; fp16 A 21.1, the cast pass 3.5), M=512 N=3072 K=12288 47.9 (64 x 192;
    // 39.5 and 5.5), M=333 N=K=3072 19.6 (14.0 and 4): the read, write and wait in
    // LDS cost the same without the conversion itself.
    if (p.a_bf16) return false;
    if (p.out_bf16) {
        if (p.b_e4m3) FEATHER_LDS_LAUNCH(true, true);
        else FEATHER_LDS_LAUNCH(true, false);
    } else {
        if (p.b_e4m3) FEATHER_LDS_LAUNCH(false, true);
        else FEATHER_LDS_LAUNCH(false, false);
    }
#undef FEATHER_LDS_LAUNCH
#undef FEATHER_LDS_LAUNCH_L
    return true;
}

}  // namespace

}  // namespace feather
