// Large tiles of the LDS-DMA GEMM (scaled_mm_lds_kernel.h) and the split-K tiles
// of the plan below.
#include <stdlib.h>

#include "scaled_mm_lds_kernel.h"

namespace feather {
namespace {

template <int PIPE>
bool launch_lds_pipe(int kernel_id, const MmArgs& p, hipStream_t stream, int ks = 1, float* partials = nullptr,
                     uint32_t* counters = nullptr) {
    switch (kernel_id) {
        // 256 x 256 and 256 x 192 on 4 x 2 waves (64 x 128 / 64 x 96 wave tiles:
        // 20% fewer LDS operand bytes per stage than 2 x 4, and wide enough
        // for the pinned schedule)
        case kLds256x256: return launch_lds<256, 256, 4, 2, PIPE>(p, stream);
        case kLds256x128: return launch_lds<256, 128, 4, 2, PIPE>(p, stream);
        case kLds128x256: return launch_lds<128, 256, 2, 4, PIPE>(p, stream);
        case kLds128x128: return launch_lds<128, 128, 2, 2, PIPE>(p, stream);
        case kLds256x192: return launch_lds<256, 192, 4, 2, PIPE>(p, stream);
        case kLds128x384: return launch_lds<128, 384, 2, 4, PIPE>(p, stream);
        // two K groups of 1 x 4 waves on a four- or five-stage ring of 128 K, both schedules' knob values
        case kLdsSk64x64: return launch_lds<64, 64, 1, 4, 1, 4, 2, true>(p, stream, ks, partials, counters);
        case kLdsSk64x128: return launch_lds<64, 128, 1, 4, 1, 4, 2, true>(p, stream, ks, partials, counters);
        case kLdsSk32x128: return launch_lds<32, 128, 1, 4, 1, 5, 2, true>(p, stream, ks, partials, counters);
        default: return false;
    }
}

}  // namespace

int lds_pipe_env() {
    // FEATHEROPS_LDS_PIPE: 1 (default) = operand-prefetch schedule, 0 = plain schedule
    static const int pipe_env = [] {
        const char* e = getenv("FEATHEROPS_LDS_PIPE");
        return e ? atoi(e) : 1;
    }();
    return pipe_env;
}

bool launch_lds_kernel(int kernel_id, const MmArgs& p, hipStream_t stream) {
    if (p.K % kBK != 0) return false;
    return lds_pipe_env() == 0 && !p.a_bf16 && p.lora_dtype == 0 ? launch_lds_pipe<0>(kernel_id, p, stream)
                                                                 : launch_lds_pipe<1>(kernel_id, p, stream);
}

// Split-K plan for the 32- and 64-row tiles: as many K splits as keep the
// grid within `target` workgroups (each split keeps at least one stage of
// 128 K; no split below K = 2048): each workgroup holds a CU's LDS.
// Stage ring (back to back, us): 64 x 64 on four stages of 128 K 9.7 at M=256
// N=K=3072, on six 9.9; 32 x 128 on five.
SplitKPlan lds_splitk_plan(int64_t M, int64_t N, int64_t K, int target) {
    SplitKPlan pl{};
    if (M <= 0 || K % kBK != 0) return pl;
    const int bm = M <= 32 ? 32 : 64;
    const int64_t nk = K / kBK;
    const int64_t nst = (K + 2 * kBK - 1) / (2 * kBK);  // the kernels' stages: 64 K for each of two groups
    auto splits = [&](int64_t tiles) {
        int64_t ks = target / tiles;
        // below 32 stages (K < 2048) the split's partial round trip costs more than the stages it
        // spreads (measured: M=256 N=K=1024 6.0 us unsplit vs 7.2 us in 4 splits, M=256 N=2048
        // K=512 4.7 vs 6.7 us; from K=2048 on splitting wins or ties)
        if (nk < 32) ks = 1;
        if (ks > nst) ks = nst;
        if (ks > 32) ks = 32;
        if (ks < 1) ks = 1;
        const int64_t per = (nst + ks - 1) / ks;
        ks = (nst + per - 1) / per;  // no empty split
        if (tiles > kWorkspaceCounters) ks = 1;  // more tiles than the counter region holds
        return ks;
    };
    // 64 rows: 64 x 64 tiles, or 64 x 128 where their grid comes closer to
    // `target` without passing it (or, past it, is smaller) in at most four K
    // splits. The last workgroup of a tile re-reads every split's partial
    // tile (32 KB at 64 x 128), so many splits of wide tiles lose: M=64 N=K=4096
    // (256 workgroups either way) 8.9 us on 64 x 64, 12.4 us on 64 x 128;
    // M=64 N=2176 K=8128 (238 workgroups in 7 splits vs 255 in 15) 10.6 vs
    // 17.1 us; M=64 N=6144 K=4096 (192 in 2 vs 240 in 5) 11.7 vs 12.7 us. Where
    // the wide grid is larger in few splits it wins: M=512 N=3072 K=12288 (384
    // vs 192 workgroups) 62.0 -> 47.3 us, M=128 N=K=5120 (160 vs 240 in 3
    // splits) 18.6 -> 15.7 us, M=48 N=9728 K=7488 (152 vs 228) 24.7 -> 20.5 us,
    // M=77 N=6448 K=10048 (202 vs 204 in 2) 28.4 -> 25.4 us (M=40 N=5552
    // K=6976, 174 vs 220 in 5 splits, would gain 5%).
    int bn = bm == 32 ? 128 : 64;
    if (bm == 64) {
        const int64_t t64 = (M + 63) / 64 * ((N + 63) / 64), t128 = (M + 63) / 64 * ((N + 127) / 128);
        const int64_t g64 = t64 * splits(t64), g128 = t128 * splits(t128);
        const bool wide = (g64 > target ? g128 < g64 : g128 <= target && g128 > g64) && splits(t128) <= 4;
        if (wide) bn = 128;
    }
    const int64_t tiles = (M + bm - 1) / bm * ((N + bn - 1) / bn);
    const int64_t ks = splits(tiles);
    pl.kernel_id = bm == 32 ? kLdsSk32x128 : bn == 128 ? kLdsSk64x128 : kLdsSk64x64;
    pl.ksplit = static_cast<int>(ks);
    pl.tiles = static_cast<int>(tiles);
    pl.workspace_bytes = ks > 1 ? kWorkspaceCounterBytes + static_cast<size_t>(tiles) * ks * bm * bn * 4 : 0;
    return pl;
}

bool launch_tile(int tile, const MmArgs& p, int ksplit, void* workspace, size_t workspace_bytes, hipStream_t stream) {
    uint32_t* counters = nullptr;
    float* partials = nullptr;
    if (ksplit > 1) {
        if (workspace == nullptr || workspace_bytes < tile_workspace_bytes(tile, p.M, p.N, ksplit)) return false;
        counters = static_cast<uint32_t*>(workspace);
        partials = reinterpret_cast<float*>(static_cast<uint8_t*>(workspace) + kWorkspaceCounterBytes);
    }
    if (tile >= kMid32x64) return launch_mid(tile, p, ksplit, partials, counters, stream);
    if (p.lora_dtype == 0 && short_k_tile(tile, p.K, ksplit)) return launch_short(tile, p, stream);
    if (tile == kLdsSk64x64 || tile == kLdsSk64x128 || tile == kLdsSk32x128)
        return launch_lds_pipe<1>(tile, p, stream, ksplit, partials, counters);
    return ksplit == 1 && launch_lds_kernel(tile, p, stream);
}

}  // namespace feather

