// Which variant serves a shape: a cost model of every tile, fitted to measured times.
//
// Time of one launch in us, from back-to-back runs on MI355X (256 shapes, M
// 17..8192, N and K 1024..13824, three rotated operand sets; least squares on the
// relative error, 3-5% rms per tile). u = 64-K steps one workgroup multiplies, f =
// share of the CUs that have a workgroup:
//   one round of workgroups:  c0 + u (b0 + b1 f)
//   R rounds:                 c0 + (R - 1) round + R u (b0 + b1)
//   K split s ways:           + s0 + s1 s (partial tile in 64 KB)
// The variant with the least modelled time is within 1% of the fastest measured one
// on average, on 90 shapes that the fit had not seen as well (worst 10%). Against
// the earlier rules (waves of workgroups x tile area, split-K tiles where their
// grid fitted one round), on the shapes that took the large tiles: 9% less time,
// the worst case 5% more.
#include <stdint.h>

#include "scaled_mm_dispatch.h"

namespace feather {
namespace {

struct TileCost {
    int tile, bm, bn, groups;
    bool any_k;  // K need not be a multiple of 64
    double c0, b0, b1, round, s0, s1;
};

constexpr TileCost kTiles[] = {
    {kMid32x64, 32, 64, 2, true, 3.77, 0.075, 0.022, 2.40, 1.07, 1.92},
    {kLdsSk32x128, 32, 128, 2, true, 4.18, 0.105, 0.040, 2.41, 1.07, 1.30},
    {kLdsSk64x64, 64, 64, 2, true, 4.07, 0.105, 0.034, 2.70, 0.98, 1.31},
    {kMid96x64, 96, 64, 2, true, 4.48, 0.149, 0.041, 3.47, 1.10, 1.06},
    {kLdsSk64x128, 64, 128, 2, true, 4.89, 0.151, 0.061, 3.17, 1.23, 0.93},
    {kMid96x128, 96, 128, 2, true, 5.48, 0.216, 0.082, 3.87, 1.20, 0.85},
    {kMid64x192, 64, 192, 2, true, 5.83, 0.220, 0.075, 4.22, 1.24, 0.84},
    {kMid96x192, 96, 192, 2, true, 6.56, 0.302, 0.100, 5.74, 1.55, 0.75},
    {kMid128x128, 128, 128, 1, true, 4.68, 0.275, 0.075, 4.69, 0, 0},
    {kMid128x192, 128, 192, 1, true, 5.62, 0.396, 0.106, 6.71, 0, 0},
    {kLds128x256, 128, 256, 1, false, 6.00, 0.501, 0.126, 7.20, 0, 0},
    {kLds256x128, 256, 128, 1, false, 6.18, 0.500, 0.129, 7.28, 0, 0},
    {kLds256x192, 256, 192, 1, false, 8.58, 0.731, 0.224, 7.93, 0, 0},
    {kLds128x384, 128, 384, 1, false, 8.48, 0.751, 0.196, 7.84, 0, 0},
    {kLds256x256, 256, 256, 1, false, 9.20, 0.991, 0.231, 8.95, 0, 0},
    {kLds128x128, 128, 128, 1, false, 0, 0, 0, 0, 0, 0},  // see cost_us
    {kTail128x256, 128, 256, 1, true, 6.00, 0.501, 0.126, 7.20, 0, 0},
};

constexpr int kMaxSplit = 16;
// Partial tiles of a split (a workspace that callers keep per stream)
constexpr size_t kMaxSplitBytes = size_t(15) << 20;

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

double cost_us(const TileCost& t, int64_t tiles, int64_t stages, int ks, int cus) {
    const int64_t groups = tiles * ks;
    const double u = static_cast<double>(ceil_div(stages, ks) * t.groups);
    const double fill = static_cast<double>(groups) / cus;
    const double rounds = static_cast<double>(ceil_div(groups, cus));
    if (t.tile == kLds128x128)  // two workgroups per CU: past one round their ramps overlap (2.7% rms)
        return 3.57 + (2.58 + 0.163 * u) * fill + 0.211 * u * rounds;
    double us = groups <= cus ? t.c0 + u * (t.b0 + t.b1 * fill)
                              : t.c0 + (rounds - 1.0) * t.round + rounds * u * (t.b0 + t.b1);
    if (ks > 1) us += t.s0 + t.s1 * ks * (t.bm * t.bn * 4 / 65536.0);
    return us;
}

// Small-M kernel, 17..48 rows. Up to 32: the lean kernel on unsplit 16-column strips
// (K % 64 == 0: fit of 29 shapes, 3.5% rms; otherwise the general kernel on those strips,
// of 23 shapes, 11% rms; the split plans lose to the 32-row tiles: M=22 N=1152
// K=10304 12.0 vs 8.6 us, M=19 N=8576 K=6144 15.3 vs 11.8). 33..48 rows: unsplit
// strips with K < 2048 (M=34 N=1792 K=1392 4.8 vs 5.4 us; longer K: M=38 N=2176
// K=6848 14.8 vs 9.1).
double smallm_us(int64_t M, int64_t N, int64_t K, int cus) {
    const double mb = static_cast<double>(N) * static_cast<double>(K) * 1e-6;
    const double rounds = static_cast<double>(ceil_div(ceil_div(N, 16), cus));
    const double steps = rounds * static_cast<double>(ceil_div(K, 64));
    if (M <= 32 && K % 64 == 0)
        return 1.78 + 0.706 * static_cast<double>(ceil_div(N, 16)) / cus + (0.0178 + 0.0012 * static_cast<double>(M)) * steps +
               0.0095 * mb;
    if (M <= 32) return 2.16 + 0.13 * rounds + (0.0347 + 0.0011 * static_cast<double>(M - 17)) * steps + 0.071 * mb;
    if (M <= 48 && K < 2048)
        return 1.02 + 0.63 * rounds + (0.108 + 0.0017 * static_cast<double>(M - 33)) * steps + 0.40 * mb;
    return 1e30;
}

const TileCost* tile_cost(int tile) {
    for (const TileCost& t : kTiles)
        if (t.tile == tile) return &t;
    return nullptr;
}

MmPlan make_plan(int64_t M, int64_t N, int64_t K, int cus, bool lora) {
    MmPlan best;
    const bool lean = M <= 32 && smallm_is_lean(M, N, K, cus, M <= 16);
    if (M <= 16 && (!lora || lean)) {
        // one row tile: the small-M kernel and its own plan. The 32 x 64 tile took up to 8%
        // less on a few wide weights (M=16 N=13824 K=5120 13.2 vs 14.3 us), but bf16
        // activations would need a cast pass of 3.5 us first, and both types take one plan
        best.tile = kSmallM;
        best.ksplit = smallm_ksplit(M, N, K, cus);
        best.workspace_bytes = smallm_workspace_bytes(M, N, K, cus);
        return best;
    }
    double best_us = 1e30;
    for (const TileCost& t : kTiles) {
        if (!t.any_k && K % 64 != 0) continue;
        if (t.tile == kTail128x256 && K % 64 == 0) continue;
        const int64_t tiles = ceil_div(M, t.bm) * ceil_div(N, t.bn);
        if (t.tile == kMid128x128 && tiles > cus && K % 64 == 0) continue;
        if (t.tile == kLds128x128 && tiles <= cus) continue;
        const int64_t stages = ceil_div(K, 64 * t.groups);
        int64_t last = 0;
        for (int ks = 1; ks <= kMaxSplit; ++ks) {
            if (ks > 1) {
                if (t.groups != 2 || tiles * ks > cus || tiles > kWorkspaceCounters) break;
                const int64_t per = ceil_div(stages, ks);
                if (per < 2) break;
                if (per == last || ceil_div(stages, per) != ks) continue;  // the same stages, or an empty split
                if (tile_workspace_bytes(t.tile, M, N, ks) > kMaxSplitBytes) break;
            }
            last = ceil_div(stages, ks);
            const double us = cost_us(t, tiles, stages, ks, cus);
            if (us < best_us) {
                best_us = us;
                best.tile = t.tile;
                best.ksplit = ks;
            }
        }
    }
    best.workspace_bytes = tile_workspace_bytes(best.tile, M, N, best.ksplit);
    if (M > 16 && M <= 48 && (!lora || lean)) {
        // bf16 activations cost a cast pass (3.5 us and more) before a tile, none on the
        // small-M kernel, and both types take one plan: where a weight is too small to
        // make the tiles the better choice for most rows, they have to win by that much
        const bool large = N * K > int64_t(4096) * 4096;
        const double margin = !large && (M <= 32 || N < 3072) ? 3.5 : 0.0;
        if (smallm_us(M, N, K, cus) <= best_us + margin) best = MmPlan{kSmallM, 1, 0};
    }
    return best;
}

}  // namespace

size_t tile_workspace_bytes(int tile, int64_t M, int64_t N, int ksplit) {
    const TileCost* t = tile_cost(tile);
    if (t == nullptr || ksplit <= 1) return 0;
    const int64_t tiles = ceil_div(M, t->bm) * ceil_div(N, t->bn);
    return kWorkspaceCounterBytes + static_cast<size_t>(tiles) * ksplit * t->bm * t->bn * 4;
}

// The plan is a pure function of its arguments and costs about a microsecond, so each
// thread keeps the last few.
static MmPlan plan(int64_t M, int64_t N, int64_t K, int cus, bool lora) {
    struct Entry {
        int64_t M = -1, N = 0, K = 0;
        int cus = 0;
        bool lora = false;
        MmPlan plan;
    };
    static thread_local Entry memo[64];
    const uint64_t h = static_cast<uint64_t>(M) * 0x9e3779b97f4a7c15ull + static_cast<uint64_t>(N) * 0xc2b2ae3d27d4eb4full +
                       static_cast<uint64_t>(K) * 0x165667b19e3779f9ull + (lora ? 1u : 0u);
    Entry& e = memo[(h ^ (h >> 29)) * 0xbf58476d1ce4e5b9ull >> 58];
    if (e.M != M || e.N != N || e.K != K || e.cus != cus || e.lora != lora)
        e = Entry{M, N, K, cus, lora, make_plan(M, N, K, cus, lora)};
    return e.plan;
}

MmPlan plan_scaled_mm(int64_t M, int64_t N, int64_t K, int cus) { return plan(M, N, K, cus, false); }
MmPlan plan_scaled_mm_lora(int64_t M, int64_t N, int64_t K, int cus) { return plan(M, N, K, cus, true); }

}  // namespace feather
