// Which variant serves a shape: a cost model of every tile, fitted to measured times.
//
// Time of one launch in us, from back-to-back runs on MI355X (256 shapes, M
// 17..8192, N and K 1024..13824, three rotated operand sets, so that most weights
// stay in the MALL; least squares on the relative error, 3-5% rms per tile; with
// the weight in HBM a call of few rows takes about 0.1 us per MB more). u = 64-K steps one workgroup multiplies, f =
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

// The same for the split-K tiles' short form (short_k_tile): 136 shapes with the weight in
// HBM, 3-4% rms, up to two workgroups per CU, which share it. Past those every workgroup's
// epilogue counts and larger tiles win (M=777 N=4928 K=64 7.5 us on 64 x 64, 6.4 on 128 x 192).
constexpr TileCost kShortTiles[] = {
    {kLdsSk32x128, 32, 128, 1, false, 3.22, 0.156, 0.021, 0.3, 0, 0},
    {kLdsSk64x64, 64, 64, 1, false, 3.16, 0.138, 0.041, 0.3, 0, 0},
    {kLdsSk64x128, 64, 128, 1, false, 3.66, 0.216, 0.053, 1.0, 0, 0},
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

// Small-M kernel, 17..48 rows: its form with the least modelled time, from graph-replayed runs
// that rotate weights past the MALL (a model's layers find their weights in HBM; fits of weights
// that stay in the MALL are up to 40% low on these forms). tile_us: the best tile, the same way.
// A form whose launch takes bf16 activations spares them the cast pass that every tile needs
// (2.3-2.9 us), and both activation types take one plan: such a form may be slower than the tile by
// that much unsplit, and by less where the tile's gain on fp16 calls is larger than the cast's
// cost to bf16 ones (K splits, weights above 4096 x 4096; none past one round of strips of those).
// strip 0: the tile.
struct SmallmChoice {
    int strip = 0, ksplit = 1;
};

SmallmChoice smallm_choice(int64_t M, int64_t N, int64_t K, int cus, bool lora, double tile_us) {
    const int64_t stages = ceil_div(K, 64), strips = ceil_div(N, 16);
    const double m = static_cast<double>(M), nst = static_cast<double>(stages);
    const double mb = static_cast<double>(N) * static_cast<double>(K) * 1e-6, a = m * static_cast<double>(K) * 1e-6;
    if (M > 32) {
        // unsplit 16-column strips, one workgroup per CU, which read fp16 activations; rows whose
        // pitch is a multiple of 128 bytes read slower (59 shapes, 3% rms). From K = 2048 on a
        // tile wins (M=34 N=736 K=9744 18.6 vs 8.6 us), past one round too (M=40 N=5456 K=320 6.2 vs 4.4)
        const double us = K % 64 == 0 ? 2.78 + 0.0033 * m * nst + 0.213 * mb : 2.56 + (0.049 + 0.0012 * m) * nst + 0.14 * mb;
        return {K < 2048 && strips <= cus && !lora && us <= tile_us ? 1 : 0, 1};
    }
    const bool large = N * K > int64_t(4096) * 4096;
    const double slack = !large ? 2.5 : strips <= cus ? 1.75 : 0.0;
    SmallmChoice best;
    double best_us = 1e30;
    bool take = false;
    auto offer = [&](int ks, double us, double allowed) {
        take = take || us <= tile_us + allowed;
        if (us < best_us) best_us = us, best = {1, ks};
    };
    if (K % 64 == 0) {
        // the lean kernel, two workgroups per CU (134 shapes, 6.3% rms); a fourth round of strips is
        // the tiles', a third on a short K too (M=26 N=12736 K=768 6.9 vs 5.7 us, N=9968 K=384 4.6 vs 4.1)
        const double rounds = static_cast<double>(ceil_div(strips, cus));
        if ((strips <= 2 * cus || (strips <= 3 * cus && K >= 512)) && (!lora || is_lean(smallm_form(M, N, K, cus, 1, 1))))
            offer(1, 1.89 + 0.484 * rounds + (0.0017 + 0.0011 * m + 0.085 * a) * rounds * nst + 0.156 * mb, slack);
    } else if (strips <= cus) {
        // the general kernel on 16-column strips (105 shapes, 6% rms)
        if (!lora) offer(1, 2.82 + (0.015 + 0.0009 * m + 0.087 * a) * nst + 0.212 * mb, slack);
    } else if (K < 1600 && !lora) {
        // past one round of those, 64-column strips (fp16 activations): 2-9% less than the best tile on 8
        // of 9 shapes up to K = 1504 (M=23 N=9520 K=752 4.8 vs 5.1 us), 1-4% more from K = 2208 on;
        // 16-column strips M=32 N=8432 K=1104 11.1 vs 6.8
        return {4, 1};
    }
    // K split of 16-column strips in one round (81 shapes, 3.9% rms, and 0.3 us that it has to be worth):
    // long K on narrow weights (M=31 N=640 K=9696 12.2 us unsplit, 7.9 in four splits). Wide split strips
    // lose to the 32-row tiles
    if (!lora)
        for (int ks = 2; ks <= 8 && ks * 16 <= stages && ks * strips <= cus; ++ks)
            offer(ks, 3.85 + (0.0187 + 0.0015 * m) * static_cast<double>(ceil_div(stages, ks)) + 0.393 * ks + 0.15 * mb,
                  0.4 * slack);
    return take ? best : SmallmChoice{};
}

const TileCost* tile_cost(int tile) {
    for (const TileCost& t : kTiles)
        if (t.tile == tile) return &t;
    return nullptr;
}

const TileCost* short_cost(int tile) {
    for (const TileCost& t : kShortTiles)
        if (t.tile == tile) return &t;
    return nullptr;
}

MmPlan make_plan(int64_t M, int64_t N, int64_t K, int cus, bool lora) {
    MmPlan best;
    if (M <= 16 && (!lora || is_lean(smallm_form(M, N, K, cus, 0, 0)))) {
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
            const TileCost* const brief =
                !lora && tiles <= 2 * cus && short_k_tile(t.tile, K, ks) ? short_cost(t.tile) : nullptr;
            const double us = brief ? cost_us(*brief, tiles, ceil_div(K, 64), 1, cus) : cost_us(t, tiles, stages, ks, cus);
            if (us < best_us) {
                best_us = us;
                best.tile = t.tile;
                best.ksplit = ks;
            }
        }
    }
    best.workspace_bytes = tile_workspace_bytes(best.tile, M, N, best.ksplit);
    if (M > 16 && M <= 48) {
        // the table's time with the weight in HBM (190 shapes of 17..48 rows, 4.4% rms)
        const double tile_us = 0.94 * best_us + 0.1e-6 * static_cast<double>(N) * static_cast<double>(K);
        const SmallmChoice c = smallm_choice(M, N, K, cus, lora, tile_us);
        if (c.strip > 0) best = MmPlan{kSmallM, c.ksplit, smallm_split_bytes(M, N, c.strip, c.ksplit), c.strip};
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
