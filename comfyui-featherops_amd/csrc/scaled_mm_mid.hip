// Mid-size and any-K tiles of the LDS-DMA GEMM (scaled_mm_lds_kernel.h): the tiles
// that fill the chip once where the split-K and large tiles of scaled_mm_lds.hip
// over- or underfill it, and the tiles for K that is no multiple of 64.
#include "scaled_mm_lds_kernel.h"

namespace feather {

bool launch_mid(int tile, const MmArgs& p, int ksplit, float* partials, uint32_t* counters, hipStream_t stream) {
    // two K groups of 1 x 4 waves; ring as many stages of 128 K as 147 KB of LDS hold (32 x 64: six, 96 KB)
    switch (tile) {
        case kMid32x64: return launch_lds<32, 64, 1, 4, 1, 6, 2, true>(p, stream, ksplit, partials, counters);
        case kMid96x64: return launch_lds<96, 64, 1, 4, 1, 4, 2, true>(p, stream, ksplit, partials, counters);
        case kMid96x128: return launch_lds<96, 128, 1, 4, 1, 3, 2, true>(p, stream, ksplit, partials, counters);
        case kMid64x192: return launch_lds<64, 192, 1, 4, 1, 3, 2, true>(p, stream, ksplit, partials, counters);
        case kMid96x192: return launch_lds<96, 192, 1, 4, 1, 3, 2, true>(p, stream, ksplit, partials, counters);
        default: break;
    }
    if (ksplit != 1) return false;
    switch (tile) {
        // eight waves, so that every SIMD has two: on one round of workgroups 2 x 2 waves leave it with
        // one (M=1024 N=K=3072 26.4 -> 22.7 us, M=256 N=13824 K=5120 45.1 -> 41.7; past one round the
        // 2 x 2 tile has two workgroups per CU: M=2048 N=K=3072 41.9 vs 46.6)
        case kMid128x128: return launch_lds<128, 128, 2, 4, 1, 5, 1, true>(p, stream);
        case kMid128x192: return launch_lds<128, 192, 2, 4, 1, 4, 1, true>(p, stream);
        case kTail128x256: return launch_lds<128, 256, 2, 4, 1, 3, 1, true>(p, stream);
        default: return false;
    }
}

// The split-K tiles unsplit on a short K: one group of 1 x 4 waves, a stage of 64 K, two
// workgroups per CU past one round. Two groups with a stage of 128 K have half the stages to
// fill their ring with and an exchange of sums at the end, about 0.7 us that a short K does not
// earn back. us with the weight in HBM, two groups -> one: 64 x 64 M=260 N=3072 K=128 4.2 -> 3.5, K=320 5.0 ->
// 4.2, K=640 5.5 -> 4.9, K=1024 6.2 -> 5.8; 64 x 128 M=600 N=3072 K=320 6.2 -> 5.2, K=768
// 7.2 -> 6.9, K=1024 7.8 -> 7.7; 32 x 128 M=64 N=7168 K=512 5.0 -> 4.5. From K = 1280 on 64 x 128 loses
// (8.5 vs 8.6), from 2048 on all do (64 x 64 with the weight in the MALL 9.3 vs 9.6).
bool launch_short(int tile, const MmArgs& p, hipStream_t stream) {
    switch (tile) {
        case kLdsSk64x64: return launch_lds<64, 64, 1, 4, 1, 5>(p, stream);
        case kLdsSk64x128: return launch_lds<64, 128, 1, 4, 1, 5>(p, stream);
        case kLdsSk32x128: return launch_lds<32, 128, 1, 4, 1, 5>(p, stream);
        default: return false;
    }
}

}  // namespace feather
