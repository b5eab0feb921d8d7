// Host-side description of one scaled_mm call and the gfx950 kernel variants
// that can serve it.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace feather {

// Shape limits every kernel family relies on: the LDS kernels build per-lane copy offsets within a
// tile in 32 bits, row * K * 2 over at most 256 rows (below 2^31) and (16-K group * N + column) * 16
// over a stage's eight groups at most (unsigned, below 2^32; the kernel asserts both).
constexpr int64_t kMaxK = int64_t{1} << 22;
constexpr int64_t kMaxN = int64_t{1} << 25;

struct MmArgs {
    const uint16_t* a;       // (M, K) fp16 (or bf16 when a_bf16), row-major
    const uint8_t* b;        // (K/16, N, 16) fp8 bytes
    const float* scale;      // device scalar, read when has_scale
    const uint16_t* bias;    // (N,) in the output type, read when has_bias
    uint16_t* c;             // (M, N) fp16 / bf16, row-major
    int64_t M, N, K;
    int has_scale, has_bias;
    bool out_bf16;
    bool b_e4m3;
    bool a_bf16;             // activations are bf16 (converted to fp16 in the kernel; e5m2 weights only)
    int group_m;             // tile raster group height (0 = default)
    int smallm_min_groups;   // small-M: workgroup count the K split aims for (0 = default)
    // rank-R term C += T . U^T: T (M, R), U (N, R)
    const uint16_t* lora_t = nullptr;
    const uint16_t* lora_u = nullptr;
    int64_t lora_rank = 0;
    int lora_dtype = 0;      // 0 none, 1 fp16 factors, 2 bf16 factors
    bool lora_after = false; // added to the finished result, in the output type
};

// Kernel variants. Values are stable: the Python autotuner de-duplicates
// reference configs by the id they map to.
enum KernelId : int {
    kKernelNone = 0,
    // tuple tiles for K % 64 != 0 (served by the tiles of a plan that take any K)
    kTile256x256 = 1,
    kTile256x128 = 2,
    kTile128x256 = 3,
    kTile128x128 = 4,
    kTile64x128 = 5,
    kTile64x64 = 6,
    kSmallM = 10,  // M <= 64: K split inside the workgroup (and across workgroups with a workspace), 16- or 64-column strips
    // LDS-DMA pipelined tiles (K % 64 == 0)
    kLds256x256 = 20,  // both 256 x 256 tuples (2,4,4,8,4) and (4,2,4,4,8)
    kLds256x128 = 22,
    kLds128x256 = 23,
    kLds128x128 = 24,
    kLds256x192 = 25,
    kLds128x384 = 26,
    // LDS-DMA tiles with a K split across workgroups (small shapes)
    kLdsSk64x64 = 30,
    kLdsSk64x128 = 31,
    kLdsSk32x128 = 34,
    // Tiles that only a plan names (feather_scaled_mm_kernel_id reports the class
    // above that a tuple's shape falls into, never one of these)
    kMid32x64 = 40,
    kMid96x64 = 41,
    kMid96x128 = 42,
    kMid64x192 = 43,
    kMid96x192 = 44,
    kMid128x128 = 45,   // 2 x 4 waves, five-stage ring (kLds128x128: 2 x 2 waves, two workgroups per CU)
    kMid128x192 = 46,
    kTail128x256 = 47,  // 128 x 256 for K that is no multiple of 64
};

// Every launcher returns false, and launches nothing, for a variant it does not
// have (bf16 activations are served by the small-M kernel with e5m2 weights only).
// K-split workspace layout, shared by the small-M kernel and the split-K LDS
// tiles: a fixed region of arrival counters (one u32 per output strip or tile)
// that nothing else ever writes, then the fp32 partials. The counter region
// must be zero before the first call and every call leaves it zero again, so
// one workspace serves calls of any shapes in any order (a counter region
// sized per call would overlap an earlier call's partials). A split that would
// need more counters than the region holds is not taken.
constexpr int64_t kWorkspaceCounters = 16384;
constexpr size_t kWorkspaceCounterBytes = static_cast<size_t>(kWorkspaceCounters) * 4;  // 64 KB

// Small-M kernel. With a workspace of at least smallm_workspace_bytes() it
// also splits K across workgroups; without one it splits K inside each
// workgroup only.
// strip: column tiles per strip and ksplit workgroups per strip as a plan chose them; 0: by the
// kernel's own cost model. Without the workspace a split needs, K is split inside the workgroup only.
bool launch_smallm_kernel(const MmArgs& p, void* workspace, size_t workspace_bytes, hipStream_t stream, int strip = 0,
                          int ksplit = 0);
size_t smallm_workspace_bytes(int64_t M, int64_t N, int64_t K, int target_groups);
int smallm_ksplit(int64_t M, int64_t N, int64_t K, int target_groups);
size_t smallm_split_bytes(int64_t M, int64_t N, int strip, int ksplit);
bool launch_lds_kernel(int kernel_id, const MmArgs& p, hipStream_t stream);

struct SplitKPlan {
    int kernel_id;          // 0: not applicable
    int ksplit;
    int tiles;
    size_t workspace_bytes; // counter region + ksplit fp32 partial tiles per output tile
};
SplitKPlan lds_splitk_plan(int64_t M, int64_t N, int64_t K, int target);

// What serves one call: a KernelId, the K split across workgroups and, for the small-M kernel,
// the column tiles per strip (0: that kernel's own choice of both).
struct MmPlan {
    int tile = kKernelNone;
    int ksplit = 1;
    size_t workspace_bytes = 0;
    int strip = 0;
};
// The variant with the least modelled time (scaled_mm_plan.hip): the same for every
// type, so bf16 activations give the bits of their fp16 cast.
MmPlan plan_scaled_mm(int64_t M, int64_t N, int64_t K, int cus);
// The same for a call with a rank-R term: the small-M kernel only where its lean form, which adds it, serves the shape.
MmPlan plan_scaled_mm_lora(int64_t M, int64_t N, int64_t K, int cus);
// The kernel behind a small-M launch: the general kernel on 16-column strips or wider ones, or
// the lean kernel with one workgroup per CU or two.
enum SmallmForm : int { kSmallmStrips = 1, kSmallmWide = 2, kSmallmLean = 3, kSmallmLeanPair = 4 };
SmallmForm smallm_form(int64_t M, int64_t N, int64_t K, int target_groups, int strip, int ksplit);
inline bool is_lean(SmallmForm f) { return f == kSmallmLean || f == kSmallmLeanPair; }
// Counter region + fp32 partial tiles of a K split (0 for ksplit 1).
size_t tile_workspace_bytes(int tile, int64_t M, int64_t N, int ksplit);
// Launches a tile with the given K split; ksplit > 1 needs tile_workspace_bytes() of
// workspace (same contract as launch_smallm_kernel's).
bool launch_tile(int tile, const MmArgs& p, int ksplit, void* workspace, size_t workspace_bytes, hipStream_t stream);
// Whether launch_tile runs a split-K tile on one group of waves, 64 K a stage, instead of two
// groups (calls without a rank-R term): see launch_short.
inline bool short_k_tile(int tile, int64_t K, int ksplit) {
    return (tile == kLdsSk64x64 || tile == kLdsSk64x128 || tile == kLdsSk32x128) && ksplit == 1 && K % 64 == 0 && K <= 1024;
}
bool launch_short(int tile, const MmArgs& p, hipStream_t stream);
int lds_pipe_env();  // FEATHEROPS_LDS_PIPE (1 unless set)
bool launch_mid(int tile, const MmArgs& p, int ksplit, float* partials, uint32_t* counters, hipStream_t stream);

}  // namespace feather
