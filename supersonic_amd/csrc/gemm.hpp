// Hand-written bf16 GEMM with a transposed right-hand side for the
// prefill-sized projections: out[m][n] = a[m][k] . w[n][k]^T, fp32
// accumulation, up to three column segments (separate weights and outputs) in
// one launch, optionally batched, with a plain bf16 store or a residual add
// in the epilogue.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace ssa {

enum GemmEpilogue { kGemmStore = 0, kGemmResidualBf16 = 1, kGemmResidualF32 = 2 };

struct GemmArgs {
    int batch = 1, m = 0, k = 0;
    const uint16_t* a = nullptr;  // [batch][m][lda]
    int64_t lda = 0, a_bs = 0;
    int nseg = 1;
    const uint16_t* w[3] = {nullptr, nullptr, nullptr};  // [n_s][k] per segment
    void* out[3] = {nullptr, nullptr, nullptr};          // [m][n_s] per segment
    int n[3] = {0, 0, 0};
    int64_t w_bs = 0, o_bs = 0;  // batch strides (elements) of w and out (segment 0 only when batched)
    int epilogue = kGemmStore;   // residual: out = bf16(out + bf16(a.w^T)), in place (one segment)
    // Optional workspace (zero-filled before its first use; every call leaves
    // each tile's two hand-over counts equal) for splitting the last partial round of tiles along
    // k; without one (or too small) the tail runs whole.
    void* ws = nullptr;
    size_t ws_bytes = 0;
};

// Workspace of a projection's split work: a header of counts at fixed places,
// whatever the shape, then the partials.  Every call leaves the tail's two
// counts of a tile equal and the arrival counters at zero, so calls of
// different shapes can follow each other on one workspace.
constexpr size_t kGemmFlagBytes = 8192;         // tail counts, two per tile (<= 1024 tail tiles)
constexpr size_t kGemmArrivalBytes = 64 << 10;  // split-k arrival counters, one per tile or column block
constexpr size_t kGemmPartOff = kGemmFlagBytes + kGemmArrivalBytes;
// Workspace bytes of the tail split for `tail` tiles.
inline size_t gemm_tail_bytes(int tail) { return kGemmPartOff + static_cast<size_t>(tail) * 8 * 32 * 64 * 16; }

// How a GEMM runs: bm x bn tiles, the last split_tiles of them over ks slices
// of k.  256 x 256 is gemm.hip's kernel (with its own tail split), the others
// gemm_tile.hip's.
struct GemmPlan {
    int bm = 256, bn = 256, ks = 1, split_tiles = 0;
};
GemmPlan gemm_plan(int m, int k, int nseg, const int* n, int batch = 1);
inline size_t gemm_split_bytes(const GemmPlan& p) {
    return p.ks > 1 ? kGemmPartOff + static_cast<size_t>(p.split_tiles) * p.ks * p.bm * p.bn * sizeof(float) : 0;
}
// Workspace bytes of a GEMM of m rows over k and the given column segments on
// a GPU of 256 CUs: the tail split's or the k split's; 0 when it has neither.
size_t gemm_ws_bytes(int m, int k, int nseg, const int* n);
int gemm_tile(hipStream_t st, const GemmArgs& g, const GemmPlan& plan);

// Launches on `st`; 0 on success.  Requires k % 8 == 0 and 16-byte aligned
// rows (lda % 8 == 0).
int gemm_bt(hipStream_t st, const GemmArgs& g);

}  // namespace ssa
