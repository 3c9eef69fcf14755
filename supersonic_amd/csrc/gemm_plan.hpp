// How a tiled product runs, and the layout of the workspace that its split work
// takes.  Host arithmetic only.
#pragma once

#include <cstddef>
#include <cstdint>

namespace ssa {

// Workspace of a projection's split work: a header of counts at fixed places,
// whatever the shape, then the partials.  Every call leaves the tail's two
// counts of a tile equal and the arrival counters at zero, so calls of
// different shapes can follow each other on one workspace.  (Where the header
// itself moves, behind the normed rows of a Q/K/V call, the call clears its counts.)
constexpr size_t kGemmFlagBytes = 8192;         // tail counts, two per tile (<= 1024 tail tiles)
constexpr size_t kGemmArrivalBytes = 64 << 10;  // split-k arrival counters, one per tile or column block
constexpr size_t kGemmPartOff = kGemmFlagBytes + kGemmArrivalBytes;
// Workspace bytes of the tail split for `tail` tiles.
inline size_t gemm_tail_bytes(int tail) { return kGemmPartOff + static_cast<size_t>(tail) * 8 * 32 * 64 * 16; }

// bm x bn tiles, the last split_tiles of them over ks slices of k (256 x 256,
// gemm.hip's kernel: the last `tail` in two halves of k; the others:
// gemm_tile.hip's).
struct GemmPlan {
    int bm = 256, bn = 256, ks = 1, split_tiles = 0, tail = 0;
    size_t bytes = 0;   // workspace that the split needs
    double us = 0;      // the estimate it was chosen by
};
// For m rows over k and the given column segments on a GPU of 256 CUs; no split
// takes more than `room` bytes of workspace.
GemmPlan gemm_plan(int m, int k, int nseg, const int* n, int batch = 1, size_t room = SIZE_MAX);

// The weight-streaming kernels' time for m <= 12 rows against ncb 16-column blocks
// of W (staged: the rows fit in LDS, the LDS-staged kernel), as GemmPlan::us.
double stream_us(int m, int k, int64_t ncb, bool staged);

}  // namespace ssa
