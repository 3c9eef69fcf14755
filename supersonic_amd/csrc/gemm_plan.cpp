// The plan of a tiled product: which tiles, and how k is split.
#include "gemm_plan.hpp"

#include <algorithm>

namespace ssa {

// Picks the tiles and the k split by an estimate of the time in microseconds:
// rounds of workgroups (one a CU; two for the 32- and 64-row tiles, whose
// LDS allows it) of `KT` 64-deep steps each, a constant a round for filling
// the pipeline and the epilogue, a term for the partials of a split, and no
// less than the HBM time of the operands.  The step times (s0 with few
// workgroups, s0 + s1 with every CU busy) were fitted to 2900 timings of the
// Q/K/V and output projections of the 8/2-, 16/4- and 16/2-head layers at 13 to
// 8192 rows (one MI355X), before the copies of weights that one workgroup reads
// passed the caches by; 240 output projections of 1 to 12 rows take 0.85 to 1.28
// times the estimate since.  256 x 256 tiles stay where one round of
// them holds the whole product and k is short (k = 1024, 2000 rows x 5120:
// 37.7 us against 41.6 for 128 x 128).
namespace {
struct TileCost {
    int bm, bn, max_m, slots;
    double s0, s1, round;
};
constexpr int kPlanCus = 256;
constexpr TileCost kTileCosts[] = {
    {256, 256, 0x7fffffff, 1, 1.437, 0.361, 4.32}, {256, 128, 0x7fffffff, 1, 0.617, 0.217, 4.77},
    {128, 128, 0x7fffffff, 1, 0.489, 0.060, 1.74}, {128, 64, 0x7fffffff, 1, 0.336, 0.073, 1.25},
    {64, 64, 600, 2, 0.290, 0.248, 1.25},          {32, 64, 200, 2, 0.192, 0.210, 1.25},
};
// `wgs` workgroups of n steps
double rounds_us(const TileCost& c, int64_t wgs, double n) {
    const int64_t slots = static_cast<int64_t>(kPlanCus) * c.slots, r = wgs / slots, rem = wgs % slots;
    double t = static_cast<double>(r) * (n * (c.s0 + c.s1) + c.round);
    if (rem) {
        const double busy = c.slots > 1 ? (rem > kPlanCus ? 1.0 : 0.0) : static_cast<double>(rem) / kPlanCus;
        t += n * (c.s0 + c.s1 * busy) + c.round;
    }
    return t;
}
}  // namespace

GemmPlan gemm_plan(int m, int k, int nseg, const int* n, int batch, size_t room) {
    GemmPlan best;
    best.us = 1e30;
    if (k <= 0 || k % 8 != 0) return best;  // not a tiled product
    const int KT_steps = (k + 63) / 64;
    double nsum = 0;
    for (int s = 0; s < nseg; ++s) nsum += n[s];
    const double hbm = 2.0 * batch * (nsum * k + static_cast<double>(m) * k + m * nsum) / 5.64e6;
    // split: tiles over ks slices of k, tail: 256 x 256 tiles in two halves
    auto take = [&](const TileCost& c, int ks, int64_t split, int64_t tail, double t, double handicap) {
        t = (std::max(t, hbm) + 1.85) * handicap;
        if (t >= best.us) return;
        const size_t bytes = tail > 0 ? gemm_tail_bytes(static_cast<int>(tail))
                             : ks > 1 ? kGemmPartOff + static_cast<size_t>(split) * ks * c.bm * c.bn * sizeof(float) : 0;
        if (bytes > room) return;
        best = GemmPlan{c.bm, c.bn, ks, static_cast<int>(split), static_cast<int>(tail), bytes, t};
    };
    for (const TileCost& c : kTileCosts) {
        if (m > c.max_m) continue;
        int64_t nt = 0;
        for (int s = 0; s < nseg; ++s) nt += (n[s] + c.bn - 1) / c.bn;
        const int64_t tiles = nt * ((m + c.bm - 1) / c.bm) * batch;
        const int64_t tail = tiles > kPlanCus ? tiles % kPlanCus : 0;
        // Rows of a and w that do not begin on 64 bytes: the copies, which set the
        // pace of the smaller tiles, straddle cache lines.  33 products of k % 32 != 0
        // took 1.19 times these tiles' estimate and 1.07 times the 256 x 256 ones' (5977
        // rows, 3112 -> 7184: 321 us in 256 x 128 tiles, 291 in 256 x 256; the other way
        // round 1134 rows, 6152 -> 20528: 349 and 366).
        const double KT = KT_steps * (c.bn != 256 && k % 32 != 0 ? 1.12 : 1.0);
        if (c.bn == 256) {
            // the last partial round in two halves of k where that is possible, whole
            // where the workspace has no room for it
            if (batch == 1 && tail > 0 && 2 * tail <= kPlanCus && KT_steps >= 4 && gemm_tail_bytes(static_cast<int>(tail)) <= room)
                take(c, 1, 0, tail, rounds_us(c, tiles - tail, KT) + rounds_us(c, 2 * tail, 0.5 * KT) + 7.5, 1.0);
            else
                take(c, 1, 0, 0, rounds_us(c, tiles, KT), 1.0);
            continue;
        }
        // Whole tiles, then a split of every tile, then of the last partial
        // round's; a split has to win 4%, the smaller tiles 2%.
        take(c, 1, 0, 0, rounds_us(c, tiles, KT), 1.02);
        if (batch > 1) continue;
        for (int all = 1; all >= 0; --all) {
            const int64_t split = all ? tiles : tail;
            for (int ks = 2; ks <= (all ? 16 : 8) && split > 0 && KT_steps / ks >= 3 && split * ks <= (all ? 1600 : 600); ++ks) {
                const int kper = (KT_steps + ks - 1) / ks, kk = (KT_steps + kper - 1) / kper;
                const double kb = c.bm * c.bn * 4.0 / 1024.0;  // one slice's partials
                double t = rounds_us(c, split * kk, kper * KT / KT_steps) + 1.4 + 0.0212 * kk * kb + split * kk * kb * 2048.0 / 11.6e6;
                if (!all) t += rounds_us(c, tiles - split, KT);
                take(c, ks, split, 0, t, 1.02 * 1.04);
            }
        }
    }
    return best;
}

// A constant and a time a round of 256 column blocks.  Staged rows: a time a
// load batch of 4096 k and a little for the length, or the HBM time of a round's
// weights, and the staging of the rows; otherwise in proportion to k.  Past k =
// 12288 more than two rounds take 1.35 times that (1 row, 16384 -> 1024 blocks:
// 121 us).  Fitted to the output projections of 1 to 12 rows, k 1024 to 12288, 272
// to 1792 blocks, with weights that come from HBM (copies of them in turn; one
// MI355X).
double stream_us(int m, int k, int64_t ncb, bool staged) {
    const double round = staged ? std::max(3.8 + 4.3 * ((k + 4095) / 4096 - 1) + 0.00027 * k, 0.0013 * k) + 2e-5 * k * (m - 1)
                                : (0.0016 * k + 0.6) * (1.0 + 0.025 * (m - 8));
    return 3.0 + static_cast<double>((ncb + 255) / 256) * round * (k > 12288 && ncb > 512 ? 1.35 : 1.0);
}

}  // namespace ssa
