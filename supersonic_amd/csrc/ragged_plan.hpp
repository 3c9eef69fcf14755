// Chunk length of the ragged decode plan (decode_split.hpp), shared by the
// device plan, the persistent layer's host-side guess of it, and the CPU test.
#pragma once

#include <cstdint>

#if defined(__HIPCC__)
#define SSA_HOST_DEVICE __host__ __device__
#else
#define SSA_HOST_DEVICE
#endif

namespace ssa {

// No chunk grows past this: the growth below multiplies it by items / target a
// step, which four times over leaves 64 bits when sequences * kv heads far
// exceed the target, and the plan divides by it in 32 bits (1024 sequences of
// 4096 tokens, 4 kv heads, 256 workgroups: 2^32, zero as an int).  Lengths are
// below it, so a sequence gets one split either way.
constexpr int64_t kRaggedMaxChunk = int64_t{1} << 30;

SSA_HOST_DEVICE inline int64_t ragged_round_chunk(int64_t c) {
    c = (c + 15) / 16 * 16;
    return c < kRaggedMaxChunk ? c : kRaggedMaxChunk;
}

// chunk = ceil(tot * Hkv / target) rounded up to 16, at least min_chunk.
// Per-sequence rounding can push the item count past the target (a second,
// mostly idle round): the chunk grows in proportion until the items fit (a few
// passes; uniform lengths need none).  items_of(c): the sequences' splits at
// chunk c, times Hkv.  strict: if four growth steps did not get there, one
// split per sequence (longest(): the longest sequence).
template <typename Items, typename Longest>
SSA_HOST_DEVICE inline int ragged_chunk(int64_t tot, int Hkv, int target, int min_chunk, bool strict,
                                        const Items& items_of, const Longest& longest) {
    // (far below the bound: tot is what a cache holds)
    int64_t c = ((tot * Hkv + target - 1) / target + 15) / 16 * 16;
    c = c > min_chunk ? c : min_chunk;
    bool fits = false;
    for (int pass = 0; pass < 5; ++pass) {
        const int64_t items = items_of(c);
        fits = items <= target;
        if (fits || pass == 4) break;
        c = ragged_round_chunk((c * items + target - 1) / target);
    }
    if (strict && !fits) {
        const int64_t l = ragged_round_chunk(longest());
        c = c > l ? c : l;
    }
    return static_cast<int>(c);
}

}  // namespace ssa
