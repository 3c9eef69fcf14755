// Causal GQA prefill attention on gfx950 MFMA.
//
// Replaces the reference's prefill attention
//   supersonic_qwen35_full_attention_prefill_kernel  kernels/full_attention.hip:246-361
//   (one wave per query row, scalar dot per key, two passes, per-key barriers)
// and, in the fused entry point, the chain around it
//   crates/runner/src/prefill_engine.rs:1951-2308
//   (split q/gate, QK RMSNorm, RoPE, transposes, cache copies, cast, gate).
//
// Kernel design (flash attention forward, fp32 accumulation):
//   workgroup = 128 query rows of one head: 8 compute wave64s of 16 rows and
//   4 copy waves; keys in tiles of 64, double-buffered in LDS and copied
//   global->LDS directly (buffer_load ... lds).  K is copied row-major into
//   padded blocks; V comes from a transposed staging copy (vt_stage_kernel)
//   so the PV operand is one conflict-free ds_read_b128 per MFMA.
//   S^T = K Q^T     v_mfma_f32_16x16x32: A = 16 key rows (LDS), B = Q^T held
//                   in registers for the whole kernel.
//   O^T += V^T P^T  the B operand (P^T) is the lane's own softmax weights.
//   Online softmax in base 2 with a lazy running max (O is rescaled only
//   when a row max grows by more than 2^8); the row sums add the 16-bit
//   weights exactly as the MFMA uses them.
//   Causal: key tiles past the workgroup's last row are never loaded; a wave
//   skips the MFMA work of tiles past its own last row; only tiles that cross
//   the diagonal or the kv_len edge are masked.  Query tiles run longest
//   first, the heads of one kv head on one XCD.
//   Chunks of few items and many keys (a short chunk behind a long prefix) run
//   as pieces of the items' keys, one a CU, with the query heads of a kv head
//   packed into the 128 rows, and prefill_merge_kernel (plan_key_split): 333
//   rows after 7001 cached tokens, 16/2 heads: 147 -> 57 us.
#include <algorithm>
#include <cstdlib>

#include <type_traits>

#include "common.hpp"
#include "kv_view.hpp"

namespace ssa {

struct PrefillParams {
    const uint16_t* q;   // element (b, h, row, d) at b*q_bs + h*q_hs + row*q_rs + d
    int64_t q_bs, q_hs, q_rs;
    KvView kv;           // K/V rows of (b, kv head, token)
    // V^T staging (vt_stage_kernel): element (b, kv head, dim, position) at
    // ((b * Hkv + h) * D + dim) * vt_ld + position
    const uint16_t* vt;
    int vt_ld;
    int Hq, Hkv, G, S, L, off;
    float scale_log2;
    int nqt;             // query tiles of 128 rows (of a query head; with a key split of a kv head)
    int B;               // sequences
    int n_wg;            // workgroups of the persistent grid
    // Dynamic schedule (NULL: the static one).  Per item list x (an XCD's, or
    // the single list) a claim counter at claims[32 x] and a finished-workgroup
    // counter at claims[32 (8 + x)], each on its own 128-byte line; both are
    // zero before a launch and the list's last workgroup to finish zeroes them.
    unsigned* claims;
    // drop-in output: f32, element (b, h, row, d) at b*o_bs + h*o_hs + row*o_rs + d
    float* out_f32;
    int64_t o_bs, o_hs, o_rs;
    // fused: bf16 output [S, Hq*D] with the sigmoid gate; Q prologue
    uint16_t* out_bf16;
    const uint16_t* gate;  // element (h, row, d) at h*q_hs + row*q_rs + d (b = 0)
    const uint16_t* q_norm_w;
    const uint16_t* cos_t;
    const uint16_t* sin_t;
    int half_rot;
    float eps;
    float rescale_slack;  // lazy-rescale slack in log2 units (0 = exact running max)
};

// The same with a key split (a type of its own: the other kernels' arguments
// stay small; with these 64 bytes more every launch took 0.3 us longer).
struct PrefillSplitParams : PrefillParams {
    // A kv head's rows are its G query heads at S
    // positions, R = S * G rows in all, row r = position r / G of query head
    // kvh * G + r % G; an item's key tiles run as pieces of at most `piece`
    // tiles, one piece a workgroup, which leave their sums here for
    // prefill_merge_kernel, by workgroup slot: the unnormalised O in accumulator
    // order ([slot][wave][16-dim block][lane] x 4 floats) and each row's (max, sum).
    int piece;
    int R;
    int lists_log2;      // 1 << lists_log2 item lists (kv heads spread over the XCDs)
    int W;               // workgroups of a list
    int hpl, nb;         // kv heads of a list; items of a query tile in it, hpl * B
    uint32_t g_mul;      // r / G = (2 r * g_mul >> 32) >> g_shift for r < 2^31:
    int g_shift;         // g_mul = ceil(2^(31 + g_shift) / G), g_shift = ceil(log2 G)
    float* part_o;
    float* part_ml;
};
template <bool SPLIT> struct PrefillArgs { typedef PrefillParams t; };
template <> struct PrefillArgs<true> { typedef PrefillSplitParams t; };

template <typename QT> struct Mfma32;
template <> struct Mfma32<bf16_t> {
    typedef bf16x8_v op;
    static __device__ __forceinline__ f32x16_v mma(const op& a, const op& b, const f32x16_v& c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
};
template <> struct Mfma32<f16_t> {
    typedef f16x8_v op;
    static __device__ __forceinline__ f32x16_v mma(const op& a, const op& b, const f32x16_v& c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
};

template <typename OP>
__device__ __forceinline__ OP to_op(const u32x4_v& w) {
    OP r;
    __builtin_memcpy(&r, &w, 16);
    return r;
}

template <typename QT>
__device__ __forceinline__ uint32_t pk2(float a, float b) {
    return Elem<QT>::from_f32(a) | (Elem<QT>::from_f32(b) << 16);
}

typedef short s16x4_v __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2_v __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_v __attribute__((ext_vector_type(2)));

// Two f32 -> packed 16-bit pair with the hardware RNE converters.
template <typename QT> __device__ __forceinline__ uint32_t cvt_pk(float a, float b);
template <> __device__ __forceinline__ uint32_t cvt_pk<bf16_t>(float a, float b) {
    f32x2_v v = {a, b};
    bf16x2_v r = __builtin_convertvector(v, bf16x2_v);
    return __builtin_bit_cast(uint32_t, r);
}
template <> __device__ __forceinline__ uint32_t cvt_pk<f16_t>(float a, float b) {
    f32x2_v v = {a, b};
    f16x2_v r = __builtin_convertvector(v, f16x2_v);
    return __builtin_bit_cast(uint32_t, r);
}

// Two 16-bit ones packed in a word (the A operand of the row-sum MFMA).
template <typename QT> constexpr uint32_t kOnePair = 0x3F803F80u;  // bf16 1.0, 1.0
template <> constexpr uint32_t kOnePair<f16_t> = 0x3C003C00u;       // f16 1.0, 1.0

// Tile geometry.  A K tile is 64 keys x D in LDS.  Copy instruction i
// (i < NR = D/8) of a tile moves rows i, i + NR, i + 2 NR, ... (64/NR rows,
// one 1 KB run) into LDS block i.  K blocks are padded by 8 words so the
// 16-row ds_read_b128 K reads hit distinct banks (SQ_LDS_BANK_CONFLICT is 0
// on gfx950).  Row r lives at (r % NR) * KBLK + (r / NR) * ROWB, so every
// inner-loop LDS offset is an immediate on one per-lane base.
//
// A V tile arrives transposed: D rows (dims) of 64 keys, 128 B each, copy
// instruction i moving dims 8i .. 8i + 7 into block i (1 KB, unpadded).  Dims
// 16 P .. 16 P + 15 fill the 2 KB pair P; inside a pair dim r's 16-byte chunk
// c (keys 8c .. 8c + 7 in staging order) sits at granule 8 r + (c ^ (r >> 1)),
// which spreads the 16 dims one ds_read_b128 of the PV loop touches over all
// 16 granule slots of a 256-byte bank row.
template <int D> struct Tile {
    static constexpr int ROWB = 2 * D;        // bytes per key row
    static constexpr int NR = D / 8;          // copy instructions (= 1 KB blocks) per tile
    static constexpr int KBLK = 1024 + 32;
    static constexpr int KBYTES = NR * KBLK;
    static constexpr int VBYTES = NR * 1024;
    static constexpr int STAGE = KBYTES + VBYTES;
    static constexpr int NI = NR / 4;         // copy instructions per copy wave (K and V each)
    static __device__ __forceinline__ constexpr int koff(int r) { return (r % NR) * KBLK + (r / NR) * ROWB; }
};

// Buffer resource for a tile base that is uniform across the wave (forced
// into SGPRs: the base can come from a block-table load the compiler cannot
// prove uniform).  Reads past `bytes` return zeros.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rsrc(const uint8_t* base, int bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(base);
    const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a >> 32));
    void* u = reinterpret_cast<void*>((static_cast<uint64_t>(hi) << 32) | lo);
    return __builtin_amdgcn_make_buffer_rsrc(u, static_cast<short>(0), bytes, 0x00020000);
}

template <typename QT> struct Mfma16;
template <> struct Mfma16<bf16_t> {
    typedef bf16x8_v op;
    static __device__ __forceinline__ f32x4_v mma(const op& a, const op& b, const f32x4_v& c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
};
template <> struct Mfma16<f16_t> {
    typedef f16x8_v op;
    static __device__ __forceinline__ f32x4_v mma(const op& a, const op& b, const f32x4_v& c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
};

// LDS read lookahead of the K-operand (reads) and V-operand (MFMAs) pipelines
constexpr int kKLA = 8;
constexpr int kVLA = 6;

constexpr int kPrefillWaves = 8;   // compute waves: 8 x 16 query rows = 128 rows
constexpr int kCopyWaves = 4;      // waves that only move K / V^T tiles into LDS
constexpr int kPrefillThreads = 64 * (kPrefillWaves + kCopyWaves);


// One workgroup = 128 query rows of one head: 8 compute waves of 16 rows each
// plus 4 copy waves that only issue the global->LDS tile copies (the copy
// path runs at about 48 B/clk per CU, and a wave that issues copies stalls
// until they are accepted, so compute waves never issue any).  Three waves
// share a SIMD (about 150 registers each); one wave's softmax VALU work
// overlaps another's MFMA chains.
//
//   S^T = K Q^T      v_mfma_f32_16x16x32: A = 16 key rows (LDS), B = Q^T (16
//                    query rows, registers).  C: lane l holds query row l & 15
//                    and keys 16 kb + 4 (l >> 4) + i of key block kb.
//   O^T += V^T P^T   per 32-key step the B operand (P^T) is the lane's own 8
//                    weights (keys 4 g + i of the two 16-key blocks), and the A
//                    operand (V^T) comes from two transposing LDS reads, each
//                    giving a lane 4 consecutive keys of dim (l & 15).
// r / G by a multiplication: a division by a run-time value takes about 40
// dependent instructions, and several of them ahead of an item's first copy
// cost 2 us.
__device__ __forceinline__ int div_g(const PrefillSplitParams& p, int r) {
    return static_cast<int>(__umulhi(2u * static_cast<uint32_t>(r), p.g_mul) >> p.g_shift);
}
// Item m of a list: its order index (query tiles from the last one on) and its
// number within the query tile.
__device__ __forceinline__ void split_item(const PrefillSplitParams& p, int m, int& qi, int& idx) {
    qi = m;
    idx = 0;
    if (p.nb > 1) {
        qi = m / p.nb;
        idx = m - qi * p.nb;
    }
}
// 64-key tiles below the last row's causal limit of query tile qt.
__device__ __forceinline__ int prefill_tiles(const PrefillParams& p, int qt) {
    const int lim = min(p.L, p.off + min(qt * 128 + 128, p.S));
    return lim > 0 ? (lim + 63) / 64 : 0;
}
__device__ __forceinline__ int prefill_tiles(const PrefillSplitParams& p, int qt) {
    return (min(p.L, p.off + div_g(p, min(qt * 128 + 128, p.R) - 1) + 1) + 63) / 64;
}
// Pieces that n key tiles run as.
__host__ __device__ __forceinline__ int prefill_pieces(int n, int piece) { return n > piece ? (n + piece - 1) / piece : 1; }

// Slots of one list before its order index qi (query tiles from the last one
// on), `nb` items a query tile; for the whole wave.
__device__ __forceinline__ int prefill_slots_before(const PrefillSplitParams& p, int qi, int nb) {
    const int lane = threadIdx.x & 63;
    int n = 0;
    for (int i = lane; i < qi; i += 64) n += prefill_pieces(prefill_tiles(p, p.nqt - 1 - i), p.piece);
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) n += __shfl_xor(n, o);
    return __builtin_amdgcn_readfirstlane(n) * nb;
}
// The piece in slot j of a list: order index of its query tile, its number
// within the query tile's pieces; false past the last.
__device__ __forceinline__ bool prefill_find_piece(const PrefillSplitParams& p, int j, int nb, int& qi, int& at) {
    const int lane = threadIdx.x & 63;
    int before = 0;
    for (int base = 0; base < p.nqt; base += 64) {
        const int i = base + lane;
        const int np = i < p.nqt ? prefill_pieces(prefill_tiles(p, p.nqt - 1 - i), p.piece) * nb : 0;
        int incl = np;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int x = __shfl_up(incl, o);
            incl += lane >= o ? x : 0;
        }
        const uint64_t hit = __ballot(before + incl > j);
        if (hit) {
            const int l = static_cast<int>(__builtin_ctzll(hit));
            qi = __builtin_amdgcn_readfirstlane(base + l);
            at = __builtin_amdgcn_readfirstlane(j - before - __shfl(incl - np, l));
            return true;
        }
        before += __builtin_amdgcn_readfirstlane(__shfl(incl, 63));
    }
    return false;
}

// SPLIT: one piece of an item a workgroup (PrefillParams::piece).
template <typename QT, int D, bool FUSED, bool SPLIT>
__global__ __launch_bounds__(kPrefillThreads) void prefill_kernel(typename PrefillArgs<SPLIT>::t p) {
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass only needs the launch stub
    typedef typename Mfma16<QT>::op op_t;
    typedef Tile<D> T;
    constexpr int KS = D / 32;        // QK^T k-steps (32 dims each)
    constexpr int DBK = D / 16;       // 16-dim output blocks
    // [stage][K | V] tiles; the fused prologue stages the query rows in one stage
    __shared__ __attribute__((aligned(1024))) uint8_t lds[2 * T::STAGE];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: copy offsets stay in SGPRs
    // Persistent grid (one workgroup per CU), items longest first.  When the
    // heads split evenly over the 8 XCDs (workgroup i runs on XCD i % 8), each
    // XCD has its own item list holding the heads that share its kv heads, so
    // its L2 keeps their K/V.  Workgroup j of a list of W takes items j,
    // 2W-1-j, 2W+j, ...: a long item pairs with a short one and every
    // workgroup gets about the same number of key tiles.  With a key split the
    // lists hold kv heads, several XCDs to a list when there are fewer than 8.
    const int bid = blockIdx.x;
    const int hpx = p.Hq / 8;
    const bool by_xcd = !SPLIT && hpx > 0 && (p.Hq % 8) == 0 && (p.n_wg % 8) == 0;
    int list, j, W;
    if constexpr (SPLIT) {
        const int ll = p.lists_log2;
        list = bid & ((1 << ll) - 1);
        j = ll ? ((bid >> 3) << (3 - ll)) + ((bid & 7) >> ll) : bid;
        W = p.W;
    } else {
        list = by_xcd ? (bid & 7) : 0;
        j = by_xcd ? (bid >> 3) : bid;
        W = by_xcd ? (p.n_wg >> 3) : p.n_wg;
    }
    const int hpi = by_xcd ? hpx : p.Hq;     // heads per item list
    int n_items = p.nqt * hpi * p.B;
    if constexpr (SPLIT) n_items = p.nqt * p.nb;
    // Key split: this workgroup's one piece, tiles [pt0, pt1) of item pm.
    int pm = 0, pt0 = 0, pt1 = 0;
    // one item, in a loop that the compiler takes for a loop: straight-line, it
    // moves the epilogue's values across the key loop (54 spilled registers)
    int one = 1;
    if constexpr (SPLIT) asm volatile("" : "+s"(one));
    if constexpr (SPLIT) {
        int qi, at;
        if (!prefill_find_piece(p, j, p.nb, qi, at)) return;  // the whole workgroup
        const int n = prefill_tiles(p, p.nqt - 1 - qi);
        const int pn = prefill_pieces(n, p.piece);
        int part, idx;
        split_item(p, at, part, idx);
        pm = qi * p.nb + idx;
        pt0 = n * part / pn;
        pt1 = n * (part + 1) / pn;
    }
    // Dynamic schedule: the list's items are claimed one at a time from a
    // counter in list order (longest first), so workgroups that start late
    // (their CUs busy with other work when the grid was dispatched) take only
    // what is left.  The first copy wave claims item r + 1 during item r and
    // leaves it in claimed[(r + 1) & 1]; every reader is at least one
    // workgroup barrier behind the write.
    __shared__ int claimed[2];
    const bool dyn = !SPLIT && p.claims != nullptr;
    unsigned* const ctr = dyn ? p.claims + 32 * list : nullptr;
    auto claim_next = [&](const int slot) {
        if (wave == kPrefillWaves && (tid & 63) == 0) {
            claimed[slot] = static_cast<int>(__hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the write is in LDS before the next barrier
        }
    };
    // Item r of this workgroup (false past the last): 128 query rows `qt` of
    // head h (SPLIT: kv head h) of sequence b over key tiles [t0, t1).  The
    // sequence of m is increasing (static schedule).
    auto item_at = [&](const int r, int& qt, int& h, int& b, int& t0, int& t1) -> bool {
        if (SPLIT && r >= one) return false;
        const int m = SPLIT ? pm : (dyn ? claimed[r & 1] : ((r & 1) ? (r + 1) * W - 1 - j : r * W + j));
        if (m >= n_items) return false;
        if constexpr (SPLIT) {
            int qi, idx;
            split_item(p, m, qi, idx);
            qt = p.nqt - 1 - qi;
            b = p.B > 1 ? idx / p.hpl : 0;
            h = list * p.hpl + idx - b * p.hpl;
            t0 = pt0;
            t1 = pt1;
        } else {
            qt = p.nqt - 1 - m / (hpi * p.B);
            const int rem = m % (hpi * p.B);
            h = (by_xcd ? (bid & 7) * hpx : 0) + rem % hpi;
            b = rem / hpi;
            t0 = 0;
            t1 = prefill_tiles(p, qt);
        }
        return true;
    };
    // Tiles alternate between the two LDS stages across items: tile `it` of
    // an item that follows gt tiles goes to stage (gt + it + 1) & 1, so the
    // next item's first tile can be copied while this item's last tile is
    // computed, and the fused query staging of an item uses stage gt & 1 (its
    // previous item's last tile, read by then).
    //
    // Copy waves: the next tile is issued once every wave has passed the
    // barrier of tile it (the stage it goes to was last read by tile it - 1)
    // and has landed by the next barrier.  Same barrier count per item as the
    // compute waves (one per tile plus the item end).
    auto copy_items = [&]() {
        const int lane = tid & 63;
        const int dma_lane = (lane / (D / 8)) * T::NR * T::ROWB + (lane % (D / 8)) * 16;
        const int vt_rowb = 2 * p.vt_ld;
        const int vt_lane0 = (lane >> 3) * vt_rowb + 16 * ((lane & 7) ^ (lane >> 4));
        const int vt_lane1 = (lane >> 3) * vt_rowb + 16 * ((lane & 7) ^ (4 + (lane >> 4)));
        // Direct global->LDS copy of key tile `it` of (h, b) into stage `st`
        // (asynchronous, counted by vmcnt).  K: lane l of copy instruction i
        // moves 16 bytes of row i + NR (l / (D/8)); rows past kv_len fall
        // outside the buffer range and read as zeros (masked later; never
        // stale cache contents).  V^T: lane l of instruction i moves chunk
        // c = (l & 7) ^ (4 (i & 1) + (l >> 4)) of dim 8 i + (l >> 3) (the
        // swizzle of the tile geometry); the staging buffer is zero past kv_len.
        auto issue_tile = [&](const int h, const int b, const int it, const int st) {
            const int kvh = SPLIT ? h : h / p.G;
            const uint16_t* vt_head = p.vt + (static_cast<int64_t>(b) * p.Hkv + kvh) * D * p.vt_ld;
            const int k0 = it * 64;
            const int64_t base = p.kv.row_uniform(b, kvh, k0, D) * 2;  // a tile lies inside one page
            const __amdgpu_buffer_rsrc_t kr = tile_rsrc(p.kv.k + base, min(64, p.L - k0) * T::ROWB);
            const __amdgpu_buffer_rsrc_t vr = tile_rsrc(reinterpret_cast<const uint8_t*>(vt_head + k0),
                                                        D * vt_rowb - 2 * k0);
            const int cw = wave - kPrefillWaves;
            const int lbase = __builtin_amdgcn_readfirstlane(st * T::STAGE + cw * T::NI * T::KBLK);
            const int vbase = __builtin_amdgcn_readfirstlane(st * T::STAGE + T::KBYTES + cw * T::NI * 1024);
#pragma unroll
            for (int jj = 0; jj < T::NI; ++jj) {
                const int i = cw * T::NI + jj;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(kr, (__attribute__((address_space(3))) void*)(lds + lbase + jj * T::KBLK),
                                                         16, dma_lane, i * T::ROWB, 0, 0);
                __builtin_amdgcn_raw_ptr_buffer_load_lds(vr, (__attribute__((address_space(3))) void*)(lds + vbase + jj * 1024),
                                                         16, (i & 1) ? vt_lane1 : vt_lane0, 8 * i * vt_rowb, 0, 0);
            }
        };
        // s_waitcnt vmcnt(0) alone (the other counters are not waited for)
        auto wait_vm0 = []() { __builtin_amdgcn_s_waitcnt(0 | (7 << 4) | (15 << 8)); };
        // first tile of the first item that has keys at all
        auto issue_first = [&](int r, const int st) {
            int qt, h, b, t0, t1;
            for (; item_at(r, qt, h, b, t0, t1); ++r) {
                if (t1 > t0) {
                    issue_tile(h, b, t0, st);
                    return;
                }
                if (dyn) return;  // only item r is claimed yet (and every item has tiles)
            }
        };
        issue_first(0, 1);
        int gt = 0, qt, h, b, t0, t1;
        for (int r = 0; item_at(r, qt, h, b, t0, t1); ++r) {
            const int nt = t1 - t0;
            // The next item is claimed as this one nears its end (at the
            // barrier of tile nt - 3, two barriers before the other copy
            // waves read the claim), so workgroups claim in the order they
            // finish: longest-processing-time-first.  Items of fewer than 3
            // tiles claim at their start.
            if (dyn && nt < 3) claim_next((r + 1) & 1);
            for (int it = 0; it < nt; ++it) {
                // Tile `it` has landed.  The compute waves' barrier also
                // orders their LDS reads; these waves read no LDS, so a bare
                // barrier (no implied wait for every load in flight) is enough.
                wait_vm0();
                __builtin_amdgcn_s_barrier();
                if (dyn && nt >= 3 && it == nt - 3) claim_next((r + 1) & 1);
                if (it + 1 < nt) issue_tile(h, b, t0 + it + 1, (gt + it + 2) & 1);
                else issue_first(r + 1, (gt + nt + 1) & 1);
            }
            __builtin_amdgcn_s_barrier();  // item end (the next tile needs no wait yet)
            gt += nt;
        }
        wait_vm0();  // no LDS write in flight when the workgroup ends
        if (dyn && wave == kPrefillWaves && (tid & 63) == 0) {
            // This workgroup's claims are over (its last one failed); the
            // list's last workgroup to get here leaves both counters at zero.
            unsigned* const done = ctr + 32 * 8;
            if (__hip_atomic_fetch_add(done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == static_cast<unsigned>(W)) {
                __hip_atomic_store(ctr, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(done, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    };
    // One work item = 128 query rows of one head (SPLIT: kv head) of one
    // sequence, run by the compute waves over key tiles [t0, t1); gt = tiles of
    // the workgroup's items before it.  A `return` inside ends the item, not
    // the workgroup.
    auto run_item = [&](const int qt, const int h, const int b, const int t0, const int t1, const int gt) {
    // position and query head of a row
    auto pos_of = [&](const int row) -> int {
        if constexpr (SPLIT) return div_g(p, row);
        else return row;
    };
    auto head_of = [&](const int row, const int ps) -> int { return SPLIT ? h * p.G + row - ps * p.G : h; };
    // Opaque per item, so the compiler does not hoist lane-derived values and
    // loads (norm weights, offsets) out of the item loop, where they would
    // stay live through the key loop.
    int lane = tid & 63;
    asm volatile("" : "+v"(lane));
    const int g4 = lane >> 4;
    const int q0 = qt * 128;
    const int row_w0 = q0 + 16 * wave;
    const int myrow = row_w0 + (lane & 15);
    int R = p.S;
    if constexpr (SPLIT) R = p.R;
    const int L = p.L, off = p.off;
    const bool row_ok = myrow < R;

    const int ntiles = t1 - t0;
    const int lim_wave = min(L, off + (SPLIT ? pos_of(min(row_w0 + 16, R) - 1) + 1 : min(row_w0 + 16, R)));
    const int first_lim = off + pos_of(row_w0) + 1;  // causal limit of the wave's first row
    const int mypos = pos_of(row_ok ? myrow : 0);
    const int lim_row = min(L, off + (SPLIT ? mypos : myrow) + 1);  // (rows past R: anything)
    const int64_t q_row = head_of(row_ok ? myrow : 0, mypos) * p.q_hs + static_cast<int64_t>(mypos) * p.q_rs;

    // ------------------------------------------------ Q^T operand (registers)
    // B operand of S^T = K Q^T: lane holds query row (lane & 15), dims 32 s + 8 g4 + j.
    op_t qb[KS];
    if constexpr (!FUSED) {
        const uint16_t* qrow = p.q + b * p.q_bs + q_row;
#pragma unroll
        for (int s = 0; s < KS; ++s)
            qb[s] = to_op<op_t>(row_ok ? ld16(qrow + 32 * s + 8 * g4) : u32x4_v{0u, 0u, 0u, 0u});
    } else if (p.half_rot % 32 == 0 || p.half_rot == 16) {
        // This wave's 16 query rows normed and rotated in the operand layout
        // itself: lane holds row myrow, dims 32 s + 8 g4 + j (64 of the row's
        // dims), RMSNorm with (1 + w) over the row (the four lanes l, l ^ 16,
        // l ^ 32, l ^ 48 hold it), then rotate-half RoPE at position off + row,
        // bf16 after each step (prefill_engine.rs:2025-2096).  A RoPE partner
        // (dim d +- half_rot) is in the same lane, chunk s +- half_rot / 32,
        // when half_rot is a multiple of 32, or in lane ^ 32, same chunk, when
        // it is 16.  Every global load is issued before any arithmetic.
        const int hr = p.half_rot;
        const int hs = hr / 32;                  // rotary chunks per half (0 for half_rot 16)
        const int pos = off + mypos;
        const uint16_t* qrow = p.q + q_row;
        u32x4_v raw[KS], wv[KS], cw[KS / 2], sw[KS / 2];
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            raw[s] = row_ok ? ld16(qrow + 32 * s + 8 * g4) : u32x4_v{0u, 0u, 0u, 0u};
            wv[s] = ld16(p.q_norm_w + 32 * s + 8 * g4);
        }
#pragma unroll
        for (int c = 0; c < KS / 2; ++c) {
            cw[c] = sw[c] = u32x4_v{0u, 0u, 0u, 0u};
            const int ci = hr == 16 ? 8 * (g4 & 1) : 32 * c + 8 * g4;  // table column of the chunk
            if (c < (hr == 16 ? 1 : hs)) {
                cw[c] = ld16(p.cos_t + static_cast<int64_t>(pos) * hr + ci);
                sw[c] = ld16(p.sin_t + static_cast<int64_t>(pos) * hr + ci);
            }
        }
        float ss = 0.f;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            float x[8];
            unpack8<bf16_t>(raw[s], x);
#pragma unroll
            for (int j = 0; j < 8; ++j) ss += x[j] * x[j];
        }
        ss = xor32_sum(xor16_sum(ss));
        const float inv = rsqrtf(ss / static_cast<float>(D) + p.eps);
        u32x4_v nq[KS];
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            float x[8], w[8];
            unpack8<bf16_t>(raw[s], x);
            unpack8<bf16_t>(wv[s], w);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                nq[s][j] = cvt_pk<bf16_t>(x[2 * j] * inv * (w[2 * j] + 1.0f), x[2 * j + 1] * inv * (w[2 * j + 1] + 1.0f));
        }
        // out = x cos + sg y sin on the normed bf16 values (sg = -1 in the first half)
        auto rot8 = [&](const u32x4_v& xv, const u32x4_v& yv, const u32x4_v& cv, const u32x4_v& sv, const float sg) {
            float x[8], y[8], cs[8], sn[8];
            unpack8<bf16_t>(xv, x);
            unpack8<bf16_t>(yv, y);
            unpack8<bf16_t>(cv, cs);
            unpack8<bf16_t>(sv, sn);
            u32x4_v o;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                o[j] = cvt_pk<bf16_t>(x[2 * j] * cs[2 * j] + sg * y[2 * j] * sn[2 * j],
                                      x[2 * j + 1] * cs[2 * j + 1] + sg * y[2 * j + 1] * sn[2 * j + 1]);
            return o;
        };
        // chunks s < 2 HS rotate with partner chunk s +- HS (a compile-time
        // index for each HS, so the arrays stay in registers)
        auto rope_hs = [&](auto hs_c) {
            constexpr int HS = decltype(hs_c)::value;
            u32x4_v o[2 * HS];
#pragma unroll
            for (int s = 0; s < 2 * HS; ++s)
                o[s] = s < HS ? rot8(nq[s], nq[s + HS], cw[s], sw[s], -1.0f)
                              : rot8(nq[s], nq[s - HS], cw[s - HS], sw[s - HS], 1.0f);
#pragma unroll
            for (int s = 0; s < 2 * HS; ++s) nq[s] = o[s];
        };
        if (hr == 16) {
            u32x4_v y;
#pragma unroll
            for (int j = 0; j < 4; ++j) y[j] = static_cast<uint32_t>(__shfl_xor(static_cast<int>(nq[0][j]), 32));
            nq[0] = rot8(nq[0], y, cw[0], sw[0], g4 < 2 ? -1.0f : 1.0f);
        } else {
            static_assert(KS / 2 <= 4, "head_dim up to 256");
            switch (hs) {
            case 1: rope_hs(std::integral_constant<int, 1>{}); break;
            case 2: if constexpr (KS / 2 >= 2) rope_hs(std::integral_constant<int, 2>{}); break;
            case 3: if constexpr (KS / 2 >= 3) rope_hs(std::integral_constant<int, 3>{}); break;
            case 4: if constexpr (KS / 2 >= 4) rope_hs(std::integral_constant<int, 4>{}); break;
            default: break;
            }
        }
#pragma unroll
        for (int s = 0; s < KS; ++s) qb[s] = to_op<op_t>(nq[s]);
    } else {
            // This wave's 16 query rows: RMSNorm with (1 + w) and rotate-half RoPE
            // at position off + row, bf16 after each step (prefill_engine.rs:2025-2096),
            // (lane c of a row holds dims 8c .. 8c+7); every global load is issued
            // before any arithmetic.  The rows are staged in LDS (stage 0), where
            // the RoPE partner dims are read back and the operand is read
            // transposed.
            uint16_t* qs = reinterpret_cast<uint16_t*>(lds + (gt & 1) * T::STAGE) + wave * 16 * D;
            constexpr int LPR = D / 8;              // lanes per row, 16 B each
            constexpr int RPI = 64 / LPR;           // rows per instruction
            constexpr int NIN = 16 / RPI;           // instructions per wave
            const int c = lane % LPR, rr = lane / LPR;
            const int hr = p.half_rot;              // a multiple of 16 (checked on the host)
            const bool rot = 8 * c < 2 * hr;
            const u32x4_v wtw = ld16(p.q_norm_w + 8 * c);
            u32x4_v qw[NIN], cw[NIN], sw[NIN];
    #pragma unroll
            for (int k = 0; k < NIN; ++k) {
                const int row = row_w0 + k * RPI + rr;
                qw[k] = cw[k] = sw[k] = u32x4_v{0u, 0u, 0u, 0u};
                if (row < R) {
                    const int ps = pos_of(row);
                    qw[k] = ld16(p.q + head_of(row, ps) * p.q_hs + static_cast<int64_t>(ps) * p.q_rs + 8 * c);
                    if (rot) {
                        const int64_t ti = static_cast<int64_t>(off + ps) * hr + (8 * c < hr ? 8 * c : 8 * c - hr);
                        cw[k] = ld16(p.cos_t + ti);
                        sw[k] = ld16(p.sin_t + ti);
                    }
                }
            }
            float wt[8];
            unpack8<bf16_t>(wtw, wt);
            // RMSNorm: the row's sum of squares over its LPR lanes on the VALU
            // (DPP within 16 lanes, a permlane swap across 16), no LDS traffic.
            u32x4_v nq[NIN];
    #pragma unroll
            for (int k = 0; k < NIN; ++k) {
                float x[8];
                unpack8<bf16_t>(qw[k], x);
                float ss = 0.f;
    #pragma unroll
                for (int j = 0; j < 8; ++j) ss += x[j] * x[j];
                if constexpr (LPR >= 16) {
                    ss = row16_sum(ss);
                    if constexpr (LPR == 32) ss = xor16_sum(ss);
                } else {
    #pragma unroll
                    for (int o = 1; o < LPR; o <<= 1) ss += __shfl_xor(ss, o);
                }
                const float inv = rsqrtf(ss / static_cast<float>(D) + p.eps);
    #pragma unroll
                for (int j = 0; j < 4; ++j)
                    nq[k][j] = cvt_pk<bf16_t>(x[2 * j] * inv * (wt[2 * j] + 1.0f), x[2 * j + 1] * inv * (wt[2 * j + 1] + 1.0f));
                st16(qs + (k * RPI + rr) * D + 8 * c, nq[k]);
            }
            if (hr > 0) {
                // RoPE: the rotating lanes read their partner's 8 normed dims back
                // (all reads are issued before any write; LDS is in order per wave).
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                const int pc = 8 * c < hr ? 8 * c + hr : 8 * c - hr;
                u32x4_v yq[NIN];
    #pragma unroll
                for (int k = 0; k < NIN; ++k)
                    yq[k] = rot ? ld16(qs + (k * RPI + rr) * D + pc) : u32x4_v{0u, 0u, 0u, 0u};
                if (rot) {
    #pragma unroll
                    for (int k = 0; k < NIN; ++k) {
                        float x[8], y[8], cs[8], sn[8];
                        unpack8<bf16_t>(nq[k], x);
                        unpack8<bf16_t>(yq[k], y);
                        unpack8<bf16_t>(cw[k], cs);
                        unpack8<bf16_t>(sw[k], sn);
                        const float sg = 8 * c < hr ? -1.0f : 1.0f;
                        u32x4_v o;
    #pragma unroll
                        for (int j = 0; j < 4; ++j)
                            o[j] = cvt_pk<bf16_t>(x[2 * j] * cs[2 * j] + sg * y[2 * j] * sn[2 * j],
                                               x[2 * j + 1] * cs[2 * j + 1] + sg * y[2 * j + 1] * sn[2 * j + 1]);
                        st16(qs + (k * RPI + rr) * D + 8 * c, o);
                    }
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    #pragma unroll
            for (int s = 0; s < KS; ++s) qb[s] = to_op<op_t>(ld16(qs + (lane & 15) * D + 32 * s + 8 * g4));
    }

    f32x4_v oacc[DBK];
#pragma unroll
    for (int d = 0; d < DBK; ++d) oacc[d] = f32x4_v{0.f, 0.f, 0.f, 0.f};
    float m_run = -1e30f;
    // Row sums on the MFMA pipe: lacc += ones * P^T sums each query's 16-bit
    // weights exactly as the PV product uses them (every lane ends up with
    // its own row's total in lacc[0]; the four entries are equal).
    f32x4_v lacc = {0.f, 0.f, 0.f, 0.f};
    const op_t ones = to_op<op_t>(u32x4_v{kOnePair<QT>, kOnePair<QT>, kOnePair<QT>, kOnePair<QT>});
    const float c2 = p.scale_log2;

    // Per-lane LDS bases: K row (lane & 15), dims 8 g4 (for r < 16,
    // koff(r + 16 m) - koff(r) does not depend on r, so the other rows are the
    // compile-time offsets koff(16 m)).  V^T: dim (lane & 15) of each pair,
    // chunk 4 u + g4 of 32-key step u (swizzled granule).
    const int kbase_off = T::koff(lane & 15) + 16 * g4;
    const int vx = (lane & 15) >> 1;
    const int vrd0 = T::KBYTES + 16 * (8 * (lane & 15) + (g4 ^ vx));
    const int vrd1 = T::KBYTES + 16 * (8 * (lane & 15) + ((4 + g4) ^ vx));
    for (int it = 0; it < ntiles; ++it) {
        const int k0 = (t0 + it) * 64;
        const int st = (gt + it + 1) & 1;
        __syncthreads();                // the copy waves' tile `it` has landed; stage st^1 is free again
        if (k0 >= lim_wave) continue;   // the whole tile is past this wave's rows

        const uint8_t* kl = lds + st * T::STAGE + kbase_off;
        const uint8_t* vl0 = lds + st * T::STAGE + vrd0;
        const uint8_t* vl1 = lds + st * T::STAGE + vrd1;

        // S^T = K Q^T, four 16-key blocks.
        f32x4_v sacc[4];
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) sacc[kb] = f32x4_v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < KS; ++s) {
#pragma unroll
            for (int kb = 0; kb < 4; ++kb) {
                const op_t ka = to_op<op_t>(ld16(kl + T::koff(16 * kb) + 64 * s));
                sacc[kb] = Mfma16<QT>::mma(ka, qb[s], sacc[kb]);
            }
        }
        __builtin_amdgcn_sched_group_barrier(0x100, kKLA, 0);
#pragma unroll
        for (int i = 0; i < 4 * KS - kKLA; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, kKLA, 0);
        __builtin_amdgcn_sched_barrier(0);

        // Online softmax, base 2, exact running max.  Lane holds row myrow and
        // keys k0 + 16 kb + 4 g4 + i.
        const bool need_mask = (k0 + 64 > first_lim) || (k0 + 64 > L);
        if (need_mask) {
            // Only tiles crossing the diagonal or kv_len: a real branch (the
            // empty volatile asm keeps the compiler from if-converting it).
            asm volatile("" ::: "memory");
            const int rem = lim_row - (k0 + 4 * g4);  // key 16 kb + i is valid iff < rem
#pragma unroll
            for (int kb = 0; kb < 4; ++kb)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (16 * kb + i >= rem) sacc[kb][i] = -INFINITY;
        }
        float mx = max3_raw(sacc[0][0], sacc[0][1], sacc[0][2]);
        mx = max3_raw(mx, sacc[0][3], sacc[1][0]);
        mx = max3_raw(mx, sacc[1][1], sacc[1][2]);
        mx = max3_raw(mx, sacc[1][3], sacc[2][0]);
        mx = max3_raw(mx, sacc[2][1], sacc[2][2]);
        mx = max3_raw(mx, sacc[2][3], sacc[3][0]);
        mx = max3_raw(mx, sacc[3][1], sacc[3][2]);
        mx = max3_raw(mx, sacc[3][3], sacc[3][3]);
        mx = xor16_max(mx);
        mx = xor32_max(mx) * c2;
        if (__any(mx > m_run + p.rescale_slack)) {
            const float m_new = fmaxf(m_run, mx);
            const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
            m_run = m_new;
#pragma unroll
            for (int i = 0; i < 4; ++i) lacc[i] *= alpha;
#pragma unroll
            for (int d = 0; d < DBK; ++d)
#pragma unroll
                for (int i = 0; i < 4; ++i) oacc[d][i] *= alpha;
        }
        const float m_use = m_run;
        op_t pk[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            u32x4_v w;
#pragma unroll
            for (int hb = 0; hb < 2; ++hb)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const float a = __builtin_amdgcn_exp2f(fmaf(sacc[2 * u + hb][2 * j], c2, -m_use));
                    const float c = __builtin_amdgcn_exp2f(fmaf(sacc[2 * u + hb][2 * j + 1], c2, -m_use));
                    w[2 * hb + j] = cvt_pk<QT>(a, c);
                }
            pk[u] = to_op<op_t>(w);
        }
        __builtin_amdgcn_sched_barrier(0);

        // O^T += V^T P^T: two 32-key steps.  A operand: dims 16 d + (lane & 15),
        // the 8 keys of staging chunk 4 u + g4, which are exactly the keys
        // 32 u + 4 g4 + {0..3} and 32 u + 16 + 4 g4 + {0..3} that the lane's
        // B operand (P^T) carries.
#pragma unroll
        for (int u = 0; u < 2; ++u) {
#pragma unroll
            for (int d = 0; d < DBK; ++d) {
                const op_t va = to_op<op_t>(ld16((u ? vl1 : vl0) + 2048 * d));
                oacc[d] = Mfma16<QT>::mma(va, pk[u], oacc[d]);
            }
            lacc = Mfma16<QT>::mma(ones, pk[u], lacc);
        }
        __builtin_amdgcn_sched_group_barrier(0x100, kVLA, 1);
#pragma unroll
        for (int i = 0; i < 2 * DBK - kVLA; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 1);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 1);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, kVLA, 1);
    }

    __syncthreads();                    // item end (the copy waves' last barrier)
    // ------------------------------------------------ epilogue
    // O^T C layout: lane holds row myrow, dims 16 d + 4 g4 + i.
    // the lane index afresh (mbcnt), so that no new value stays live through
    // the key loop, which runs at the register limit
    int ln = static_cast<int>(__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)));
    if constexpr (SPLIT) {
        asm volatile("" : "+v"(ln));  // not computed ahead of the key loop
        // the piece's sums as they are, for prefill_merge_kernel (with the gate
        // epilogue here too, for items of one piece, the compiler spilled 54
        // registers)
        const int64_t slot = list * W + j;
        float* po = p.part_o + (slot * kPrefillWaves + wave) * DBK * 256;
        if (row_w0 < R) {
#pragma unroll
            for (int d = 0; d < DBK; ++d) *reinterpret_cast<f32x4_v*>(po + d * 256 + ln * 4) = oacc[d];
            if (ln < 16) *reinterpret_cast<f32x2_v*>(p.part_ml + (slot * 128 + 16 * wave + ln) * 2) = f32x2_v{m_run, lacc[0]};
        }
        return;
    }
    const float l_tot = lacc[0];
    const float inv = l_tot > 0.f ? 1.0f / l_tot : 0.f;
    if constexpr (!FUSED) {
        if (!row_ok) return;
        float* orow = p.out_f32 + b * p.o_bs + h * p.o_hs + static_cast<int64_t>(myrow) * p.o_rs;
#pragma unroll
        for (int d = 0; d < DBK; ++d) {
            f32x4_v o = {oacc[d][0] * inv, oacc[d][1] * inv, oacc[d][2] * inv, oacc[d][3] * inv};
            *reinterpret_cast<f32x4_v*>(orow + 16 * d + 4 * g4) = o;
        }
    } else {
        // bf16(attn) * sigmoid(gate), bf16 out [S, Hq*D] (prefill_engine.rs:2263-2308).
        // The accumulator layout gives a lane 8 bytes of each of 16 rows, so
        // the rows go through the wave's own LDS rows (the stage the next
        // item stages its queries in; its tiles are read by now) and the gate
        // loads and output stores move 16 contiguous bytes a lane: row
        // k RPI + rr, dims 8c .. 8c+7.  16-byte chunks are XOR-swizzled by
        // row, so the 16 rows of a write land in different banks.
        constexpr int LPR = D / 8, RPI = 64 / LPR, NIN = 16 / RPI, CM = LPR - 1;
        const int c = ln % LPR, rr = ln / LPR, g4e = ln >> 4;
        u32x4_v gq[NIN];
#pragma unroll
        for (int k = 0; k < NIN; ++k) {
            const int row = min(row_w0 + k * RPI + rr, R - 1);
            gq[k] = ld16(p.gate + h * p.q_hs + static_cast<int64_t>(row) * p.q_rs + 8 * c);
        }
        uint8_t* const os = lds + ((gt + ntiles) & 1) * T::STAGE + wave * 16 * D * 2;
        const int r16 = ln & 15;
#pragma unroll
        for (int d = 0; d < DBK; ++d) {
            const int ch = 2 * d + (g4e >> 1);
            const u32x2_v a = {cvt_pk<bf16_t>(oacc[d][0] * inv, oacc[d][1] * inv),
                               cvt_pk<bf16_t>(oacc[d][2] * inv, oacc[d][3] * inv)};
            *reinterpret_cast<u32x2_v*>(os + r16 * D * 2 + ((ch ^ (r16 & CM)) * 16) + (g4e & 1) * 8) = a;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int k = 0; k < NIN; ++k) {
            const int rl = k * RPI + rr, row = row_w0 + rl;
            const u32x4_v av = ld16(os + rl * D * 2 + ((c ^ (rl & CM)) * 16));
            u32x4_v o;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float r2[2];
#pragma unroll
                for (int hh = 0; hh < 2; ++hh) {
                    const float a = bf16_bits_to_f32(hh ? av[e] >> 16 : av[e] & 0xFFFFu);
                    const float g = bf16_bits_to_f32(hh ? gq[k][e] >> 16 : gq[k][e] & 0xFFFFu);
                    // sigmoid(g) = 1 / (1 + 2^(-g log2 e)), hardware exp2 and reciprocal
                    r2[hh] = a * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-g * kLog2e));
                }
                o[e] = cvt_pk<bf16_t>(r2[0], r2[1]);
            }
            if (row < R) st16(p.out_bf16 + static_cast<int64_t>(row) * p.Hq * D + h * D + 8 * c, o);
        }
    }
    };

    // Separate loops for the copy and the compute waves (same items, same
    // barrier count per item), so neither keeps the other's registers live.
    if (dyn) {
        claim_next(0);
        __builtin_amdgcn_s_barrier();  // item 0's claim is visible to every wave
    }
    if (wave >= kPrefillWaves) {
        copy_items();
    } else {
        int gt = 0, qt, h, b, t0, t1;
        for (int r = 0; item_at(r, qt, h, b, t0, t1); ++r) {
            run_item(qt, h, b, t0, t1, gt);
            gt += t1 - t0;
        }
    }
#endif
}

// Merge of a key split's pieces, and the epilogue: workgroup (item, 16-row
// block of a compute wave), its four waves a quarter of the dims each, in the
// layout the pieces left (16-byte accesses, lane-contiguous).  Pieces are
// added in key order.  Bound by reading the pieces' sums (128 KB a piece at
// D 256, at most one piece a CU).
template <int D, bool FUSED>
__global__ __launch_bounds__(256) void prefill_merge_kernel(PrefillSplitParams p) {
    constexpr int DBK = D / 16, DW = DBK / 4;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int list = blockIdx.x & ((1 << p.lists_log2) - 1), wb = blockIdx.y;
    const int nb = p.nb, W = p.W;
    int qi, idx;
    split_item(p, blockIdx.x >> p.lists_log2, qi, idx);
    const int qt = p.nqt - 1 - qi;
    const int np = prefill_pieces(prefill_tiles(p, qt), p.piece);
    const int row0 = qt * 128 + 16 * wb;
    if (row0 >= p.R) return;
    const int64_t slot0 = list * W + prefill_slots_before(p, qi, nb) + idx;
    const float* ml = p.part_ml + (slot0 * 128 + 16 * wb + (lane & 15)) * 2;
    const float* po = p.part_o + ((slot0 * kPrefillWaves + wb) * DBK + wave * DW) * 256 + lane * 4;
    const int64_t step = static_cast<int64_t>(nb) * kPrefillWaves * DBK * 256;
    f32x4_v acc[DW];
#pragma unroll
    for (int d = 0; d < DW; ++d) acc[d] = f32x4_v{0.f, 0.f, 0.f, 0.f};
    float l_tot = 0.f, mx = -1e30f;
    // Four pieces at a time, every load issued ahead of the arithmetic (past
    // the last piece the last one again, with no weight).
    constexpr int NP = 4;
    for (int i0 = 0; i0 < np; i0 += NP) {
        f32x2_v v[NP];
        f32x4_v o[NP][DW];
#pragma unroll
        for (int u = 0; u < NP; ++u) {
            const int64_t i = min(i0 + u, np - 1);
            v[u] = *reinterpret_cast<const f32x2_v*>(ml + i * nb * 256);
#pragma unroll
            for (int d = 0; d < DW; ++d) o[u][d] = *reinterpret_cast<const f32x4_v*>(po + i * step + d * 256);
        }
        float m_new = mx;
#pragma unroll
        for (int u = 0; u < NP; ++u) m_new = fmaxf(m_new, v[u][0]);
        const float a = __builtin_amdgcn_exp2f(mx - m_new);
        mx = m_new;
        l_tot *= a;
#pragma unroll
        for (int d = 0; d < DW; ++d)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[d][e] *= a;
#pragma unroll
        for (int u = 0; u < NP; ++u) {
            if (i0 + u >= np) break;
            const float w = __builtin_amdgcn_exp2f(v[u][0] - m_new);
            l_tot += v[u][1] * w;
#pragma unroll
            for (int d = 0; d < DW; ++d)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[d][e] += o[u][d][e] * w;
        }
    }
    const int row = row0 + (lane & 15), g4 = lane >> 4;
    if (row >= p.R) return;
    const float inv = l_tot > 0.f ? 1.0f / l_tot : 0.f;
    const int b = p.B > 1 ? idx / p.hpl : 0, kvh = list * p.hpl + idx - b * p.hpl;
    const int ps = div_g(p, row), h = kvh * p.G + row - ps * p.G;
#pragma unroll
    for (int d = 0; d < DW; ++d) {
        const int dim = 16 * (wave * DW + d) + 4 * g4;
        if constexpr (!FUSED) {
            *reinterpret_cast<f32x4_v*>(p.out_f32 + b * p.o_bs + h * p.o_hs + static_cast<int64_t>(ps) * p.o_rs + dim) =
                f32x4_v{acc[d][0] * inv, acc[d][1] * inv, acc[d][2] * inv, acc[d][3] * inv};
        } else {
            const u32x2_v gw = *reinterpret_cast<const u32x2_v*>(p.gate + h * p.q_hs + static_cast<int64_t>(ps) * p.q_rs + dim);
            u32x2_v o;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                float r2[2];
#pragma unroll
                for (int hh = 0; hh < 2; ++hh) {
                    const float a = bf16_round(acc[d][2 * e + hh] * inv);
                    const float g = bf16_bits_to_f32(hh ? gw[e] >> 16 : gw[e] & 0xFFFFu);
                    r2[hh] = a * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-g * kLog2e));
                }
                o[e] = cvt_pk<bf16_t>(r2[0], r2[1]);
            }
            *reinterpret_cast<u32x2_v*>(p.out_bf16 + (static_cast<int64_t>(ps) * p.Hq + h) * D + dim) = o;
        }
    }
}

// ----------------------------------------------------------------------------
// fp32 prefill (drop-in dtype 1): one wave per query row, online softmax.
// ----------------------------------------------------------------------------
__global__ __launch_bounds__(256) void prefill_f32_kernel(const float* q, const float* k, const float* v, float* out,
                                                          int B, int Hq, int Hkv, int S, int L, int D, int G,
                                                          float scale, int off) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= B * Hq * S) return;
    const int qp = row % S, h = (row / S) % Hq, b = row / (S * Hq);
    const int kvh = h / G;
    const int lim = min(L, off + qp + 1);
    const float* qr = q + static_cast<int64_t>(row) * D;
    const float* kb = k + (static_cast<int64_t>(b) * Hkv + kvh) * L * D;
    const float* vb = v + (static_cast<int64_t>(b) * Hkv + kvh) * L * D;
    float qv[8], acc[8];
    for (int e = 0; e < 8; ++e) {
        const int d = lane + 64 * e;
        qv[e] = d < D ? qr[d] : 0.f;
        acc[e] = 0.f;
    }
    float m = -1e30f, l = 0.f;
    for (int t = 0; t < lim; ++t) {
        float part = 0.f;
        for (int e = 0; e < 8; ++e) {
            const int d = lane + 64 * e;
            if (d < D) part += qv[e] * kb[static_cast<int64_t>(t) * D + d];
        }
        const float s = wave_sum(part) * scale;
        const float mn = fmaxf(m, s);
        const float a = expf(m - mn), w = expf(s - mn);
        l = l * a + w;
        for (int e = 0; e < 8; ++e) {
            const int d = lane + 64 * e;
            acc[e] = acc[e] * a + (d < D ? w * vb[static_cast<int64_t>(t) * D + d] : 0.f);
        }
        m = mn;
    }
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    for (int e = 0; e < 8; ++e) {
        const int d = lane + 64 * e;
        if (d < D) out[static_cast<int64_t>(row) * D + d] = acc[e] * inv;
    }
}

// ----------------------------------------------------------------------------
// V^T staging for the prefill kernel.  The PV product needs, per lane, 8
// consecutive keys of one dim; the cache stores token rows.  This pass writes
// each kv head's V transposed, dims as rows of vt_ld positions (kv_len rounded
// up to 64, zero past kv_len), with the keys of every 32-key group stored in
// the order the S^T accumulator hands them to the PV MFMA: position
// 8 g + j holds key 4 g + j for j < 4 and key 16 + 4 g + (j - 4) for j >= 4.
// One workgroup per (64-key tile, kv head, sequence).
// ----------------------------------------------------------------------------
__device__ __forceinline__ constexpr int vt_key_of_position(int p) {
    return (p & ~31) + ((p & 4) ? 16 : 0) + 4 * ((p & 31) >> 3) + (p & 3);
}

template <int D>
__global__ __launch_bounds__(256) void vt_stage_kernel(KvView kv, uint16_t* vt, int Hkv, int L, int ld) {
    __shared__ __attribute__((aligned(16))) uint16_t tile[64][D + 8];
    const int t0 = blockIdx.x * 64, h = blockIdx.y, b = blockIdx.z;
    for (int idx = threadIdx.x; idx < 64 * (D / 8); idx += 256) {
        const int r = idx / (D / 8), c = idx % (D / 8);
        const int t = t0 + r;
        u32x4_v w = {0u, 0u, 0u, 0u};
        if (t < L) w = ld16(reinterpret_cast<const uint16_t*>(kv.v) + kv.row(b, h, t, D) + 8 * c);
        *reinterpret_cast<u32x4_v*>(&tile[r][8 * c]) = w;
    }
    __syncthreads();
    uint16_t* dst = vt + (static_cast<int64_t>(b) * Hkv + h) * D * ld + t0;
    for (int idx = threadIdx.x; idx < D * 8; idx += 256) {
        const int d = idx >> 3, c = idx & 7;
        u32x4_v w;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            w[j] = static_cast<uint32_t>(tile[vt_key_of_position(8 * c + 2 * j)][d]) |
                   (static_cast<uint32_t>(tile[vt_key_of_position(8 * c + 2 * j + 1)][d]) << 16);
        st16(dst + static_cast<int64_t>(d) * ld + 8 * c, w);
    }
}

// Fused prefill, bf16 cache: one pass that appends the chunk's new tokens to
// the cache and does vt_stage_kernel's work for every position.  One
// workgroup per (64-position tile, kv head); lane c of a row holds dims
// 8c .. 8c + 7 (16-byte accesses).  New tokens (position >= off): K gets
// RMSNorm with (1 + w) and rotate-half RoPE (bf16 after each step, RoPE
// partners read back through an LDS row), K and V go to the cache, and V to
// the LDS tile; prefix positions read V back from the cache; the tile is then
// written out transposed in the PV operand's key order.
struct KvStageParams {
    const uint16_t* k_new;  // [S, Hkv*D]
    const uint16_t* v_new;
    const uint16_t* k_norm_w;
    const uint16_t* cos_t;
    const uint16_t* sin_t;
    KvView kv;
    uint16_t* vt;           // [Hkv, D, ld]
    uint16_t* kst;          // fp8 cache: bf16 K rows [Hkv, ld, D] for the attention kernel
    int S, Hkv, off, L, ld, half_rot;
    float eps;
};

constexpr int kKvStageWaves = 16;  // 4 per SIMD: the rows' memory round trips overlap

// One row's e4m3 codes with the per-(token, head) absmax scale, as the fused
// decode append writes them (full_attention_4b.hip:5228-5281, OCP codec): the
// row's LPR lanes hold 8 values each; returns the lane's 8 codes, sets sc.
template <int LPR>
__device__ __forceinline__ u32x2_v quantize_row8(const float (&x)[8], float& sc) {
    float am = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) am = fmaxf(am, fabsf(x[e]));
#pragma unroll
    for (int m = 1; m < LPR; m <<= 1) am = fmaxf(am, __shfl_xor(am, m));
    sc = fmaxf(am / 448.0f, 1e-12f);
    const float inv = 1.0f / sc;
    return u32x2_v{f32x4_to_fp8x4(x[0] * inv, x[1] * inv, x[2] * inv, x[3] * inv),
                   f32x4_to_fp8x4(x[4] * inv, x[5] * inv, x[6] * inv, x[7] * inv)};
}

// 8 e4m3 codes times their row scale, rounded to bf16.
__device__ __forceinline__ u32x4_v dequant8_bf16(u32x2_v w, float sc) {
    u32x4_v r;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const f32x2_v lo = fp8x2_to_f32(w[i], false);
        const f32x2_v hi = fp8x2_to_f32(w[i], true);
        r[2 * i] = pk2<bf16_t>(lo[0] * sc, lo[1] * sc);
        r[2 * i + 1] = pk2<bf16_t>(hi[0] * sc, hi[1] * sc);
    }
    return r;
}

template <int D, bool FP8>
__global__ __launch_bounds__(64 * kKvStageWaves) void kv_stage_kernel(KvStageParams p) {
    __shared__ __attribute__((aligned(16))) uint16_t vtile[64][D + 8];
    constexpr int LPR = D / 8;          // lanes per row
    constexpr int RPI = 64 / LPR;       // rows per wave instruction
    __shared__ __attribute__((aligned(16))) uint16_t krow[kKvStageWaves][RPI][D];  // per-wave RoPE exchange
    const int t0 = blockIdx.x * 64, h = blockIdx.y;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int c = lane % LPR;
    const int hr = p.half_rot;
    const bool rot = 8 * c < 2 * hr;
    float wt[8];
    unpack8<bf16_t>(ld16(p.k_norm_w + 8 * c), wt);
    for (int r0 = wave * RPI; r0 < 64; r0 += kKvStageWaves * RPI) {
        const int r = r0 + lane / LPR;
        const int pos = t0 + r;
        u32x4_v vw = {0u, 0u, 0u, 0u};
        if (pos < p.L) {
            const int64_t o = p.kv.row(0, h, pos, D) + 8 * c;
            if (pos >= p.off) {
                const int64_t src = (static_cast<int64_t>(pos - p.off) * p.Hkv + h) * D + 8 * c;
                const u32x4_v kw = ld16(p.k_new + src);
                vw = ld16(p.v_new + src);
                u32x4_v cw4 = {0u, 0u, 0u, 0u}, sw4 = {0u, 0u, 0u, 0u};
                if (rot) {
                    const int64_t ti = static_cast<int64_t>(pos) * hr + (8 * c < hr ? 8 * c : 8 * c - hr);
                    cw4 = ld16(p.cos_t + ti);
                    sw4 = ld16(p.sin_t + ti);
                }
                float x[8];
                unpack8<bf16_t>(kw, x);
                float ss = 0.f;
#pragma unroll
                for (int e = 0; e < 8; ++e) ss += x[e] * x[e];
                // the row's LPR lanes are aligned groups of the wave
#pragma unroll
                for (int m = 1; m < LPR; m <<= 1) ss += __shfl_xor(ss, m);
                const float inv = rsqrtf(ss / static_cast<float>(D) + p.eps);
                u32x4_v nq;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    nq[e] = pk2<bf16_t>(x[2 * e] * inv * (wt[2 * e] + 1.0f), x[2 * e + 1] * inv * (wt[2 * e + 1] + 1.0f));
                st16(&krow[wave][lane / LPR][8 * c], nq);
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                if (rot) {
                    const int pc = 8 * c < hr ? 8 * c + hr : 8 * c - hr;
                    float xn[8], y[8], cs[8], sn[8];
                    unpack8<bf16_t>(nq, xn);
                    unpack8<bf16_t>(ld16(&krow[wave][lane / LPR][pc]), y);
                    unpack8<bf16_t>(cw4, cs);
                    unpack8<bf16_t>(sw4, sn);
                    const float sg = 8 * c < hr ? -1.0f : 1.0f;
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        nq[e] = pk2<bf16_t>(xn[2 * e] * cs[2 * e] + sg * y[2 * e] * sn[2 * e],
                                            xn[2 * e + 1] * cs[2 * e + 1] + sg * y[2 * e + 1] * sn[2 * e + 1]);
                }
                if constexpr (!FP8) {
                    st16(reinterpret_cast<uint16_t*>(p.kv.k) + o, nq);
                    st16(reinterpret_cast<uint16_t*>(p.kv.v) + o, vw);
                } else {
                    // the attention reads this chunk's K and V unquantised (the
                    // reference runs prefill in bf16 and quantises the cache
                    // afterwards); the cache gets the e4m3 codes and scales
                    st16(p.kst + (static_cast<int64_t>(h) * p.ld + pos) * D + 8 * c, nq);
                    float xk[8], xv[8], sk, sv;
                    unpack8<bf16_t>(nq, xk);
                    unpack8<bf16_t>(vw, xv);
                    const u32x2_v qk8 = quantize_row8<LPR>(xk, sk);
                    const u32x2_v qv8 = quantize_row8<LPR>(xv, sv);
                    *reinterpret_cast<u32x2_v*>(p.kv.k + o) = qk8;
                    *reinterpret_cast<u32x2_v*>(p.kv.v + o) = qv8;
                    if (c == 0) {
                        const int64_t so = p.kv.srow(0, h, pos);
                        p.kv.ks[so] = sk;
                        p.kv.vs[so] = sv;
                    }
                }
            } else if constexpr (!FP8) {
                vw = ld16(reinterpret_cast<const uint16_t*>(p.kv.v) + o);
            } else {
                // prefix from the fp8 cache: codes times scale, as bf16
                const int64_t so = p.kv.srow(0, h, pos);
                st16(p.kst + (static_cast<int64_t>(h) * p.ld + pos) * D + 8 * c,
                     dequant8_bf16(*reinterpret_cast<const u32x2_v*>(p.kv.k + o), p.kv.ks[so]));
                vw = dequant8_bf16(*reinterpret_cast<const u32x2_v*>(p.kv.v + o), p.kv.vs[so]);
            }
        }
        st16(&vtile[r][8 * c], vw);
    }
    __syncthreads();
    uint16_t* dst = p.vt + static_cast<int64_t>(h) * D * p.ld + t0;
    for (int idx = threadIdx.x; idx < D * 8; idx += 64 * kKvStageWaves) {
        const int d = idx >> 3, cc = idx & 7;
        u32x4_v w;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            w[j] = static_cast<uint32_t>(vtile[vt_key_of_position(8 * cc + 2 * j)][d]) |
                   (static_cast<uint32_t>(vtile[vt_key_of_position(8 * cc + 2 * j + 1)][d]) << 16);
        st16(dst + static_cast<int64_t>(d) * p.ld + 8 * cc, w);
    }
}

// Stages V^T for `B` sequences of `L` keys into the prefill workspace slot of
// `device` and points `p` at it.  Returns hipSuccess or the failing error.
static hipError_t stage_vt(int device, hipStream_t st, const KvView& kv, int B, int Hkv, int L, int D,
                           PrefillParams& p) {
    const int ld = (L + 63) / 64 * 64;
    const size_t bytes = static_cast<size_t>(B) * Hkv * D * ld * 2;
    void* ws = device_workspace(device, bytes, kWorkspacePrefill);
    if (!ws) return hipErrorOutOfMemory;
    p.vt = static_cast<const uint16_t*>(ws);
    p.vt_ld = ld;
    const dim3 grid(ld / 64, Hkv, B);
    uint16_t* vt = static_cast<uint16_t*>(ws);
    switch (D) {
    case 64: hipLaunchKernelGGL(vt_stage_kernel<64>, grid, dim3(256), 0, st, kv, vt, Hkv, L, ld); break;
    case 128: hipLaunchKernelGGL(vt_stage_kernel<128>, grid, dim3(256), 0, st, kv, vt, Hkv, L, ld); break;
    case 256: hipLaunchKernelGGL(vt_stage_kernel<256>, grid, dim3(256), 0, st, kv, vt, Hkv, L, ld); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// ----------------------------------------------------------------------------
// Host side
// ----------------------------------------------------------------------------
// Key split: when a query head's 128-row items leave CUs without work, or with
// one short item each, the items run as pieces over the kv heads' rows.
constexpr int kSplitMinTiles = 4;  // key tiles a piece has at least
static size_t prefill_part_bytes(int D, int n_wg) { return static_cast<size_t>(n_wg) * 128 * (D + 2) * sizeof(float); }
// Chunks whose workspace holds room for a key split: at most 8192 tokens of the
// kv heads (at 4 query heads a kv head one 128-row item a CU), and keys for
// pieces that win more than their merge costs.
static bool prefill_may_split(size_t S, size_t L, size_t Hkv) {
    return S * Hkv <= 8192 && L > 2 * 64 * kSplitMinTiles;
}

// Room for a key split's sums where the caller gave none (NULL: the chunk runs
// whole): a library buffer of one size, so that it never moves, apart from the
// staging's, so that the split never makes that one move.  While `st` is captured
// only a buffer that is there already.
static void* pieces_workspace(int device, hipStream_t st, size_t* bytes) {
    *bytes = prefill_part_bytes(256, std::max(device_cu_count(device), 256));
    return stream_capturing(st) ? device_workspace_held(device, *bytes, kWorkspacePieces)
                                : device_workspace(device, *bytes, kWorkspacePieces);
}

// Fills in p's split (piece 0: none) for n workgroups.  The estimates are in
// microseconds (one MI355X, D 256): a tile takes 1.25 with up to half the CUs
// busy, and with all of them 1.4 in items of falling length but 2.0 in equal
// pieces; a split costs 11 more (its sums to memory, and the merge).  Measured,
// whole call, 16/4 heads: 64 rows after 8000 cached tokens 157 -> 45 us, 333
// rows 168 -> 70, 300 after 1000 39 -> 32, 1000 after 16000 348 -> 272; left
// whole: 1000 rows of a prompt 35.5 (split 37.6), 1500 after 1000 68.8 (75.6).
// At D 64 and 128, where a tile costs less, the rule leaves whole what it should
// (67 and 64 random chunks: 0.56 and 0.63 of the whole walk's time on average, the
// best choice 0.56 and 0.62, none slower than two runs differ by).
static void plan_key_split(PrefillSplitParams& p, int n) {
    p.piece = 0;
    const int lists = n % 8 ? 1 : (p.Hkv % 8 == 0 ? 8 : (8 % p.Hkv == 0 ? p.Hkv : 1));
    p.lists_log2 = lists == 8 ? 3 : (lists == 4 ? 2 : (lists == 2 ? 1 : 0));
    p.W = n / lists;
    p.hpl = p.Hkv / lists;
    p.nb = p.hpl * p.B;
    p.g_shift = 0;
    while ((1 << p.g_shift) < p.G) ++p.g_shift;
    p.g_mul = static_cast<uint32_t>(((1ull << (31 + p.g_shift)) + p.G - 1) / p.G);
    if (static_cast<int64_t>(p.S) * p.G > 0x3fffffff) return;
    p.R = p.S * p.G;
    const int nqt = (p.R + 127) / 128;
    if (static_cast<int64_t>(nqt) * p.nb > p.W) return;
    auto tiles = [&](int qt) {
        const int64_t lim = std::min<int64_t>(p.L, static_cast<int64_t>(p.off) + (std::min(qt * 128 + 128, p.R) - 1) / p.G + 1);
        return static_cast<int>((lim + 63) / 64);
    };
    auto pieces = [&](int c) {
        int64_t t = 0;
        for (int qt = 0; qt < nqt; ++qt) t += prefill_pieces(tiles(qt), c);
        return t * p.nb;
    };
    const int longest = tiles(nqt - 1);
    int lo = kSplitMinTiles, hi = longest;  // the least piece whose pieces fit one round
    while (lo < hi) {
        const int c = (lo + hi) / 2;
        if (pieces(c) <= p.W) hi = c;
        else lo = c + 1;
    }
    const double busy = std::min(1.0, static_cast<double>(p.nqt) * p.Hq * p.B / n);
    const double busy_s = static_cast<double>(pieces(lo)) / p.W;
    const double whole = longest * (1.25 + 0.3 * std::max(0.0, busy - 0.5));
    const double split = lo * (1.25 + 1.5 * std::max(0.0, busy_s - 0.5)) + 11.0;
    if (split + 2.0 < whole) {
        p.piece = lo;
        p.nqt = nqt;
        p.n_wg = n;
    }
}

template <typename QT, int D, bool FUSED>
static hipError_t launch_prefill_d(hipStream_t st, const PrefillSplitParams& p) {
    const dim3 grid(static_cast<unsigned>(p.n_wg)), blk(kPrefillThreads);
    if (!p.piece) {
        hipLaunchKernelGGL((prefill_kernel<QT, D, FUSED, false>), grid, blk, 0, st, static_cast<const PrefillParams&>(p));
        return hipGetLastError();
    }
    hipLaunchKernelGGL((prefill_kernel<QT, D, FUSED, true>), grid, blk, 0, st, p);
    const dim3 mgrid(static_cast<unsigned>(p.nqt * p.Hkv * p.B), kPrefillWaves);
    hipLaunchKernelGGL((prefill_merge_kernel<D, FUSED>), mgrid, dim3(256), 0, st, p);
    return hipGetLastError();
}

// Persistent grid: one workgroup per CU (a workgroup's LDS allows no second
// one), a multiple of 8 so the XCD-aware item lists stay aligned, and never
// more workgroups than items.  part: room of part_bytes for a key split's sums,
// or NULL for none.
template <typename QT, bool FUSED>
static hipError_t launch_prefill(int device, int D, hipStream_t st, PrefillSplitParams& p, void* part, size_t part_bytes,
                                 int free_wgs = 0) {
    const int items = p.nqt * p.Hq * p.B;
    int n = device_cu_count(device);
    if (n <= 0) n = 256;
    n = n >= 8 ? n & ~7 : n;
    p.n_wg = items < n ? items : n;
    p.piece = 0;
    // beside a decode (dynamic schedule) the pieces share the CUs it leaves
    const int ns = p.claims ? std::min(free_wgs, n) & ~7 : n;
    if (part && ns >= 8 && part_bytes >= prefill_part_bytes(D, ns)) plan_key_split(p, ns);
    p.part_ml = static_cast<float*>(part);
    p.part_o = p.part_ml + (part ? static_cast<size_t>(ns) * 256 : 0);
    switch (D) {
    case 64: return launch_prefill_d<QT, 64, FUSED>(st, p);
    case 128: return launch_prefill_d<QT, 128, FUSED>(st, p);
    case 256: return launch_prefill_d<QT, 256, FUSED>(st, p);
    default: return hipErrorInvalidValue;
    }
}

static float rescale_slack() {
    const char* v = getenv("SUPERSONIC_PREFILL_RESCALE_SLACK");
    return (v && *v) ? static_cast<float>(atof(v)) : 8.0f;
}

int prefill_dropin(int dtype, size_t device, size_t B, size_t Hq, size_t Hkv, size_t q_len, size_t kv_len, size_t D,
                   size_t groups, float scale, size_t off, const void* q, const void* k, const void* v, void* out) {
    if (dtype != 0 && dtype != 1 && dtype != 2) return 64;
    if (D == 0 || D > 512 || Hkv == 0 || groups == 0 || Hq != Hkv * groups) return 14;
    if (dtype != 1 && D != 64 && D != 128 && D != 256) {
        // General head size (the reference takes any D <= 512): D <= 256 runs
        // the MFMA kernel on copies zero-padded to the next native tile (the
        // zero dims add nothing to q.k, and the padded output dims are dropped);
        // larger D runs the f32 kernel on f32 copies.
        ScopedDevice scoped(static_cast<int>(device));
        if (B == 0 || Hq == 0 || q_len == 0) return hipDeviceSynchronize() == hipSuccess ? 0 : 12;
        const int64_t nq = static_cast<int64_t>(B * Hq * q_len), nk = static_cast<int64_t>(B * Hkv * kv_len);
        const int d = static_cast<int>(D);
        ScratchBuffers sb;
        int rc;
        if (D <= 256) {
            const int dp = D <= 64 ? 64 : (D <= 128 ? 128 : 256);
            void* qp = sb.get(nq * dp * 2);
            void* kp = sb.get(nk * dp * 2);
            void* vp = sb.get(nk * dp * 2);
            void* op = sb.get(nq * dp * 4);
            if (!qp || !kp || !vp || !op) return 2;
            if (repack_rows(dtype, dtype, q, qp, nq, 1, d, 0, d, dp, nullptr) != hipSuccess ||
                repack_rows(dtype, dtype, k, kp, nk, 1, d, 0, d, dp, nullptr) != hipSuccess ||
                repack_rows(dtype, dtype, v, vp, nk, 1, d, 0, d, dp, nullptr) != hipSuccess)
                return 11;
            rc = prefill_dropin(dtype, device, B, Hq, Hkv, q_len, kv_len, dp, groups, scale, off, qp, kp, vp, op);
            if (rc == 0 && repack_rows(1, 1, op, out, nq, 1, dp, 0, d, d, nullptr) != hipSuccess) rc = 11;
        } else {
            void* qf = sb.get(nq * d * 4);
            void* kf = sb.get(nk * d * 4);
            void* vf = sb.get(nk * d * 4);
            if (!qf || !kf || !vf) return 2;
            if (repack_rows(dtype, 1, q, qf, nq, 1, d, 0, d, d, nullptr) != hipSuccess ||
                repack_rows(dtype, 1, k, kf, nk, 1, d, 0, d, d, nullptr) != hipSuccess ||
                repack_rows(dtype, 1, v, vf, nk, 1, d, 0, d, d, nullptr) != hipSuccess)
                return 11;
            rc = prefill_dropin(1, device, B, Hq, Hkv, q_len, kv_len, D, groups, scale, off, qf, kf, vf, out);
        }
        if (hipDeviceSynchronize() != hipSuccess && rc == 0) rc = 12;
        return rc;
    }
    ScopedDevice scoped(static_cast<int>(device));
    if (B == 0 || Hq == 0 || q_len == 0) return hipDeviceSynchronize() == hipSuccess ? 0 : 12;
    if (dtype == 1) {
        const size_t rows = B * Hq * q_len;
        hipLaunchKernelGGL(prefill_f32_kernel, dim3(grid1d(rows, 4)), dim3(256), 0, 0,
                           static_cast<const float*>(q), static_cast<const float*>(k), static_cast<const float*>(v),
                           static_cast<float*>(out), static_cast<int>(B), static_cast<int>(Hq),
                           static_cast<int>(Hkv), static_cast<int>(q_len), static_cast<int>(kv_len),
                           static_cast<int>(D), static_cast<int>(groups), scale, static_cast<int>(off));
        if (hipGetLastError() != hipSuccess) return 11;
        if (hipDeviceSynchronize() != hipSuccess) return 12;
        return 0;
    }
    PrefillSplitParams p{};
    p.q = static_cast<const uint16_t*>(q);
    p.q_rs = static_cast<int64_t>(D);
    p.q_hs = static_cast<int64_t>(q_len) * D;
    p.q_bs = static_cast<int64_t>(Hq) * q_len * D;
    p.kv.k = static_cast<uint8_t*>(const_cast<void*>(k));
    p.kv.v = static_cast<uint8_t*>(const_cast<void*>(v));
    p.kv.page_size = 1;
    p.kv.head_stride = static_cast<int64_t>(kv_len) * D;
    p.kv.seq_stride = static_cast<int64_t>(Hkv) * kv_len * D;
    p.Hq = static_cast<int>(Hq);
    p.Hkv = static_cast<int>(Hkv);
    p.G = static_cast<int>(groups);
    p.S = static_cast<int>(q_len);
    p.L = static_cast<int>(kv_len);
    p.off = static_cast<int>(off);
    p.scale_log2 = scale * kLog2e;
    p.rescale_slack = rescale_slack();
    p.nqt = static_cast<int>((q_len + 127) / 128);
    p.out_f32 = static_cast<float*>(out);
    p.o_rs = p.q_rs;
    p.o_hs = p.q_hs;
    p.o_bs = p.q_bs;
    p.B = static_cast<int>(B);
    const int dev = static_cast<int>(device);
    void* part = nullptr;
    size_t part_bytes = 0;
    if (prefill_may_split(q_len * B, kv_len, Hkv)) part = pieces_workspace(dev, nullptr, &part_bytes);
    if (kv_len > 0 && stage_vt(dev, nullptr, p.kv, static_cast<int>(B), static_cast<int>(Hkv), static_cast<int>(kv_len),
                               static_cast<int>(D), p) != hipSuccess)
        return 11;
    const hipError_t e = dtype == 0 ? launch_prefill<f16_t, false>(dev, static_cast<int>(D), nullptr, p, part, part_bytes)
                                    : launch_prefill<bf16_t, false>(dev, static_cast<int>(D), nullptr, p, part, part_bytes);
    if (e != hipSuccess) return 11;
    if (hipDeviceSynchronize() != hipSuccess) return 12;
    return 0;
}

}  // namespace ssa

using namespace ssa;

extern "C" int supersonic_qwen35_hip_full_attention_prefill(
    int dtype, size_t device_ordinal, size_t batch_size, size_t q_heads, size_t kv_heads, size_t q_len,
    size_t kv_len, size_t head_dim, size_t num_kv_groups, float scale, size_t seqlen_offset, const void* query,
    const void* key, const void* value, void* out) {
    return prefill_dropin(dtype, device_ordinal, batch_size, q_heads, kv_heads, q_len, kv_len, head_dim,
                          num_kv_groups, scale, seqlen_offset, query, key, value, out);
}

extern "C" int supersonic_qwen35_4b_hip_full_attention_prefill(
    int dtype, size_t device_ordinal, size_t batch_size, size_t q_heads, size_t kv_heads, size_t q_len,
    size_t kv_len, size_t head_dim, size_t num_kv_groups, float scale, size_t seqlen_offset, const void* query,
    const void* key, const void* value, void* out) {
    return prefill_dropin(dtype, device_ordinal, batch_size, q_heads, kv_heads, q_len, kv_len, head_dim,
                          num_kv_groups, scale, seqlen_offset, query, key, value, out);
}

// The part of a prefill workspace that a call cannot do without: the V^T
// staging, and the bf16 K rows of an fp8 cache.
size_t ssa::prefill_stage_bytes(int kv_dtype, size_t kv_heads, size_t head_dim, size_t chunk_len, size_t chunk_start) {
    const size_t L = chunk_start + chunk_len;
    if (L > 0x7FFFFFFF || kv_heads > 4096 || head_dim > 512) return 0;
    const size_t stage = kv_heads * head_dim * ((L + 63) / 64 * 64) * 2;
    return kv_dtype == SUPERSONIC_KV_FP8_E4M3 ? 2 * stage : stage;
}

extern "C" size_t supersonic_attn_gfx950_prefill_workspace_size(int kv_dtype, size_t kv_heads, size_t head_dim,
                                                                size_t chunk_len, size_t chunk_start) {
    const size_t L = chunk_start + chunk_len;
    const size_t stages = prefill_stage_bytes(kv_dtype, kv_heads, head_dim, chunk_len, chunk_start);
    // + a key split's sums
    return stages + (stages && prefill_may_split(chunk_len, L, kv_heads) ? prefill_part_bytes(static_cast<int>(head_dim), 256) : 0);
}

namespace ssa {
// The fused prefill with an optional dynamic schedule (claims: zeroed claim
// counters, PrefillParams::claims); supersonic_attn_gfx950_prefill is the
// static one.
int prefill_native(size_t device_ordinal, void* stream, int kv_dtype, size_t q_heads, size_t kv_heads,
                   size_t head_dim, size_t rotary_dim, size_t chunk_len, size_t chunk_start, float eps, float scale,
                   const void* q_proj, const void* k_new, const void* v_new, const void* q_norm_w,
                   const void* k_norm_w, const void* cos_table, const void* sin_table,
                   const supersonic_kv_cache* cache, void* out, void* workspace, size_t workspace_bytes,
                   unsigned* claims, int free_wgs) {
    if (kv_dtype != SUPERSONIC_KV_BF16 && kv_dtype != SUPERSONIC_KV_FP8_E4M3) return SUPERSONIC_ERR_DTYPE;
    const bool fp8 = kv_dtype == SUPERSONIC_KV_FP8_E4M3;
    if (head_dim != 64 && head_dim != 128 && head_dim != 256) return SUPERSONIC_ERR_HEAD_DIM;
    if (kv_heads == 0 || q_heads % kv_heads != 0) return SUPERSONIC_ERR_HEADS;
    if (rotary_dim > head_dim || (rotary_dim / 2) % 16 != 0) return SUPERSONIC_ERR_ROTARY;
    if (!q_proj || !k_new || !v_new || !q_norm_w || !k_norm_w || !out) return SUPERSONIC_ERR_NULL;
    if (rotary_dim > 0 && (!cos_table || !sin_table)) return SUPERSONIC_ERR_NULL;
    if (chunk_len + chunk_start > 0x7FFFFFFF || q_heads > 4096) return SUPERSONIC_ERR_RANGE;
    KvView kv;
    if (int rc = make_view(cache, fp8, &kv)) return rc;
    if (kv.bt && kv.page_size % 64 != 0) return SUPERSONIC_ERR_CACHE;
    if (chunk_len == 0) return 0;
    ScopedDevice scoped(static_cast<int>(device_ordinal));
    hipStream_t st = static_cast<hipStream_t>(stream);


    PrefillSplitParams p{};
    p.q = static_cast<const uint16_t*>(q_proj);
    p.q_bs = 0;
    p.q_hs = 2 * static_cast<int64_t>(head_dim);
    p.q_rs = static_cast<int64_t>(q_heads) * 2 * head_dim;
    p.kv = kv;
    p.Hq = static_cast<int>(q_heads);
    p.Hkv = static_cast<int>(kv_heads);
    p.G = static_cast<int>(q_heads / kv_heads);
    p.S = static_cast<int>(chunk_len);
    p.L = static_cast<int>(chunk_start + chunk_len);
    p.off = static_cast<int>(chunk_start);
    p.scale_log2 = scale * kLog2e;
    p.rescale_slack = rescale_slack();
    p.nqt = static_cast<int>((chunk_len + 127) / 128);
    p.out_bf16 = static_cast<uint16_t*>(out);
    p.gate = static_cast<const uint16_t*>(q_proj) + head_dim;
    p.q_norm_w = static_cast<const uint16_t*>(q_norm_w);
    p.cos_t = static_cast<const uint16_t*>(cos_table);
    p.sin_t = static_cast<const uint16_t*>(sin_table);
    p.half_rot = static_cast<int>(rotary_dim / 2);
    p.eps = eps;
    p.B = 1;
    p.claims = claims;
    void* part = nullptr;  // room for a key split's sums
    size_t part_bytes = 0;
    // K norm + RoPE + cache append for the chunk and the V^T staging of every
    // position, in one pass
    {
        const int ld = (p.L + 63) / 64 * 64;
        // V^T staging, then (fp8 cache) the bf16 K rows the attention reads
        const size_t stage_bytes = static_cast<size_t>(p.Hkv) * head_dim * ld * 2;
        const size_t need = fp8 ? 2 * stage_bytes : stage_bytes;
        const bool may_split = prefill_may_split(chunk_len, p.L, kv_heads);
        void* ws = workspace;
        if (ws) {
            if (workspace_bytes < need) return SUPERSONIC_ERR_WORKSPACE;
            // (need is a multiple of 128)
            if (may_split && workspace_bytes > need) {
                part = static_cast<uint8_t*>(ws) + need;
                part_bytes = workspace_bytes - need;
            }
        } else {
            ws = device_workspace(static_cast<int>(device_ordinal), need, kWorkspacePrefill);
            if (ws && may_split) part = pieces_workspace(static_cast<int>(device_ordinal), st, &part_bytes);
        }
        if (!ws) return SUPERSONIC_ERR_WORKSPACE;
        p.vt = static_cast<const uint16_t*>(ws);
        p.vt_ld = ld;
        uint16_t* kst = fp8 ? reinterpret_cast<uint16_t*>(static_cast<uint8_t*>(ws) + stage_bytes) : nullptr;
        if (fp8) {
            // the attention kernel's K: the contiguous staging rows
            KvView ks{};
            ks.k = reinterpret_cast<uint8_t*>(kst);
            ks.head_stride = static_cast<int64_t>(ld) * head_dim;
            ks.seq_stride = static_cast<int64_t>(p.Hkv) * ld * head_dim;
            ks.page_size = 1;
            p.kv = ks;
        }
        KvStageParams kp{};
        kp.k_new = static_cast<const uint16_t*>(k_new);
        kp.v_new = static_cast<const uint16_t*>(v_new);
        kp.k_norm_w = static_cast<const uint16_t*>(k_norm_w);
        kp.cos_t = static_cast<const uint16_t*>(cos_table);
        kp.sin_t = static_cast<const uint16_t*>(sin_table);
        kp.kv = kv;
        kp.vt = static_cast<uint16_t*>(ws);
        kp.kst = kst;
        kp.S = static_cast<int>(chunk_len);
        kp.Hkv = static_cast<int>(kv_heads);
        kp.off = static_cast<int>(chunk_start);
        kp.L = p.L;
        kp.ld = ld;
        kp.half_rot = static_cast<int>(rotary_dim / 2);
        kp.eps = eps;
        const dim3 grid(ld / 64, kp.Hkv);
        const dim3 blk(64 * kKvStageWaves);
        switch (head_dim * 2 + (fp8 ? 1 : 0)) {
        case 128: hipLaunchKernelGGL((kv_stage_kernel<64, false>), grid, blk, 0, st, kp); break;
        case 129: hipLaunchKernelGGL((kv_stage_kernel<64, true>), grid, blk, 0, st, kp); break;
        case 256: hipLaunchKernelGGL((kv_stage_kernel<128, false>), grid, blk, 0, st, kp); break;
        case 257: hipLaunchKernelGGL((kv_stage_kernel<128, true>), grid, blk, 0, st, kp); break;
        case 512: hipLaunchKernelGGL((kv_stage_kernel<256, false>), grid, blk, 0, st, kp); break;
        default: hipLaunchKernelGGL((kv_stage_kernel<256, true>), grid, blk, 0, st, kp); break;
        }
        if (hipGetLastError() != hipSuccess) return SUPERSONIC_ERR_LAUNCH;
    }
    const ProfileEvents prof = take_profile_events();
    if (prof.before) (void)hipEventRecord(prof.before, st);
    if (launch_prefill<bf16_t, true>(static_cast<int>(device_ordinal), static_cast<int>(head_dim), st, p, part, part_bytes, free_wgs) != hipSuccess)
        return SUPERSONIC_ERR_LAUNCH;
    if (prof.after) (void)hipEventRecord(prof.after, st);
    return 0;
}
}  // namespace ssa

extern "C" int supersonic_attn_gfx950_prefill(
    size_t device_ordinal, void* stream, int kv_dtype, size_t q_heads, size_t kv_heads, size_t head_dim,
    size_t rotary_dim, size_t chunk_len, size_t chunk_start, float eps, float scale, const void* q_proj,
    const void* k_new, const void* v_new, const void* q_norm_w, const void* k_norm_w, const void* cos_table,
    const void* sin_table, const supersonic_kv_cache* cache, void* out, void* workspace, size_t workspace_bytes) {
    return ssa::prefill_native(device_ordinal, stream, kv_dtype, q_heads, kv_heads, head_dim, rotary_dim, chunk_len,
                               chunk_start, eps, scale, q_proj, k_new, v_new, q_norm_w, k_norm_w, cos_table,
                               sin_table, cache, out, workspace, workspace_bytes, nullptr);
}
