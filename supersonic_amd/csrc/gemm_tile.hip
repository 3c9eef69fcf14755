// bf16 GEMM out = a . w^T in tiles of 32 x 64 to 256 x 128, whole or split along
// k: decode batches past the weight-streaming kernels' rows, short and medium
// prefill chunks, and the full chunks whose tiles fill the CUs' rounds better
// than gemm.hip's 256 x 256 (gemm_plan chooses).  What bounds it: up to about
// 100 rows the weights' HBM stream; then the global->LDS copies, which run at
// about 53 GB/s a CU whatever the tile (128 x 64: 0.45 us a step of 24 KB,
// 128 x 128: 0.61, 256 x 128: 0.95; with every copy served by L2 and no MFMAs
// 0.40 / 0.45 / 0.58), and at 256 x 128 the MFMAs at the clock they leave.
// Measured (one MI355X, 256 x 256 tiles before): o_proj 4096 -> 4096 at 32 rows
// 91.7 -> 11.0 us, 128 rows 100 -> 17.0, 512 rows 104 -> 29.8, 1000 rows 103 ->
// 40.0, 2000 rows 103 -> 63.0 (1.07 PFLOP/s), 4096 rows 127.9 -> 124.3; norm +
// Q/K/V 4096 -> 10240 at 32 rows 95.3 -> 22.3, 512 rows 109 -> 58, 4096 rows
// 325 -> 306.
//
// Workgroup: a BM x BN tile of out over a slice of k, four or eight compute
// waves (1 x 4 for BM = 32, 2 x 2, 2 x 4 or 4 x 2) on v_mfma_f32_16x16x32_bf16 and four copy waves that
// only issue the global->LDS copies (two copy waves: 5-10% slower at 128 x 128
// and 256 x 128).  k advances 64 at a time through NST LDS stages; the copy
// waves run NST - 1 tiles ahead (128 x 128 with 2 stages instead of 4: 69 us
// instead of 42 at 1000 rows).  (Copies issued by the
// compute waves would make the compiler wait for all of them before an LDS
// read: it cannot tell the stages apart.)  LDS rows are 128 bytes, the 16-byte
// chunk c of row r at c ^ ((r >> 1) & 7), so the 16 rows an operand read
// touches cover all 64 banks.  Rows past m or n and chunks past k read as
// zeros.
//
// Split k: when the tiles alone leave CUs idle, each runs as `ks` workgroups
// over equal runs of k-tiles.  Every workgroup stores its fp32 accumulators
// device-coherently and counts its arrival; the last one adds the slices in
// slice order (the result does not depend on the arrival order), resets the
// counter and writes the output.  Nothing waits for another workgroup.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "gemm.hpp"
#include "gemm_epi.hpp"

namespace ssa {

constexpr int kTileBK = 64;
constexpr int kTileRowB = 128;      // LDS row: 64 bf16
constexpr int kTileCopyWaves = 4;
constexpr int kNontemporal = 2;     // cache-policy bit of a copy

struct GemmTileParams {
    const uint16_t* a;
    int64_t lda, a_bs;
    const uint16_t* w[3];
    void* out[3];
    int n[3];
    int nt_end[3];  // cumulative n-tiles of the segments
    int64_t w_bs, o_bs;
    int m, k, mt, nt, tiles;
    int vec_mask;   // bit s: segment s takes 16-byte output chunks
    int full;       // tiles that run whole; the others run as ks slices of kper k-tiles
    int ks, kper;
    float* part;        // [tiles][ks][BM * BN] accumulators in lane order
    unsigned* arrivals; // [tiles], zero between calls
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t gemm_tile_rsrc(const uint16_t* base, int64_t bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(base);
    const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a >> 32));
    void* u = reinterpret_cast<void*>((static_cast<uint64_t>(hi) << 32) | lo);
    const int nb = static_cast<int>(min(bytes, static_cast<int64_t>(0x7ffffff0)));
    return __builtin_amdgcn_make_buffer_rsrc(u, static_cast<short>(0), __builtin_amdgcn_readfirstlane(nb), 0x00020000);
}

// s_waitcnt vmcnt(N) alone (gfx9 encoding: bits 3:0 and 15:14).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}
// At most `tiles` (<= MAX) tiles of C copies still in flight.
template <int C, int MAX>
__device__ __forceinline__ void wait_tiles(int tiles) {
    if (tiles >= MAX) wait_vmcnt<C * MAX>();
    else if constexpr (MAX > 0) wait_tiles<C, MAX - 1>(tiles);
}

template <int BM, int BN, int NST, int NW, int EPI>
__global__ __launch_bounds__(64 * (NW + kTileCopyWaves)) __attribute__((amdgpu_waves_per_eu(3))) void gemm_tile_kernel(GemmTileParams p) {
    constexpr int kTileWaves = NW;
    constexpr int kATile = BM * kTileRowB, kWTile = BN * kTileRowB, kStage = kATile + kWTile;
    constexpr int WGM = BM == 32 ? 1 : (BM == 256 ? 4 : 2), WGN = kTileWaves / WGM;  // wave grid
    constexpr int WM = BM / WGM, WN = BN / WGN;                    // wave tile
    constexpr int MB = WM / 16, NB = WN / 16;
    constexpr int kEpiRow = 2 * WN + 16;
    static_assert(NST * kStage >= kTileWaves * WM * kEpiRow, "epilogue rows fit the stages");
    __shared__ __attribute__((aligned(1024))) uint8_t lds[NST * kStage];
    __shared__ int last_s;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int b = blockIdx.y;

    // ---- tile and k slice of this workgroup.  The k slices of one tile are
    // consecutive workgroups of one XCD's range; the ranges are contiguous in
    // an order of bands of 8 m-tiles, n-major within a band, so an XCD's L2
    // serves the rows of a and w its tiles share.
    const bool split = static_cast<int>(blockIdx.x) >= p.full;
    const int i = split ? blockIdx.x - p.full : blockIdx.x;
    const int T = split ? (p.tiles - p.full) * p.ks : p.full;
    const int q = T / 8, r = T % 8;
    const int xcd = i % 8, slot = i / 8;
    const int u = xcd < r ? xcd * (q + 1) + slot : r * (q + 1) + (xcd - r) * q + slot;
    const int ts = split ? u / p.ks : 0, sl = split ? u - ts * p.ks : 0;
    const int t = split ? p.full + ts : u;
    constexpr int kBand = 8;
    const int band = t / (kBand * p.nt);
    const int gm = min(kBand, p.mt - band * kBand);
    const int tin = t - band * kBand * p.nt;
    const int tm = band * kBand + tin % gm;
    const int tn = tin / gm;
    const int seg = tn < p.nt_end[0] ? 0 : (tn < p.nt_end[1] ? 1 : 2);
    const int tn_s = tn - (seg == 0 ? 0 : (seg == 1 ? p.nt_end[0] : p.nt_end[1]));
    const int ns = pick3(p.n, seg);
    const int m0 = tm * BM, n0 = tn_s * BN;
    const int KT_all = (p.k + kTileBK - 1) / kTileBK;
    const int kt0 = sl * p.kper;
    const int KT = split ? min(kt0 + p.kper, KT_all) : KT_all;

    f32x4_v acc[MB][NB];
#pragma unroll
    for (int ib = 0; ib < MB; ++ib)
#pragma unroll
        for (int jb = 0; jb < NB; ++jb) acc[ib][jb] = f32x4_v{0.f, 0.f, 0.f, 0.f};

    const int wm = WGM == 1 ? 0 : wave / WGN, wn = WGM == 1 ? wave : wave % WGN;
    if (wave >= kTileWaves) {
        // ---- copy waves.  Copy instruction c of a tile moves 8 rows (1 KB):
        // rows of a for c < BM / 8, then rows of w; copy wave cw takes
        // instructions cw, cw + kTileCopyWaves, ...  Lane l: row l / 8, physical chunk
        // l % 8.  The whole offset goes in the per-lane operand (the range
        // check does not cover the scalar offset).
        constexpr int kCopies = (BM + BN) / 8 / kTileCopyWaves;
        constexpr int kOOB = 0x7ffffff0;  // past any range: reads zero
        const int cw = wave - kTileWaves;
        const uint16_t* abase = p.a + b * p.a_bs + static_cast<int64_t>(m0) * p.lda;
        const uint16_t* wbase = pick3(p.w, seg) + b * p.w_bs + static_cast<int64_t>(n0) * p.k;
        const __amdgpu_buffer_rsrc_t ar = gemm_tile_rsrc(abase, static_cast<int64_t>(p.m - m0) * p.lda * 2);
        const __amdgpu_buffer_rsrc_t wr = gemm_tile_rsrc(wbase, static_cast<int64_t>(ns - n0) * p.k * 2);
        const int crow = lane >> 3;
        auto issue = [&](int kt, auto once) {
            const int k0 = kt * kTileBK;
            uint8_t* st = lds + ((kt - kt0) % NST) * kStage;
#pragma unroll
            for (int j = 0; j < kCopies; ++j) {
                const int c = kTileCopyWaves * j + cw;
                const bool isa = kTileCopyWaves * j < BM / 8;   // the same for every copy wave (kTileCopyWaves divides BM / 8)
                const int row = 8 * (isa ? c : c - BM / 8) + crow;
                const int ch = (lane & 7) ^ ((row >> 1) & 7);
                const int off = k0 + 8 * ch < p.k ? row * static_cast<int>(isa ? p.lda : p.k) * 2 + (k0 + 8 * ch) * 2 : kOOB;
                if (isa)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(ar, (__attribute__((address_space(3))) void*)(st + 1024 * c), 16,
                                                             off, 0, 0, 0);
                else if constexpr (decltype(once)::value)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (__attribute__((address_space(3))) void*)(st + 1024 * c), 16,
                                                             off, 0, 0, kNontemporal);
                else
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (__attribute__((address_space(3))) void*)(st + 1024 * c), 16,
                                                             off, 0, 0, 0);
            }
        };
        auto copy_tiles = [&](auto once) {
            for (int v = 0; v < NST - 1; ++v)
                if (kt0 + v < KT) issue(kt0 + v, once);
            for (int kt = kt0; kt < KT; ++kt) {
                wait_tiles<kCopies, NST - 2>(KT - 1 - kt);  // tile kt has landed
                __builtin_amdgcn_s_barrier();               // ... and the stage of tile kt - 1 has been read
                if (kt + NST - 1 < KT) issue(kt + NST - 1, once);
            }
        };
        // One m-tile: each weight is read by one workgroup and passes the caches
        // by (norm + Q/K/V 4096 -> 10240 at 8 rows 22.0 -> 19.7 us, 32 rows
        // 24.0 -> 22.3; o_proj 4096 -> 4096 at 16 rows 11.0 -> 10.6).
        if (BM <= 64 && p.mt == 1) copy_tiles(std::true_type{});
        else copy_tiles(std::false_type{});
    } else {
        // ---- compute waves.  Operand reads: row lane % 16 of a 16-row block,
        // logical chunk 4 s + lane / 16 of k32 step s.
        const int orow = lane & 15;
        const int sw_x = (orow >> 1) & 7;
        const int a_rd = (wm * WM + orow) * kTileRowB;
        const int w_rd = kATile + (wn * WN + orow) * kTileRowB;
        auto read_frags = [&](int kt, int s, bf16x8_v (&af)[MB], bf16x8_v (&bf)[NB]) {
            const uint8_t* st = lds + ((kt - kt0) % NST) * kStage;
            const int ck = ((4 * s + (lane >> 4)) ^ sw_x) * 16;
#pragma unroll
            for (int ib = 0; ib < MB; ++ib)
                af[ib] = *reinterpret_cast<const bf16x8_v*>(st + a_rd + ib * 16 * kTileRowB + ck);
#pragma unroll
            for (int jb = 0; jb < NB; ++jb)
                bf[jb] = *reinterpret_cast<const bf16x8_v*>(st + w_rd + jb * 16 * kTileRowB + ck);
        };
        auto mma = [&](const bf16x8_v (&af)[MB], const bf16x8_v (&bf)[NB]) {
#pragma unroll
            for (int ib = 0; ib < MB; ++ib)
#pragma unroll
                for (int jb = 0; jb < NB; ++jb)
                    acc[ib][jb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[ib], bf[jb], acc[ib][jb], 0, 0, 0);
        };
        // Two register sets: the operands of the next k32 step are read while
        // the MFMAs of the current one run, also across the tile barrier.
        bf16x8_v a0[MB], b0[NB], a1[MB], b1[NB];
        lds_barrier();
        read_frags(kt0, 0, a0, b0);
        for (int kt = kt0; kt < KT; ++kt) {
            read_frags(kt, 1, a1, b1);
            mma(a0, b0);
            if (kt + 1 < KT) {
                lds_barrier();  // waits for this wave's reads of tile kt, then for tile kt + 1
                read_frags(kt + 1, 0, a0, b0);
            }
            mma(a1, b1);
        }
    }

    // ---- split k: hand the slice over; the last to arrive goes on with the sum
    if (split) {
        constexpr int kBlocks = MB * NB;
        float* tp = p.part + static_cast<int64_t>(ts) * p.ks * (BM * BN);
        const int wo = wave * kBlocks * 256;  // this wave's accumulators in a slice
        if (wave < kTileWaves) {
            float* mine = tp + static_cast<int64_t>(sl) * (BM * BN) + wo;
#pragma unroll
            for (int ib = 0; ib < MB; ++ib)
#pragma unroll
                for (int jb = 0; jb < NB; ++jb) {
                    u32x4_v v;
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = __float_as_uint(acc[ib][jb][e]);
                    st_coh<4>(mine + (ib * NB + jb) * 256, lane * 16, v);
                }
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
            __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's stores are complete
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
        }
        __syncthreads();
        if (tid == 0)
            last_s = __hip_atomic_fetch_add(p.arrivals + ts, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
                     static_cast<unsigned>(p.ks - 1);
        __syncthreads();
        if (!last_s) return;
        if (tid == 0) __hip_atomic_store(p.arrivals + ts, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (wave < kTileWaves) {
            f32x4_v sum[MB][NB];
#pragma unroll
            for (int ib = 0; ib < MB; ++ib)
#pragma unroll
                for (int jb = 0; jb < NB; ++jb) sum[ib][jb] = f32x4_v{0.f, 0.f, 0.f, 0.f};
            for (int v = 0; v < p.ks; ++v) {
                const float* src = tp + static_cast<int64_t>(v) * (BM * BN) + wo;
#pragma unroll
                for (int ib = 0; ib < MB; ++ib)
#pragma unroll
                    for (int jb = 0; jb < NB; ++jb) {
                        const u32x4_v x = ld_coh<4>(src + (ib * NB + jb) * 256, lane * 16);
#pragma unroll
                        for (int e = 0; e < 4; ++e) sum[ib][jb][e] += __uint_as_float(x[e]);
                    }
            }
#pragma unroll
            for (int ib = 0; ib < MB; ++ib)
#pragma unroll
                for (int jb = 0; jb < NB; ++jb) acc[ib][jb] = sum[ib][jb];
        }
    } else {
        lds_barrier();  // every wave is done with the operand stages
    }
    if (wave >= kTileWaves) return;

    // ---- epilogue, through LDS: lane holds rows 16 ib + 4 (lane / 16) + e,
    // column 16 jb + lane % 16 of its wave's tile; rows go out as 16-byte chunks.
    uint8_t* blk = lds + wave * (WM * kEpiRow);
#pragma unroll
    for (int ib = 0; ib < MB; ++ib)
#pragma unroll
        for (int jb = 0; jb < NB; ++jb)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                *reinterpret_cast<uint16_t*>(blk + (ib * 16 + 4 * (lane >> 4) + e) * kEpiRow + (jb * 16 + (lane & 15)) * 2) =
                    static_cast<uint16_t>(f32_to_bf16_bits(acc[ib][jb][e]));
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    void* outp = pick3(p.out, seg);
    const bool vec = (p.vec_mask >> seg) & 1;  // ns % 8 == 0 and 16-byte aligned rows
    const int64_t obase = b * p.o_bs;
    constexpr int kCpr = WN / 8;
#pragma unroll
    for (int it = 0; it < WM * kCpr / 64; ++it) {
        const int qd = it * 64 + lane;
        const int rr = qd / kCpr, c = qd % kCpr;
        const int row = m0 + wm * WM + rr, col = n0 + wn * WN + 8 * c;
        if (row >= p.m || col >= ns) continue;
        const u32x4_v v = *reinterpret_cast<const u32x4_v*>(blk + rr * kEpiRow + c * 16);
        gemm_store_chunk<EPI>(outp, obase + static_cast<int64_t>(row) * ns + col, v, vec, ns - col);
    }
}

template <int BM, int BN, int NST, int NW>
static int launch_tile(hipStream_t st, const GemmTileParams& p, int batch, int epilogue) {
    const dim3 grid(static_cast<unsigned>(p.full + (p.tiles - p.full) * p.ks), static_cast<unsigned>(batch)), blk(64 * (NW + kTileCopyWaves));
    switch (epilogue) {
    case kGemmResidualBf16: hipLaunchKernelGGL((gemm_tile_kernel<BM, BN, NST, NW, kGemmResidualBf16>), grid, blk, 0, st, p); break;
    case kGemmResidualF32: hipLaunchKernelGGL((gemm_tile_kernel<BM, BN, NST, NW, kGemmResidualF32>), grid, blk, 0, st, p); break;
    default: hipLaunchKernelGGL((gemm_tile_kernel<BM, BN, NST, NW, kGemmStore>), grid, blk, 0, st, p); break;
    }
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

int gemm_tile(hipStream_t st, const GemmArgs& g) {
    const GemmPlan& plan = g.plan;
    GemmTileParams p{};
    p.a = g.a;
    p.lda = g.lda;
    p.a_bs = g.a_bs;
    p.w_bs = g.w_bs;
    p.o_bs = g.o_bs;
    p.m = g.m;
    p.k = g.k;
    p.mt = (g.m + plan.bm - 1) / plan.bm;
    int nt = 0;
    for (int s = 0; s < 3; ++s) {
        const int n = s < g.nseg ? g.n[s] : 0;
        p.w[s] = s < g.nseg ? g.w[s] : g.w[0];
        p.out[s] = s < g.nseg ? g.out[s] : g.out[0];
        p.n[s] = n;
        const uintptr_t op = reinterpret_cast<uintptr_t>(p.out[s]);
        if (n % 8 == 0 && op % 16 == 0 && (g.o_bs % 8) == 0) p.vec_mask |= 1 << s;
        nt += (n + plan.bn - 1) / plan.bn;
        p.nt_end[s] = nt;
    }
    p.nt = nt;
    p.tiles = p.mt * nt;
    const int KT = (g.k + kTileBK - 1) / kTileBK;
    p.kper = (KT + plan.ks - 1) / plan.ks;
    p.ks = KT > 0 ? (KT + p.kper - 1) / p.kper : 1;  // no empty slice
    p.full = p.ks > 1 ? p.tiles - plan.split_tiles : p.tiles;
    if (p.ks > 1) {
        p.arrivals = reinterpret_cast<unsigned*>(static_cast<uint8_t*>(g.ws) + kGemmFlagBytes);
        p.part = reinterpret_cast<float*>(static_cast<uint8_t*>(g.ws) + kGemmPartOff);
    }
    switch (plan.bm * 1000 + plan.bn) {
    case 32064: return launch_tile<32, 64, 6, 4>(st, p, g.batch, g.epilogue);
    case 64064: return launch_tile<64, 64, 4, 4>(st, p, g.batch, g.epilogue);
    case 128064: return launch_tile<128, 64, 6, 8>(st, p, g.batch, g.epilogue);
    case 128128: return launch_tile<128, 128, 4, 8>(st, p, g.batch, g.epilogue);
    case 256128: return launch_tile<256, 128, 3, 8>(st, p, g.batch, g.epilogue);
    default: return 1;
    }
}

}  // namespace ssa
