// Persistent decode layer: the whole attention layer of a decode step in one
// kernel, the attention phase as a device function between the projections
// (the reference's persistent megakernel pattern,
// kernels/qwen36_moe_persistent/full_attn_phase.cuh:1-20, and the HIP
// megakernel's steps A-G, kernels/full_attention_4b.hip:4842-5577).
//
// One workgroup per compute unit (an ordinary launch, see below), three phases
// separated by device-wide barriers:
//   1. input RMSNorm (applied while each workgroup stages the rows in LDS) and
//      the Q/K/V weight stream, 16 output columns per workgroup task;
//   2. the split-K attention step (QK RMSNorm, partial RoPE, KV append, online
//      softmax, last-arriver log-sum-exp merge, sigmoid gate): work item w of
//      the ragged plan on workgroup w;
//   3. the output projection with the residual add, in place on the hidden rows.
// Every value one phase hands to the next is stored and loaded with
// device-coherent accesses, so a barrier is: each wave waits for its own
// stores, one lane bumps a counter, the last to arrive raises a flag, and only
// the workgroups that read the previous phase's output wait (bounded) for the
// flag.  Launch fill and drain are paid once per layer instead of once per
// kernel.
#include <algorithm>
#include <cstdlib>
#include <mutex>
#include <vector>

#include "common.hpp"
#include "decode_split.hpp"
#include "kv_view.hpp"
#include "skinny.hpp"
#include "supersonic_attn.h"

namespace ssa {

struct LayerParams {
    SkinnyLdsParams qkv;  // phase 1: three segments, NORM staging from the hidden rows
    DecodeParams dec;     // phase 2: fused decode step, ragged plan over the grid
    SkinnyLdsParams op;   // phase 3: attn -> hidden (residual in place)
    unsigned* bar;        // barrier counters [0..2] and flags [32], [48] (another cache line), zero between calls
    unsigned* ids;        // [grid] who has which part (IdState), zero between calls
    int polls;            // bound of a barrier wait (kLayerSpin)
    // > 0: the decode step is expected to have this many work items (one
    // sequence of length max_kv_len); the last `hint` workgroups then take
    // them and skip phase 1, which the others share.
    int hint;
    int layer_len;        // host: the expected sequence length (max_kv_len), for the hint
};

constexpr int kLayerThreads = 64 * kSkinnyWaves;  // = 64 * decode_waves(4)
constexpr int kLayerSpin = 1 << 20;               // bounded barrier wait
constexpr int kLayerMissingPolls = 64;            // ... after which missing workgroups' parts are taken over (40 us)
constexpr int kLayerMaxGrid = 1024;               // workspace bound on the grid (partial rows, ids)

// Every value one phase hands to the next is written and read with
// device-coherent (sc1) accesses, so the barrier needs no cache writeback or
// invalidate: each wave waits for its own stores to complete, then one lane
// counts the workgroup in; the last to arrive raises a flag on another cache
// line, which the waiting workgroups poll (polls on the counter's own line
// measured to hold back the arrivals' atomics).  The arriving lane is the
// last wave's first: it waits for the count to come back, and wave 0 goes on.
// Split form: arrive (after this workgroup's stores are complete), do
// independent work, then wait.
//
// Ordering: the producer's data stores are sc1 (written through to the
// device coherence point); `s_waitcnt vmcnt(0)` makes each wave wait until
// they are acknowledged there, the workgroup barrier orders every wave's wait
// before the counting atomic, and the compiler fences keep the stores above
// the wait.  A consumer issues its sc1 loads only after its poll has returned
// the flag (the poll result is waited for before the branch, and the
// workgroup barrier after the poll orders the other waves' loads after it),
// and sc1 loads are served from the coherence point, not from a stale
// per-XCD cache line.  This is what an agent-scope release / acquire pair
// provides, without the L2 writeback and invalidate those emit.
//
// The launch does not promise that every workgroup of the grid is running, and
// no wait depends on one that is not.  (A cooperative launch does promise it,
// through a queue of its own: 17-20 us a call on this runtime.)  The layer's
// work comes in one part an id, 0 .. grid - 1: the column blocks, decode item
// and output columns above.  A workgroup takes the id of its index as it
// starts, with an atomic whose round trip runs beside the weight stream and
// whose result is needed before the first store.  Where a wait lasts
// (kLayerMissingPolls) while arrivals are missing from barrier 0, the waiting
// workgroup takes an id that no workgroup has started yet, runs its part of
// phase 1, arrives for it, and later runs its decode item and output columns
// behind its own.  A workgroup that finds its id taken leaves.  So whatever
// the number of workgroups that find a CU (two layers on two streams hold a
// part of the CUs each), those that did go on: every id is in the hands of a
// running workgroup before barrier 0 opens, and decode items never wait for
// each other.  1 sequence of 2048 tokens, 8/2 heads, hidden 1024: 48.8 us a
// layer with the cooperative launch, 32.5 with an ordinary one and a kernel
// behind it for the case that workgroups are missing, 29.4 with this (29.3
// without any of it); such layers on two streams 39.4 us each with
// the cooperative launch, 17.9 with this.
// A wait only expires on a workspace whose counters were not zero: it then sets
// kWaitLayerBarrier in the error word and carries on, so that the kernel still
// exits.
enum IdState : unsigned { kIdFree = 0u, kIdTaken = 1u, kIdProjected = 2u };  // projected: phase 1 done
enum LayerWait { kLayerGo, kLayerMissing };
constexpr int kArriveThread = kLayerThreads - 64;
struct LayerShared {
    int mine;                        // this workgroup got the id it is working on
    int res;                         // grid_wait's polls and take_over's id
    int first;                       // free_id's result
    uint16_t taken[kLayerMaxGrid];   // [1 ..]: ids taken over
};
// Whether this workgroup has its id, known by the time the outputs go out.
struct OwnId {
    unsigned before;  // the id's state before it was taken (kArriveThread)
    int& mine;
    __device__ void park() const {
        if (threadIdx.x == kArriveThread) mine = before == kIdFree;
    }
    __device__ bool open() const { return __builtin_amdgcn_readfirstlane(mine) != 0; }
};
// This workgroup's coherent stores are complete, for all of its threads.
__device__ __forceinline__ void stores_complete() {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's stores are complete
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();
}
// Counts one id in; stores_complete() comes first.
__device__ __forceinline__ void grid_arrive(unsigned* ctr, unsigned* flag, unsigned n) {
    if (threadIdx.x == kArriveThread) {
        const unsigned prev = __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (prev == n - 1) __hip_atomic_store(flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}
// The first id from w on that no workgroup has started, as its distance from
// w; nwg: every id is taken, nwg + 1: and has its phase 1 done.
__device__ __forceinline__ int free_id(const LayerParams& P, int w, int nwg, LayerShared& sh) {
    __syncthreads();
    if (threadIdx.x == 0) sh.first = nwg + 1;
    __syncthreads();
    for (int i = threadIdx.x; i < nwg; i += kLayerThreads) {
        const unsigned s = load_agent_u32(P.ids + (w + i < nwg ? w + i : w + i - nwg));
        if (s != kIdProjected) atomicMin(&sh.first, s == kIdFree ? i : nwg);
    }
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(sh.first);
}
// Waits for barrier `which` (0 or 1).  kLayerMissing: it lasted, arrivals are
// missing from barrier 0 and an id is free.  (With every id taken the wait goes
// on, so that a decode item is not planned again; with every id's phase 1 done
// barrier 0 opens whatever its counter says.)  spent: polls of the waits that
// found a free id, in all.
__device__ __forceinline__ LayerWait grid_wait(const LayerParams& P, int which, int w, unsigned nwg, int& spent,
                                               LayerShared& sh) {
    int at = 0, look = spent ? 8 : min(P.polls, kLayerMissingPolls);
    for (;;) {
        if (threadIdx.x == 0) {
            unsigned* const ctr = P.bar + which;
            unsigned* const flag = P.bar + 32 + 16 * which;
            auto missing = [&](unsigned* c) { return static_cast<int>(load_agent_u32(c)) < static_cast<int>(nwg); };
            // a wait expires after P.polls polls once every arrival has been counted
            // for kLayerMissingPolls of them (the flag follows the count)
            int r = 0, late = 0;
            for (int it = at;; ++it) {
                if (load_agent_u32(flag) != 0u) break;
                if (it >= look && spent < kLayerSpin && load_agent_u32(P.bar + 32) == 0u && missing(P.bar)) {
                    r = it + 1;
                    break;
                }
                if (it >= P.polls && !missing(ctr)) ++late;
                if (late >= kLayerMissingPolls || it >= kLayerSpin || spent >= kLayerSpin) {
                    wait_expired(kWaitLayerBarrier);
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
            }
            sh.res = r;
        }
        __syncthreads();
        at = __builtin_amdgcn_readfirstlane(sh.res);
        if (at == 0) return kLayerGo;
        const int f = free_id(P, w, static_cast<int>(nwg), sh);
        if (f < static_cast<int>(nwg)) {
            spent += at;
            return kLayerMissing;
        }
        if (f > static_cast<int>(nwg) && threadIdx.x == 0)
            __hip_atomic_store(P.bar + 32, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        look = at + kLayerMissingPolls;
    }
}
// Takes the next id after w that no workgroup has started; -1: there is none
// any more.
__device__ __forceinline__ int take_over(const LayerParams& P, int w, int nwg, LayerShared& sh) {
    const int f = free_id(P, w, nwg, sh);
    if (threadIdx.x == 0) {
        int v = -1;
        if (f < nwg) {
            v = w + f < nwg ? w + f : w + f - nwg;
            if (atomicCAS(P.ids + v, static_cast<unsigned>(kIdFree), static_cast<unsigned>(kIdTaken)) != kIdFree) v = -1;
        }
        sh.res = v;
    }
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(sh.res);
}

// The kernel's arguments, read again where they are asked for: kept in scalar
// registers around the loops below they spill (259 of them, and 39 vector
// registers with them; 57 and none so).
__device__ __forceinline__ const LayerParams& layer_args() {
    typedef const __attribute__((address_space(4))) LayerParams* Kernarg;
    uint64_t a = reinterpret_cast<uint64_t>(__builtin_amdgcn_kernarg_segment_ptr());
    asm volatile("" : "+s"(a));
    return *(const LayerParams*)reinterpret_cast<Kernarg>(a);
}

template <typename HT, bool FP8, int D>
__global__ __launch_bounds__(kLayerThreads) void decode_layer_kernel(LayerParams) {
    static_assert(decode_waves(4) * 64 == kLayerThreads, "one workgroup shape for every phase");
    // (sh first: LDS below 64 KB is reached with an immediate offset)
    __shared__ struct {
        LayerShared sh;
        union {
            DecodeLds<D, 4> d;
            SkinnyLds s;
        };
    } lds;
    LayerShared& sh = lds.sh;
    const LayerParams& P = layer_args();
    const int w = blockIdx.x;
    const unsigned nwg = gridDim.x;
    const int ncb_qkv = P.qkv.cb_end[2], ncb_op = P.op.cb_end[2];
    const int nq = static_cast<int>(nwg) - P.hint;
    const int shift = min(max(ncb_qkv - static_cast<int>(nwg), 0), static_cast<int>(nwg));
    auto item_of = [&](int v) {
        return P.hint > 0 ? (v >= nq ? v - nq : P.hint + v)
                          : (v - shift + static_cast<int>(nwg)) % static_cast<int>(nwg);
    };
    // Ahead of every load, so that no later wait has to count it.
    OwnId own{kIdFree, sh.mine};
    if (threadIdx.x == kArriveThread)
        own.before = atomicCAS(P.ids + w, static_cast<unsigned>(kIdFree), static_cast<unsigned>(kIdTaken));
    int n_ids = 1, n_items = 0;      // ids of this workgroup, and those whose decode item is done
    bool has_op = w < ncb_op;
    int spent = 0;
    for (int v = w;;) {
        const LayerParams& P = layer_args();
        if (v >= 0) {
            // 1. input norm + Q/K/V projections on the first nq ids: column
            // blocks v, v + nq, ...; with two left they run together
            // (one staging of the rows, both weight streams in flight)
            const SkinnyLdsParams qkv = P.qkv;
            for (int cb = v; cb < ncb_qkv && v < nq;) {
                if (cb + nq < ncb_qkv) {
                    skinny_lds_body<bf16_t, false, false, true, HT, false, true, SkinnyLds, true>(
                        qkv, RopeEpi{}, cb, 0, lds.s, cb + nq, own);
                    cb += 2 * nq;
                } else {
                    skinny_lds_body<bf16_t, false, false, true, HT, false, true, SkinnyLds, false>(
                        qkv, RopeEpi{}, cb, 0, lds.s, -1, own);
                    cb += nq;
                }
                __syncthreads();
            }
            own.park();
            stores_complete();
            if (!own.open()) break;
            own.before = kIdFree;
            if (threadIdx.x == kArriveThread)
                __hip_atomic_store(P.ids + v, static_cast<unsigned>(kIdProjected), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            grid_arrive(&P.bar[0], &P.bar[32], nwg);
        }
        // 2. attention step (every workgroup plans the same ragged split).  The
        // work items go first to the ids with one phase-1 task (the
        // first ncb_qkv - nwg have two), so the items start with their plan and
        // first K/V block (the cache does not depend on phase 1) while phase 1
        // finishes.  The workgroup arrives at barrier 0 first, then plans its item
        // and fetches its first block, and only then waits; without
        // an item it does not wait (only the readers of phase 1's output do).
        // With a hint the expected items sit on the ids without phase-1
        // work (any further item on the others).
        LayerWait res = kLayerGo;
        for (; n_items < n_ids; ++n_items) {
            const LayerParams& P = layer_args();
            const int u = n_items == 0 ? w : __builtin_amdgcn_readfirstlane(sh.taken[n_items]);
            const DecodeParams dec = P.dec;
            bool had_item = false;
            decode_split_body<bf16_t, FP8, D, 4, true>(dec, item_of(u), 0, 0, lds.d, [&]() {
                res = grid_wait(P, 0, w, nwg, spent, sh);
                had_item = true;
                return res == kLayerGo;
            });
            // (the body's way out depends on its plan, in LDS: say that it is one for all lanes)
            res = static_cast<LayerWait>(__builtin_amdgcn_readfirstlane(res));
            had_item = __builtin_amdgcn_readfirstlane(had_item) != 0;
            if (res != kLayerGo) break;
            if (!had_item && u < ncb_op) {
                // An output-projection workgroup without a decode item copies its
                // first task's weight rows into an LDS sink while the items run, so
                // that phase 3 finds them in this XCD's L2.  (The copies complete
                // before it arrives at barrier 1, which waits for its loads.)
                const int k = P.op.k;
                const int bytes = min(kSkinnyCols, P.op.n_seg[0] - u * kSkinnyCols) * k * 2;
                const __amdgpu_buffer_rsrc_t r =
                    uniform_rsrc(reinterpret_cast<const uint8_t*>(P.op.w[0] + static_cast<int64_t>(u) * kSkinnyCols * k), bytes);
                const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
                for (int off = wave * 1024; off < bytes; off += kSkinnyWaves * 1024)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds.s.xs, 16,
                                                             off + lane * 16, 0, 0, 0);
            }
            // Barrier 1: every id arrives; the workgroups with an
            // output-projection task wait for all of them.
            stores_complete();
            grid_arrive(&P.bar[1], &P.bar[48], nwg);
        }
        if (res == kLayerGo && has_op) res = grid_wait(P, 1, w, nwg, spent, sh);
        if (res == kLayerGo) {
            // 3. output projection + residual
            for (int i = 0; i < n_ids; ++i) {
                const int u = i == 0 ? w : __builtin_amdgcn_readfirstlane(sh.taken[i]);
                for (int cb = u; cb < ncb_op; cb += nwg) {
                    const SkinnyLdsParams op = layer_args().op;
                    skinny_lds_body<HT, true, false, false, bf16_t, true, false>(op, RopeEpi{}, cb, 0, lds.s);
                    __syncthreads();
                }
            }
            break;
        }
        v = take_over(P, w, static_cast<int>(nwg), sh);
        if (v >= 0) {
            if (threadIdx.x == 0) sh.taken[n_ids] = static_cast<uint16_t>(v);  // (read behind stores_complete)
            ++n_ids;
            has_op |= v < ncb_op;
        }
    }
    // The last workgroup to finish resets every counter, flag and id: each
    // workgroup counts itself in here after its last arrival and its last
    // poll, so nothing reads or bumps them any more in this call, whether or
    // not a wait gave up.
    if (threadIdx.x < 64) {
        unsigned prev = 0;
        if (threadIdx.x == 0) prev = __hip_atomic_fetch_add(&P.bar[2], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__builtin_amdgcn_readfirstlane(prev) == nwg - 1) {
            auto zero = [](unsigned* p) { __hip_atomic_store(p, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
            if (threadIdx.x == 0) {
                zero(&P.bar[0]);
                zero(&P.bar[1]);
                zero(&P.bar[32]);
                zero(&P.bar[48]);
                zero(&P.bar[2]);
            }
            for (int i = threadIdx.x; i < static_cast<int>(nwg); i += 64) zero(P.ids + i);
        }
    }
}

// Workgroups of one layer-kernel instance resident at once, per device.
template <typename HT, bool FP8, int D>
static int layer_grid(int device) {
    static std::mutex mu;
    static std::vector<int> cap;
    std::lock_guard<std::mutex> lock(mu);
    if (device < 0) return 0;
    if (static_cast<size_t>(device) >= cap.size()) cap.resize(device + 1, -1);
    if (cap[device] < 0) {
        int per_cu = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, decode_layer_kernel<HT, FP8, D>, kLayerThreads, 0) !=
            hipSuccess)
            per_cu = 0;
        cap[device] = per_cu * device_cu_count(device);
    }
    return cap[device];
}

constexpr size_t kLayerBarBytes = 256;
constexpr size_t kLayerArrivalBytes = 64 << 10;

inline size_t al256(size_t x) { return (x + 255) & ~static_cast<size_t>(255); }

struct LayerWs {
    size_t bar, ids, arrivals, part_o, part_ml, q_proj, k_new, v_new, attn, total;
};

inline LayerWs layer_ws(int B, int Hq, int Hkv, int D, int max_len) {
    (void)max_len;
    // ragged plan: at most (ceil(target / Hkv) + B) * Hq partial rows
    const size_t rows = (static_cast<size_t>((kLayerMaxGrid + Hkv - 1) / Hkv) + B) * Hq;
    LayerWs w{};
    w.bar = 0;
    w.ids = kLayerBarBytes;
    w.arrivals = w.ids + kLayerMaxGrid * sizeof(unsigned);
    w.part_o = w.arrivals + kLayerArrivalBytes;
    w.part_ml = w.part_o + al256(rows * D * 4);
    w.q_proj = w.part_ml + al256(rows * 2 * 4);
    w.k_new = w.q_proj + al256(static_cast<size_t>(B) * Hq * 2 * D * 2);
    w.v_new = w.k_new + al256(static_cast<size_t>(B) * Hkv * D * 2);
    w.attn = w.v_new + al256(static_cast<size_t>(B) * Hkv * D * 2);
    w.total = w.attn + al256(static_cast<size_t>(B) * Hq * D * 2);
    return w;
}

template <typename HT, bool FP8, int D>
static int launch_layer(int device, hipStream_t st, LayerParams& P) {
    const int grid = std::min(layer_grid<HT, FP8, D>(device), kLayerMaxGrid);
    if (grid <= 0) return SUPERSONIC_ERR_LAUNCH;
    // one workgroup per item: every (sequence, kv head) needs one
    if (P.dec.B * P.dec.Hkv > grid) return SUPERSONIC_ERR_RANGE;
    P.dec.target = grid;
    P.dec.strict = 1;
    P.hint = 0;
    if (P.dec.B == 1 && P.layer_len > 0) {
        // the device plan for one sequence of the expected length
        const int64_t l = P.layer_len, Hkv = P.dec.Hkv;
        auto items_of = [&](int64_t c) { return std::max<int64_t>(1, (l + c - 1) / c) * Hkv; };
        const int64_t items = items_of(ragged_chunk(l, P.dec.Hkv, grid, P.dec.min_chunk, true, items_of, [&]() { return l; }));
        if (2 * items <= grid) P.hint = static_cast<int>(items);
    }
    P.polls = wait_polls(kLayerSpin);
    P.dec.merge_polls = wait_polls(kMergePoll);
    hipLaunchKernelGGL((decode_layer_kernel<HT, FP8, D>), dim3(grid), dim3(kLayerThreads), 0, st, P);
    return hipGetLastError() == hipSuccess ? 0 : SUPERSONIC_ERR_LAUNCH;
}

hipError_t take_wait_error_layer(unsigned* bits) { return take_wait_error(bits); }

}  // namespace ssa

using namespace ssa;

extern "C" size_t supersonic_attn_gfx950_decode_layer_workspace_size(size_t batch, size_t hidden_dim, size_t q_heads,
                                                                     size_t kv_heads, size_t head_dim,
                                                                     size_t max_kv_len) {
    (void)hidden_dim;
    if (batch == 0 || batch > 64 || kv_heads == 0 || q_heads > 4096 || head_dim > 512 || max_kv_len > 0x7FFFFFFF)
        return 0;
    return layer_ws(static_cast<int>(batch), static_cast<int>(q_heads), static_cast<int>(kv_heads),
                    static_cast<int>(head_dim), static_cast<int>(max_kv_len)).total;
}

extern "C" int supersonic_attn_gfx950_decode_layer(
    size_t device_ordinal, void* stream, int hidden_dtype, int kv_dtype, size_t batch, size_t hidden_dim,
    size_t q_heads, size_t kv_heads, size_t head_dim, size_t rotary_dim, size_t max_kv_len, float eps, float qk_eps,
    float scale, void* hidden, const void* input_norm_w, const void* q_proj_w, const void* k_proj_w,
    const void* v_proj_w, const void* q_norm_w, const void* k_norm_w, const void* o_proj_w, const void* cos_table,
    const void* sin_table, const int32_t* positions, const supersonic_kv_cache* cache, void* workspace,
    size_t workspace_bytes) {
    if (hidden_dtype != SUPERSONIC_DTYPE_BF16 && hidden_dtype != SUPERSONIC_DTYPE_F32) return SUPERSONIC_ERR_DTYPE;
    if (kv_dtype != SUPERSONIC_KV_BF16 && kv_dtype != SUPERSONIC_KV_FP8_E4M3) return SUPERSONIC_ERR_DTYPE;
    if (head_dim != 128 && head_dim != 256) return SUPERSONIC_ERR_HEAD_DIM;
    if (kv_heads == 0 || q_heads % kv_heads != 0 || q_heads / kv_heads > 4) return SUPERSONIC_ERR_HEADS;
    if (rotary_dim % 2 != 0 || rotary_dim > head_dim) return SUPERSONIC_ERR_ROTARY;
    if (batch == 0) return 0;
    const size_t B = batch, Hq = q_heads, Hkv = kv_heads, D = head_dim, hid = hidden_dim;
    const size_t nq = Hq * 2 * D, nkv = Hkv * D, adim = Hq * D;
    // both projections take the LDS-staged weight stream: rows * width <= 32768 elements
    if (B > 16 || hid == 0 || hid % 16 != 0 || B * hid > static_cast<size_t>(kXsMax) ||
        B * adim > static_cast<size_t>(kXsMax) || max_kv_len == 0 || max_kv_len > 0x7FFFFFFF ||
        B * Hkv > kLayerArrivalBytes / 4)
        return SUPERSONIC_ERR_RANGE;
    if (!hidden || !input_norm_w || !q_proj_w || !k_proj_w || !v_proj_w || !q_norm_w || !k_norm_w || !o_proj_w ||
        !positions || !workspace)
        return SUPERSONIC_ERR_NULL;
    if (rotary_dim > 0 && (!cos_table || !sin_table)) return SUPERSONIC_ERR_NULL;
    const uintptr_t al = reinterpret_cast<uintptr_t>(hidden) | reinterpret_cast<uintptr_t>(input_norm_w) |
                         reinterpret_cast<uintptr_t>(q_proj_w) | reinterpret_cast<uintptr_t>(k_proj_w) |
                         reinterpret_cast<uintptr_t>(v_proj_w) | reinterpret_cast<uintptr_t>(o_proj_w);
    if (al & 15) return SUPERSONIC_ERR_RANGE;
    const bool fp8 = kv_dtype == SUPERSONIC_KV_FP8_E4M3;
    const LayerWs L = layer_ws(static_cast<int>(B), static_cast<int>(Hq), static_cast<int>(Hkv), static_cast<int>(D),
                               static_cast<int>(max_kv_len));
    if (workspace_bytes < L.total) return SUPERSONIC_ERR_WORKSPACE;
    LayerParams P{};
    if (int rc = make_view(cache, fp8, &P.dec.kv)) return rc;
    ScopedDevice scoped(static_cast<int>(device_ordinal));
    uint8_t* ws = static_cast<uint8_t*>(workspace);
    uint16_t* q_proj = reinterpret_cast<uint16_t*>(ws + L.q_proj);
    uint16_t* k_new = reinterpret_cast<uint16_t*>(ws + L.k_new);
    uint16_t* v_new = reinterpret_cast<uint16_t*>(ws + L.v_new);
    uint16_t* attn = reinterpret_cast<uint16_t*>(ws + L.attn);
    P.bar = reinterpret_cast<unsigned*>(ws + L.bar);
    P.ids = reinterpret_cast<unsigned*>(ws + L.ids);
    P.layer_len = static_cast<int>(max_kv_len);
    // phase 1
    SkinnyLdsParams& q = P.qkv;
    q.xn = hidden;
    q.norm_w = static_cast<const uint16_t*>(input_norm_w);
    q.norm_eps = eps;
    q.w[0] = static_cast<const uint16_t*>(q_proj_w);
    q.w[1] = static_cast<const uint16_t*>(k_proj_w);
    q.w[2] = static_cast<const uint16_t*>(v_proj_w);
    q.out[0] = q_proj;
    q.out[1] = k_new;
    q.out[2] = v_new;
    q.n_seg[0] = static_cast<int>(nq);
    q.n_seg[1] = q.n_seg[2] = static_cast<int>(nkv);
    q.cb_end[0] = static_cast<int>(nq / kSkinnyCols);
    q.cb_end[1] = q.cb_end[0] + static_cast<int>(nkv / kSkinnyCols);
    q.cb_end[2] = q.cb_end[1] + static_cast<int>(nkv / kSkinnyCols);
    q.m = static_cast<int>(B);
    q.k = static_cast<int>(hid);
    // phase 2: the fused decode step's parameters (supersonic_attn_gfx950_decode)
    DecodeParams& p = P.dec;
    p.q = q_proj;
    p.q_bstride = static_cast<int64_t>(nq);
    p.q_hstride = 2 * static_cast<int64_t>(D);
    p.lens = positions;
    p.len_plus = 1;
    p.Hq = static_cast<int>(Hq);
    p.Hkv = static_cast<int>(Hkv);
    p.G = static_cast<int>(Hq / Hkv);
    p.ragged = 1;
    p.B = static_cast<int>(B);
    p.min_chunk = std::max(64, []() {
        const char* v = getenv("SUPERSONIC_DECODE_MIN_CHUNK");
        return (v && *v) ? atoi(v) : 128;
    }());
    p.det = []() {
        const char* v = getenv("SUPERSONIC_DECODE_DETERMINISTIC");
        return (v && *v) ? (atoi(v) != 0) : 0;
    }();
    p.scale_log2 = scale * kLog2e;
    p.fused = 1;
    p.k_new = k_new;
    p.v_new = v_new;
    p.q_norm_w = static_cast<const uint16_t*>(q_norm_w);
    p.k_norm_w = static_cast<const uint16_t*>(k_norm_w);
    p.cos_t = static_cast<const uint16_t*>(cos_table);
    p.sin_t = static_cast<const uint16_t*>(sin_table);
    p.half_rot = static_cast<int>(rotary_dim / 2);
    p.eps = qk_eps;
    p.part_o = reinterpret_cast<float*>(ws + L.part_o);
    p.part_ml = reinterpret_cast<float*>(ws + L.part_ml);
    p.arrivals = reinterpret_cast<unsigned*>(ws + L.arrivals);
    p.arr_stride = arrival_stride(static_cast<long long>(B) * Hkv, static_cast<long long>(kLayerArrivalBytes / 4));
    p.gate = q_proj + D;
    p.g_bstride = static_cast<int64_t>(nq);
    p.g_hstride = 2 * static_cast<int64_t>(D);
    p.out = attn;
    // phase 3
    SkinnyLdsParams& o = P.op;
    o.x = attn;
    o.w[0] = o.w[1] = o.w[2] = static_cast<const uint16_t*>(o_proj_w);
    o.out[0] = o.out[1] = o.out[2] = hidden;
    o.res = hidden;
    o.n_seg[0] = o.n_seg[1] = o.n_seg[2] = static_cast<int>(hid);
    o.cb_end[0] = o.cb_end[1] = o.cb_end[2] = static_cast<int>(hid / kSkinnyCols);
    o.m = static_cast<int>(B);
    o.k = static_cast<int>(adim);
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int dev = static_cast<int>(device_ordinal);
    const ProfileEvents ev = take_profile_events();
    if (ev.before) (void)hipEventRecord(ev.before, st);
    int rc;
    const bool f32 = hidden_dtype == SUPERSONIC_DTYPE_F32;
    if (D == 256) {
        if (f32) rc = fp8 ? launch_layer<float, true, 256>(dev, st, P) : launch_layer<float, false, 256>(dev, st, P);
        else rc = fp8 ? launch_layer<bf16_t, true, 256>(dev, st, P) : launch_layer<bf16_t, false, 256>(dev, st, P);
    } else {
        if (f32) rc = fp8 ? launch_layer<float, true, 128>(dev, st, P) : launch_layer<float, false, 128>(dev, st, P);
        else rc = fp8 ? launch_layer<bf16_t, true, 128>(dev, st, P) : launch_layer<bf16_t, false, 128>(dev, st, P);
    }
    if (rc) return rc;
    if (ev.after) (void)hipEventRecord(ev.after, st);
    return 0;
}
