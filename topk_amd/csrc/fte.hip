// FTE (full-table evaluation) top-k on gfx950.
//
// Reference: cpu/TPAc.h:118-358 (scoring order, heap semantics) and the
// empty GPU stub gpu/GFA.h:47-50.  A query is one launch on the context's
// stream (fte_stream_kernel; exact mode: a seed launch before it):
//
//  1. threshold tau, a ranking key:
//       - own sample (stores up to 2^19 objects, calls that re-run on a bad
//         guess): every workgroup takes the same sample of 4096 objects and
//         the same element of it.
//       - shared sample: the first 32 workgroups score up to 128 chunks of
//         1024 objects spread over the id range and publish their best; tau
//         is the ks-th largest of the whole sample.  The other workgroups
//         have their first tile in flight meanwhile; what is late they score
//         themselves.  A guess like the own sample, checked at the end (>= k
//         candidates).
//       - exact (fte_seed_kernel): contiguous chunks [0, P); the prefix's
//         k-th key is a proven lower bound of the global k-th key, and the
//         prefix's top k are written to the candidate list.
//  2. stream: each workgroup streams whole tiles of contiguous column
//     segments, scores stay in registers, and keys >= tau go to the
//     workgroup's own candidate slots (wave ballot + one LDS atomic per
//     wave; no global atomic).  No barrier in the loop: a pure HBM stream.
//  3. select: the last workgroup to finish scans the per-workgroup counts,
//     checks the candidate total, selects the exact top k and writes them
//     best first, to device memory or straight to pinned host memory.
//
// Exactness: with c >= k candidates of key >= tau, every other object has a
// key < tau and is beaten by c >= k objects, so the top k are among the
// candidates.  Too few candidates (a sample guess that was too high) raise
// STATUS_RETRY, too many for the buffer STATUS_OVERFLOW; the host then runs
// the exact mode, with an n-entry buffer if needed.
#include <string.h>

#include <algorithm>
#include <cmath>
#include <mutex>

#include "device.hpp"
#include "emit.hpp"
#include "fte_plan.hpp"
#include "internal.hpp"
#include "select.hpp"

namespace topk {

constexpr int SEED_BS = 256;
constexpr int FINAL_BS = 512;            // separate final select
constexpr int FINAL_KPT = 16;            // candidate keys per final-select thread (8192 in registers)
constexpr int FLAT_BS = 1024;            // fallback final select over a large flat list

// Runtime-width scores of VPT float4 vectors v, v + step, ... (at most last): the
// loads of G columns, eight a lane, are issued before the first of them is used
// (a loop of one column per step waited on memory once per term), terms in
// query order; real-data scores divide after every term.
template <bool NT>
__device__ __forceinline__ f4 ld_col(const float *p) {
    if constexpr (NT) return ld_stream(p);
    else return *reinterpret_cast<const f4 *>(p);
}
template <int VPT, bool NT = true, int G = VPT < 8 ? 8 / VPT : 1>
__device__ __forceinline__ void score_wide(const QCols &q, uint32_t v, uint32_t step, uint32_t last, f4 (&acc)[VPT]) {
#pragma unroll
    for (int u = 0; u < VPT; u++) acc[u] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    for (uint32_t j0 = 0; j0 < q.m; j0 += G) {
        f4 x[G][VPT];
#pragma unroll
        for (int t = 0; t < G; t++)
            if (j0 + t < q.m) {
#pragma unroll
                for (int u = 0; u < VPT; u++) x[t][u] = ld_col<NT>(q.col[j0 + t] + (uint64_t)tile_vec(v + u * step, last) * 4);
            }
#pragma unroll
        for (int t = 0; t < G; t++)
            if (j0 + t < q.m) {
#pragma unroll
                for (int u = 0; u < VPT; u++) {
                    f4 p = x[t][u] * q.w[j0 + t];
                    acc[u] = acc[u] + p;
                    if (q.div != 0.0f) acc[u] = acc[u] / q.div;
                }
            }
    }
}

// Score of the 4 objects of float4 vector v: acc = fl(acc + fl(x*w)) in
// attribute order, accumulator starting at +0 (cpu/TPAc.h:129-142).
// NT: nontemporal loads (data read once).
template <int M, bool NT = true>
__device__ __forceinline__ f4 score_vec(const QCols &q, uint64_t v) {
    f4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (M > 0) {
        f4 x[M];
#pragma unroll
        for (int j = 0; j < M; j++) x[j] = ld_col<NT>(q.col[j] + v * 4);
#pragma unroll
        for (int j = 0; j < M; j++) {
            f4 p = x[j] * q.w[j];
            acc = acc + p;
        }
    } else {
        f4 s1[1];
        score_wide<1, NT, 16>(q, (uint32_t)v, 0, 0xFFFFFFFFu, s1);
        acc = s1[0];
    }
    return acc;
}

// ---------------------------------------------------------------------------
// 1. seed pass
// ---------------------------------------------------------------------------
// Block b scores objects [b*chunk_stride, +256*OPT) of the first n_eff objects.
// total_valid = number of non-zero keys the blocks deposit in blk.
template <int M, int OPT>
__global__ __launch_bounds__(SEED_BS) void fte_seed_kernel(QCols q, uint64_t n_eff, uint64_t chunk_stride,
                                                           uint32_t ks, uint32_t total_valid,
                                                           uint64_t *__restrict__ blk,
                                                           uint64_t *__restrict__ pre,
                                                           FteState *__restrict__ st,
                                                           const uint32_t *__restrict__ gate) {
    __shared__ SelectScratch ss;
    __shared__ uint32_t is_last;
    if (gate && *gate == 0) return;  // the pass this one backs up settled the query
    const uint32_t tid = threadIdx.x;
    const uint64_t base = (uint64_t)blockIdx.x * chunk_stride;

    constexpr uint32_t TILE = SEED_BS * OPT;
    RegKeys<OPT> rk;
#pragma unroll
    for (int j = 0; j < OPT / 4; j++) {
        const uint64_t v = base / 4 + j * SEED_BS + tid;
        const f4 s = score_vec<M>(q, v);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint64_t id = v * 4 + e;
            rk.k[j * 4 + e] = id < n_eff ? rkey(s[e], (uint32_t)id) : 0ull;
        }
    }
    const uint64_t left = n_eff > base ? n_eff - base : 0;
    const uint32_t valid = (uint32_t)(left < TILE ? left : TILE);
    uint64_t thr = 1;
    if (valid > ks) thr = block_kth_largest<SEED_BS>(rk, valid, ks, ss);
    uint64_t *out = blk + (uint64_t)blockIdx.x * ks;
    const uint32_t got = block_gather_ge<SEED_BS>(rk, thr, out, ss);
    for (uint32_t i = got + tid; i < ks; i += SEED_BS) out[i] = 0;
    // the last block to arrive merges the block winners
    __threadfence();
    __syncthreads();
    if (tid == 0) is_last = (atomicAdd(&st->arrive, 1u) == gridDim.x - 1);
    __syncthreads();
    if (!is_last) return;
    __threadfence();

    const uint32_t nk = gridDim.x * ks;
    uint64_t tau = 1;
    if (total_valid > ks) tau = block_kth_largest<SEED_BS>(MemKeys<SEED_BS>{blk, nk}, total_valid, ks, ss);
    uint32_t c = 0;
    if (pre) c = block_gather_ge<SEED_BS>(MemKeysUniform<SEED_BS>{blk, nk}, tau, pre, ss);
    if (tid == 0) {
        st->tau = tau;
        st->pre_count = c;
        st->arrive = 0;
    }
}

// ---------------------------------------------------------------------------
// final select + sort
// ---------------------------------------------------------------------------

// The ks-th largest of the keys the wave's lanes hold (NPL per lane; 0: no
// key) -- 0 with fewer than ks keys -- by bisection on ballot counts, score
// half first, then the id half among the keys that share the score (only if
// several do).  32 steps of NPL compares whatever ks is (rounds of wave
// maxima cost ks x 0.4 us).
template <int NPL>
__device__ __forceinline__ uint64_t wave_kth_bisect(const uint64_t (&v)[NPL], uint32_t ks) {
    uint32_t t = 0;
    for (int b = 31; b >= 0; b--) {
        const uint32_t c = t | (1u << b);
        uint32_t cnt = 0;
#pragma unroll
        for (int j = 0; j < NPL; j++) cnt += (uint32_t)__popcll(__ballot((uint32_t)(v[j] >> 32) >= c));
        if (cnt >= ks) t = c;
    }
    if (t == 0) return 0;
    uint32_t above = 0, equal = 0;
#pragma unroll
    for (int j = 0; j < NPL; j++) {
        above += (uint32_t)__popcll(__ballot((uint32_t)(v[j] >> 32) > t));
        equal += (uint32_t)__popcll(__ballot((uint32_t)(v[j] >> 32) == t));
    }
    const uint32_t need = ks - above;  // >= 1
    uint32_t lo = 0;
    if (equal == need && equal == 1) {
        // one key holds the score: its id half
        uint32_t mine = 0;
#pragma unroll
        for (int j = 0; j < NPL; j++) mine |= (uint32_t)(v[j] >> 32) == t ? (uint32_t)v[j] : 0u;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) mine |= (uint32_t)__shfl_xor((int)mine, o, 64);
        lo = mine;
    } else {
        for (int b = 31; b >= 0; b--) {
            const uint32_t c = lo | (1u << b);
            uint32_t cnt = 0;
#pragma unroll
            for (int j = 0; j < NPL; j++)
                cnt += (uint32_t)__popcll(__ballot((uint32_t)(v[j] >> 32) == t && (uint32_t)v[j] >= c));
            if (cnt >= need) lo = c;
        }
    }
    return ((uint64_t)t << 32) | lo;
}

// The ks-th largest of the wave's keys (hi / lo as wave_pop_max's): rounds of
// maxima for a shallow rank (about 0.1 us each), else bisection.
template <int NPL>
__device__ __forceinline__ uint64_t wave_kth(uint32_t (&hi)[NPL], const uint32_t (&lo)[NPL], uint32_t ks) {
    uint64_t r = 0;
    if (ks <= 16) {
        for (uint32_t i = 0; i < ks; i++) r = wave_pop_max<NPL>(hi, lo);
        return r;
    }
    uint64_t v[NPL];
#pragma unroll
    for (int j = 0; j < NPL; j++) v[j] = hi[j] ? ((uint64_t)hi[j] << 32) | lo[j] : 0ull;
    return wave_kth_bisect<NPL>(v, ks);
}

// The wave's W (<= 64) largest keys, largest first, key i on lane i (0: fewer).
template <int NPL>
__device__ __forceinline__ uint64_t wave_top(uint32_t (&hi)[NPL], const uint32_t (&lo)[NPL], uint32_t W) {
    uint64_t mine = 0;
    for (uint32_t i = 0; i < W; i++) {
        const uint64_t key = wave_pop_max<NPL>(hi, lo);
        mine = lane_id() == i ? key : mine;
    }
    return mine;
}

// The same of the cnt <= 64 * NPL keys at p (LDS).
template <int NPL>
__device__ __forceinline__ uint64_t top_of_list(const uint64_t *p, uint32_t cnt, uint32_t W) {
    uint32_t hi[NPL], lo[NPL];
#pragma unroll
    for (int j = 0; j < NPL; j++) {
        const uint32_t i = j * 64 + lane_id();
        const uint64_t v = i < cnt ? p[i] : 0ull;
        hi[j] = (uint32_t)(v >> 32);
        lo[j] = (uint32_t)v;
    }
    return wave_top<NPL>(hi, lo, W);
}

// Shared sample: its chunks (1024 objects each, at multiples of chunk_stride)
// are dealt into SAMPLE_WGS pieces, chunk c to piece c % SAMPLE_WGS, and the W
// largest keys of piece p are published at st->win[p * W ...].  The workgroup
// with index p takes piece p; of fewer workgroups, any takes the pieces left.
//
// No workgroup waits on another's progress: one that has polled for a while
// in vain takes a missing piece itself and polls again.  A piece's winners
// depend on the query alone, so it does not matter who publishes them or how
// often, every workgroup gets the same tau, and after at most 32 pieces of
// its own work all of them are there.  (The first workgroups of one launch
// start first, but two launches in flight may hold each other's compute
// units, each XCD starting another of them first.)
struct SampleScratch {
    uint64_t keys[STREAM_NW * SAMPLE_MAX_W];
};
constexpr uint32_t NO_PIECE = 0xFFFFFFFFu;
template <int M>
__device__ __forceinline__ void sample_publish(const QCols &q, uint64_t n, uint32_t chunks, uint64_t chunk_stride,
                                               uint32_t W, uint32_t piece, FteState *__restrict__ st,
                                               SampleScratch &sc) {
    const uint32_t tid = threadIdx.x, wave = tid / 64, lane = lane_id();
    constexpr uint32_t PER = STREAM_BS * 4 / SAMPLE_TILE;  // chunks per step of the workgroup
    {
        uint32_t hi[4 * SAMPLE_VEC], lo[4 * SAMPLE_VEC];
#pragma unroll
        for (int u = 0; u < SAMPLE_VEC; u++) {
            const uint32_t c = piece + (u * PER + tid / (SAMPLE_TILE / 4)) * SAMPLE_WGS;
            const uint64_t v = (c < chunks ? c * chunk_stride : 0ull) / 4 + tid % (SAMPLE_TILE / 4);
            const f4 s = score_vec<(M > 8 ? 0 : M)>(q, v);  // 16 columns at once would spill
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint64_t id = v * 4 + e;
                hi[u * 4 + e] = c < chunks && id < n ? okey(s[e]) : 0u;
                lo[u * 4 + e] = 0xFFFFFFFFu - (uint32_t)id;
            }
        }
        const uint64_t mine = wave_top<4 * SAMPLE_VEC>(hi, lo, W);
        if (lane < W) sc.keys[wave * W + lane] = mine;
    }
    __syncthreads();
    if (wave == 0) {
        const uint64_t mine = W <= 16 ? top_of_list<STREAM_NW * 16 / 64>(sc.keys, STREAM_NW * W, W)
                                      : top_of_list<STREAM_NW * SAMPLE_MAX_W / 64>(sc.keys, STREAM_NW * W, W);
        if (lane < W) store_agent(reinterpret_cast<uint64_t *>(&st->win[piece * W + lane]), mine ? mine : 1ull);
    }
    __syncthreads();
}

// The threshold of the sample's ks-th key with ks < k.  Among tied scores a
// chunk's ids are consecutive, and the key of one of them alone would admit
// only that chunk's: ks candidates and a second run on any column with more
// than ks ties in its first chunk.  So the id half is widened, to four times the
// ids that k ties take at the rate of the chunk so far, at most to the next
// chunk.  (To the next chunk always, the select of n / 128 ties cost more than
// the second run of one column: 2^24 equal objects, k = 10, 194 us against 122.)
__device__ __forceinline__ uint64_t sample_threshold(uint64_t key, uint64_t chunk_stride, uint32_t k, uint32_t ks) {
    if (ks >= k || key <= 1) return key;  // a proven bound; no key, or the mark of a piece without one
    const uint32_t id = rkey_id(key), stride = (uint32_t)chunk_stride, at = id % stride;
    const uint32_t more = min(stride - at, 4 * (min(at, SAMPLE_TILE) + 1) * ((k + ks - 1) / ks));
    const uint64_t end = (uint64_t)id + more;
    return (key & ~0xFFFFFFFFull) | (end < 0xFFFFFFFFull ? 0xFFFFFFFFull - end : 0ull);
}

// Consumer side, one wave, W <= 16: polls the winners (a winner is its own flag: a
// store and a load apart, where a counter would add two more trips to
// memory).  With all of them there, tau is the ks-th largest and the result
// NO_PIECE; after `polls` tries it is a missing piece, the first one from this
// workgroup's own number on, so that many workgroups take different ones.
__device__ __forceinline__ uint32_t sample_tau(FteState *__restrict__ st, uint32_t W, uint32_t ks, uint32_t polls,
                                               uint64_t &tau) {
    constexpr int NPL = SAMPLE_WGS * 16 / 64;
    const uint32_t nwin = SAMPLE_WGS * W;
    for (uint32_t s = 1;; s++) {
        uint32_t hi[NPL], lo[NPL];
        bool all = true;
#pragma unroll
        for (int j = 0; j < NPL; j++) {
            const uint32_t i = j * 64 + lane_id();
            uint64_t v = 0;
            if (i < nwin) {
                v = __hip_atomic_load(&st->win[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                all = all && v != 0;
            }
            hi[j] = (uint32_t)(v >> 32);
            lo[j] = (uint32_t)v;
        }
        if (!__ballot(!all)) {
            tau = wave_kth<NPL>(hi, lo, ks);
            return NO_PIECE;
        }
        if (s >= polls) {
            const uint32_t from = blockIdx.x % SAMPLE_WGS;
            uint32_t near = 0;  // SAMPLE_WGS less the steps from there to the nearest missing piece
#pragma unroll
            for (int j = 0; j < NPL; j++) {
                const uint32_t i = j * 64 + lane_id(), p = i / W;
                const uint32_t left = p >= from ? SAMPLE_WGS - (p - from) : from - p;
                near = i < nwin && (hi[j] | lo[j]) == 0 && left > near ? left : near;
            }
            return (from + SAMPLE_WGS - wave_max_u32(near)) % SAMPLE_WGS;
        }
        __builtin_amdgcn_s_sleep(8);
    }
}

// The same by the whole workgroup, a winner a thread, for any W: more than
// eight winners a lane and the tile in flight don't fit the registers.
__device__ __forceinline__ uint32_t sample_tau_deep(FteState *__restrict__ st, uint32_t W, uint32_t ks, uint32_t polls,
                                                    uint64_t &tau, uint32_t &s_near, SelectScratchT<256> &ss) {
    const uint32_t i = threadIdx.x;
    const bool mine = i < SAMPLE_WGS * W;
    for (uint32_t s = 1;; s++) {
        uint64_t v = 0;
        if (mine) v = __hip_atomic_load(&st->win[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (i == 0) s_near = 0;
        __syncthreads();
        if (mine && v == 0) {
            const uint32_t p = i / W, from = blockIdx.x % SAMPLE_WGS;
            atomicMax(&s_near, p >= from ? SAMPLE_WGS - (p - from) : from - p);
        }
        __syncthreads();
        const uint32_t near = s_near;
        __syncthreads();
        if (near == 0) {
            RegKeys<1> rk;
            rk.k[0] = v;
            tau = block_kth_largest<STREAM_BS, RegKeys<1>, 8>(rk, SAMPLE_WGS * W, ks, ss);
            return NO_PIECE;
        }
        if (s >= polls) return (blockIdx.x % SAMPLE_WGS + SAMPLE_WGS - near) % SAMPLE_WGS;
        __builtin_amdgcn_s_sleep(8);
    }
}

// Own sample: tau of a stream workgroup from the same OWN_OBJS objects in
// every workgroup -- OWN_SPOTS runs of 16 objects at the starts of equal
// strata of the store (each wave's runs alternate over the whole range) --
// as the ks-th largest of their keys, from each wave's W largest.  The id
// half is widened to the end of the stratum the key lies in: among tied
// scores a run's ids are consecutive, and the key of one of them alone would
// admit only that run's ids.
struct OwnScratch {
    uint64_t keys[STREAM_NW * OWN_MAX_W];
    uint64_t tau;
};
template <int M>
__device__ __forceinline__ uint64_t own_sample_tau(const QCols &q, uint64_t n, uint32_t ks, uint32_t W, OwnScratch &os) {
    const uint32_t wave = threadIdx.x / 64, lane = lane_id();
    const uint32_t lines = (uint32_t)((n + 15) / 16);
    {
        uint32_t hi[4 * OWN_VEC], lo[4 * OWN_VEC];
#pragma unroll
        for (int u = 0; u < OWN_VEC; u++) {
            const uint32_t spot = lane / 4 * (STREAM_NW * OWN_VEC) + wave * OWN_VEC + u;
            const uint32_t v = (uint32_t)((uint64_t)spot * lines / OWN_SPOTS) * 4 + (lane & 3);
            const f4 s = score_vec<(M > 8 ? 0 : M), false>(q, v);  // every workgroup reads them: cached
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t o = v * 4 + e;
                hi[u * 4 + e] = o < n ? okey(s[e]) : 0u;
                lo[u * 4 + e] = 0xFFFFFFFFu - o;
            }
        }
        const uint64_t mine = wave_top<4 * OWN_VEC>(hi, lo, W);
        if (lane < W) os.keys[wave * W + lane] = mine;
    }
    __syncthreads();
    if (wave == 0) {
        constexpr int NPL = STREAM_NW * OWN_MAX_W / 64;
        uint32_t hi[NPL], lo[NPL];
#pragma unroll
        for (int j = 0; j < NPL; j++) {
            const uint32_t i = j * 64 + lane;
            const uint64_t v = i < STREAM_NW * W ? os.keys[i] : 0ull;
            hi[j] = (uint32_t)(v >> 32);
            lo[j] = (uint32_t)v;
        }
        uint64_t tau = wave_kth<NPL>(hi, lo, ks);
        if (tau) {
            const uint32_t id = rkey_id(tau);
            const uint64_t next = (uint64_t)(id / 16) * OWN_SPOTS / lines + 1;  // the next run
            const uint64_t end = next * lines / OWN_SPOTS * 16;
            if (end > id) tau = (tau & ~0xFFFFFFFFull) | (0xFFFFFFFFu - (uint32_t)end);
        }
        if (lane == 0) os.tau = tau;
    }
    __syncthreads();
    return os.tau;
}

// ---------------------------------------------------------------------------
// 2. stream pass
// ---------------------------------------------------------------------------
// One stream pass.
struct StreamArgs {
    uint64_t n, obj_begin, ntiles;
    uint64_t nstatic;      // tiles dealt out in turn; the rest as workgroups get free
    FteState *st;
    CandSet cs;
    int tau;               // TAU_*: every object a candidate, st->tau, the shared sample, the own sample
    uint32_t ks;           // rank of tau in the sample
    uint32_t chunks;       // of the shared sample
    uint32_t W;            // winners per piece of the shared sample, or per wave of the own one
    uint64_t chunk_stride; // objects between the chunks' first objects
    uint32_t polls;        // tries before a workgroup takes a missing piece of the sample
    int select;            // the last workgroup selects and emits (else a later launch does)
    uint32_t cap, kp2, k, kreq;
    FinalOut fo;
    const uint32_t *gate;
};

// Each workgroup streams whole tiles of TILE = 4096*VPT objects: for every
// queried column it reads one contiguous TILE*4-byte segment (VPT float4 per
// lane).  Block-contiguous segments keep HBM near 88% of peak where a
// thread-level grid stride over the columns stays near 72%.  A tile may end
// past the store: its lanes there read the last vector (tile_vec).
//
// One workgroup of 16 waves per CU holds 8 or more loads of 16 bytes per lane
// in flight, which is all HBM needs (512 to 3072 workgroups of 256 threads
// stream at the same 6.8 TB/s), leaves few arrivals at the end and 1024
// threads to the select.  Of two workgroups on a CU the older one goes
// first: two of 512 threads per CU ended between 203 and 334 us at N = 2^26.
//
// XCDs do not run at one speed either (at N = 2^26 four of the eight are 6%
// behind), so the last tiles are handed out by a ticket, taken while the
// tile before is processed (device atomics on one address serialise at
// about 20 ns, so only the last ones).
//
// Bound by HBM above a few million objects: at N = 2^26, m = 8 the launch takes
// 332.7 us on average under a kernel trace (6.45 TB/s with its sample and
// select; as launches of their own sample, stream and select took 13.8 + 317.2
// + 17.5), and two queries in flight hide those, 6.9 TB/s.  Below, by the chain
// of launch, sample, arrival and select.  A synchronous call, before (three
// launches, two result copies) and now: 16k objects 50.7 -> 34.0 us, 2^20 x 4
// 64.0 -> 36.2, 8M x 7 divided 115 -> 78, 4.2M x 20 with k = 1000 223 -> 107,
// 2^26 x 8 374 -> 344; 32 queued queries of 16M x 5 1945 -> 1844.  At 2^20 tau is
// known after 10 us, the last workgroup arrives at 13 and has selected at 19.
//
// The select runs in the last workgroup to finish.  Its inputs cross XCDs
// without an L2 write-back per workgroup: candidates, counts and spilled
// keys are agent-scope (write-through) stores, each wave waits for its own
// before the workgroup takes its arrival ticket, and the last workgroup
// invalidates its caches once.  Arrivals are counted in ARRIVE_GROUPS
// groups on cache lines of their own and then across groups: on one counter
// they serialise at about 20 ns each.
template <int M, int VPT>
__global__ __launch_bounds__(STREAM_BS, 4) void fte_stream_kernel(QCols q, StreamArgs a) {
    constexpr uint32_t TILE = STREAM_BS * 4 * VPT;
    extern __shared__ uint64_t dyn[];  // cap keys | block offsets, later cap keys
    __shared__ uint32_t lcount, is_last, s_next[2], s_piece;
    __shared__ uint64_t s_tau;
    __shared__ union {
        OwnScratch own;
        SampleScratch sam;
        FuseScratch sel;
    } sh;
    if (a.gate && *a.gate == 0) return;
    const uint32_t lane = lane_id();
    if (threadIdx.x == 0) lcount = 0;
    // the first tile's loads are in flight while tau is found
    constexpr int MX = M > 0 ? M : 1;
    f4 x[MX][VPT];
    uint64_t t = blockIdx.x;
    const uint32_t last = (uint32_t)((a.n - 1) / 4);
    auto load = [&](uint32_t v0) {
        if constexpr (M > 0) {
#pragma unroll
            for (int j = 0; j < M; j++)
#pragma unroll
                for (int u = 0; u < VPT; u++)
                    x[j][u] = ld_stream(q.col[j] + (uint64_t)tile_vec(v0 + u * STREAM_BS, last) * 4);
        }
    };
    const uint32_t first_v = (uint32_t)((a.obj_begin + t * TILE) / 4) + threadIdx.x;  // the grid never exceeds the tiles
    uint64_t tau = 0;
    if (a.tau == TAU_SHARED) {
        auto publish = [&](uint32_t piece) __attribute__((always_inline)) {
            sample_publish<M>(q, a.n, a.chunks, a.chunk_stride, a.W, piece, a.st, sh.sam);
        };
        if (blockIdx.x < SAMPLE_WGS) publish(blockIdx.x);
        uint32_t piece = NO_PIECE;
        const bool deep = a.W > 16;
        if (!deep) {
            load(first_v);
            if (threadIdx.x < 64) {
                uint64_t v = 0;
                const uint32_t p = sample_tau(a.st, a.W, a.ks, a.polls, v);
                if (lane == 0) {
                    s_tau = sample_threshold(v, a.chunk_stride, a.k, a.ks);
                    s_piece = p;
                }
            }
            __syncthreads();
            tau = s_tau;
            piece = __builtin_amdgcn_readfirstlane(s_piece);
        }
        if (deep || piece != NO_PIECE) {
            for (;;) {
                if (piece != NO_PIECE) publish(piece);
                piece = sample_tau_deep(a.st, a.W, a.ks, a.polls, tau, s_piece, sh.sel.rs);
                if (piece == NO_PIECE) break;
            }
            tau = sample_threshold(tau, a.chunk_stride, a.k, a.ks);
            uint32_t v0 = first_v;
            asm volatile("" : "+v"(v0));  // the addresses are made anew, not kept over the sample
            load(v0);
        }
    } else {
        load(first_v);
        if (a.tau == TAU_OWN) {
            tau = own_sample_tau<M>(q, a.n, a.ks, a.W, sh.own);
        } else {
            if (a.tau == TAU_STATE) tau = a.st->tau;
            __syncthreads();
        }
    }
    const uint32_t tau_hi = (uint32_t)(tau >> 32);
    const CandSet &cs = a.cs;
    uint64_t *my = cs.keys + (uint64_t)blockIdx.x * cs.slot;
    for (bool first = true, par = false;; first = false) {
        // past the dealt tiles, the next one's ticket travels while this one is processed
        const bool draw = t + gridDim.x >= a.nstatic && a.nstatic < a.ntiles;  // uniform
        uint32_t nx = 0;
        if (draw && threadIdx.x == 0)
            nx = __hip_atomic_fetch_add(&a.st->ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t v0 = (uint32_t)((a.obj_begin + t * TILE) / 4) + threadIdx.x;
        f4 s[VPT];
        if constexpr (M > 0) {
            if (!first) load(v0);
#pragma unroll
            for (int u = 0; u < VPT; u++) {
                f4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int j = 0; j < M; j++) {
                    f4 p = x[j][u] * q.w[j];
                    acc = acc + p;
                }
                s[u] = acc;
            }
        } else {
            score_wide<VPT>(q, v0, STREAM_BS, last, s);
        }
        // filter: key >= tau (score key first; the id only matters on ties)
        uint32_t npass = 0;
        uint64_t kk[VPT * 4];
#pragma unroll
        for (int u = 0; u < VPT; u++) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint64_t id = (uint64_t)(v0 + u * STREAM_BS) * 4 + e;
                const uint32_t ok = okey(s[u][e]);
                const uint64_t key = rkey_from_okey(ok, (uint32_t)id);
                const bool p = ok >= tau_hi && key >= tau && id < a.n;
                kk[u * 4 + e] = p ? key : 0ull;
                npass += p ? 1u : 0u;
            }
        }
        if (__ballot(npass != 0)) {
            const uint32_t incl = wave_incl_scan(npass);
            uint32_t base = 0;
            if (lane == 63) base = atomicAdd(&lcount, incl);
            base = __shfl(base, 63, 64);
            const uint32_t wtotal = __shfl(incl, 63, 64);
            // positions >= slot spill to the shared region (one global atomic per wave)
            const uint32_t first_spill = base > cs.slot ? base : cs.slot;
            const uint32_t nspill = base + wtotal > first_spill ? base + wtotal - first_spill : 0u;
            uint32_t sbase = 0;
            if (nspill) {
                if (lane == 63) sbase = atomicAdd(&a.st->spill, nspill);
                sbase = __shfl(sbase, 63, 64);
            }
            uint32_t pos = base + incl - npass;
#pragma unroll
            for (int j = 0; j < VPT * 4; j++) {
                if (kk[j]) {
                    if (pos < cs.slot) {
                        store_agent(my + pos, kk[j]);
                    } else {
                        const uint32_t sp = sbase + (pos - first_spill);
                        if (sp < cs.spill_cap) store_agent(cs.spill + sp, kk[j]);
                    }
                    pos++;
                }
            }
        }
        if (draw) {
            if (threadIdx.x == 0) s_next[par] = nx;
            __syncthreads();
            t = a.nstatic + s_next[par];
            par = !par;
        } else {
            t += gridDim.x;
        }
        if (t >= a.ntiles) break;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's candidates have reached memory
    __syncthreads();
    if (threadIdx.x == 0) {
        __hip_atomic_store(&cs.counts[blockIdx.x], lcount < cs.slot ? lcount : cs.slot, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
        if (a.select) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            is_last = last_to_arrive(a.st);
        }
    }
    if (!a.select) return;
    __syncthreads();
    if (!is_last) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    fused_select<STREAM_BS>(a.st, cs, a.k, a.kreq, a.cap, a.kp2, a.fo, dyn, dyn + a.cap, sh.sel);
}

// Final select as a launch of its own (one workgroup): stores that fit the
// exact seed's prefix.
__global__ __launch_bounds__(FINAL_BS) void fte_final_kernel(FteState *__restrict__ st, CandSet cs, uint32_t k,
                                                             uint32_t kreq, FinalOut fo,
                                                             const uint32_t *__restrict__ gate) {
    __shared__ uint32_t off[MAX_STREAM_GRID];
    if (gate && *gate == 0) return;
    __shared__ uint64_t top[TOPK_MAX_K];
    __shared__ uint64_t sorted[TOPK_MAX_K];
    __shared__ uint32_t wsum[FINAL_BS / 64];
    __shared__ uint32_t total;
    __shared__ SelectScratch ss;
    const uint32_t tid = threadIdx.x;
    // per-block counts -> LDS (coalesced), then exclusive offsets in place
    for (uint32_t b = tid; b < cs.nblk; b += FINAL_BS) off[b] = cs.counts[b];
    __syncthreads();
    const uint32_t per = (cs.nblk + FINAL_BS - 1) / FINAL_BS;
    const uint32_t b0 = tid * per < cs.nblk ? tid * per : cs.nblk;
    const uint32_t b1 = b0 + per < cs.nblk ? b0 + per : cs.nblk;
    uint32_t mine = 0;
    for (uint32_t b = b0; b < b1; b++) mine += off[b];
    uint32_t run = block_excl_scan<FINAL_BS>(mine, wsum, &total);
    for (uint32_t b = b0; b < b1; b++) {
        const uint32_t c = off[b];
        off[b] = run;
        run += c;
    }
    const uint32_t spilled = st->spill;
    const uint32_t nspill = spilled < cs.spill_cap ? spilled : cs.spill_cap;
    __syncthreads();
    if (tid == 0) st->spill = 0;  // ready for the next query
    const uint32_t npre = cs.pre ? st->pre_count : 0u;
    const uint32_t c = npre + total + nspill;
    const uint32_t bad = spilled > cs.spill_cap ? STATUS_OVERFLOW : (c < kreq ? STATUS_RETRY : 0u);
    if (bad) {
        if (tid == 0) {
            st->status |= bad;
            if (fo.status) *fo.status = bad;
        }
        return;
    }
    if (tid == 0) {
        st->cand_last = c;
        if (fo.cand) *fo.cand = c;
    }
    const SlotView v{cs.pre, npre, cs.keys, cs.slot, off, cs.nblk, total, cs.spill};
    select_and_emit<FINAL_BS, FINAL_KPT>(v, c, k, fo, top, sorted, ss);
}

// Fallback path for candidate sets too large for the regular slots: the
// per-block counts are scanned into global offsets, every block copies its
// slot region into one flat array, and the final select reads that array.
__global__ __launch_bounds__(FLAT_BS) void cand_offsets_kernel(FteState *__restrict__ st, CandSet cs,
                                                               uint32_t *__restrict__ offsets,
                                                               uint64_t *__restrict__ flat) {
    __shared__ uint32_t wsum[FLAT_BS / 64];
    __shared__ uint32_t total;
    const uint32_t tid = threadIdx.x;
    const uint32_t per = (cs.nblk + FLAT_BS - 1) / FLAT_BS;
    const uint32_t b0 = tid * per < cs.nblk ? tid * per : cs.nblk;
    const uint32_t b1 = b0 + per < cs.nblk ? b0 + per : cs.nblk;
    uint32_t mine = 0;
    for (uint32_t b = b0; b < b1; b++) mine += cs.counts[b];
    const uint32_t npre = cs.pre ? st->pre_count : 0u;
    uint32_t run = npre + block_excl_scan<FLAT_BS>(mine, wsum, &total);
    for (uint32_t b = b0; b < b1; b++) {
        offsets[b] = run;
        run += cs.counts[b];
    }
    for (uint32_t i = tid; i < npre; i += FLAT_BS) flat[i] = cs.pre[i];
    if (tid == 0) {
        st->total = npre + total;
        st->spill = 0;
    }
}

__global__ __launch_bounds__(256) void cand_compact_kernel(CandSet cs, const uint32_t *__restrict__ offsets,
                                                           uint64_t *__restrict__ flat) {
    const uint32_t b = blockIdx.x;
    const uint32_t c = cs.counts[b];
    const uint64_t *src = cs.keys + (uint64_t)b * cs.slot;
    uint64_t *dst = flat + offsets[b];
    for (uint32_t i = threadIdx.x; i < c; i += 256) dst[i] = src[i];
}

__global__ __launch_bounds__(FLAT_BS) void fte_final_flat_kernel(FteState *__restrict__ st,
                                                                  const uint64_t *__restrict__ flat, uint32_t k,
                                                                  uint32_t kreq, FinalOut fo) {
    __shared__ uint64_t top[TOPK_MAX_K];
    __shared__ uint64_t sorted[TOPK_MAX_K];
    __shared__ SelectScratch ss;
    const uint32_t c = st->total;
    if (c < kreq) {
        if (threadIdx.x == 0) {
            st->status |= STATUS_RETRY;
            if (fo.status) *fo.status = STATUS_RETRY;
        }
        return;
    }
    if (threadIdx.x == 0) {
        st->cand_last = c;
        if (fo.cand) *fo.cand = c;
    }
    select_and_emit<FLAT_BS, 8>(FlatView{flat}, c, k, fo, top, sorted, ss);
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

// Everything one run of the FTE pipeline needs besides the query: the store
// size, the stream, the scratch its kernels use and the launch shape.
struct FteRun {
    hipStream_t s;
    uint64_t n;
    FteState *st;
    uint64_t *blk;        // seed-pass block winners (SAMPLE_CHUNKS * TOPK_MAX_K keys)
    uint64_t *pre;        // exact-mode prefix keys (TOPK_MAX_K)
    uint32_t *counts;     // per-stream-block counts (MAX_STREAM_GRID)
    uint64_t *cand;       // candidate slots
    uint64_t cand_cap;
    bool big;             // cand holds every object of every block (exact re-run after an overflow)
    uint64_t *spill;
    uint32_t spill_cap;
    int vpt;              // 0: chosen from the query width
    uint32_t grid_cap;    // 0: default
    uint32_t polls;       // of the shared sample (0: default)
    const uint32_t *gate; // non-null: every kernel exits at once unless *gate != 0
    topk_ctx *timed;      // non-null: bracket the stream pass for topk_timing_*
};

// Enqueues the threshold pass, if the plan has one, and the stream pass (with
// the select, unless r.big leaves it to the caller) for one query on r.s.
// Returns the candidate set the select reads.
static CandSet fte_launch(const FteRun &r, uint32_t k, const QCols &q, const FinalOut &fo, int mode) {
    const uint64_t n = r.n;
    hipStream_t s = r.s;
    const SeedPlan sp = seed_plan(n, k, mode);
    uint64_t *pre = sp.first ? r.pre : nullptr;
    // kernels unrolled for the query width, or the runtime-width ones (the
    // only ones that divide real-data scores)
    const uint32_t msw = q.div != 0.0f ? 0u : q.m;
#define TK_SEED(MM)                                                                                              \
    hipLaunchKernelGGL((fte_seed_kernel<MM, SEED_TILE / SEED_BS>), dim3(sp.blocks), dim3(SEED_BS), 0, s, q, sp.n_eff, \
                       sp.stride, sp.ks, sp.total_valid, r.blk, pre, r.st, r.gate)
    if (sp.tau == TAU_STATE) TK_SWITCH_M(msw, TK_SEED);
#undef TK_SEED

    const StreamPlan pl = stream_plan(n, sp.first, q.m, r.big, r.vpt, r.grid_cap, r.cand_cap);
    const uint32_t g = pl.grid;
    StreamArgs a{};
    a.n = n;
    a.obj_begin = sp.first;
    a.ntiles = pl.ntiles;
    a.nstatic = pl.nstatic;
    a.st = r.st;
    a.tau = sp.tau;
    a.ks = sp.ks;
    a.chunks = sp.blocks;
    a.W = sp.W;
    a.chunk_stride = sp.stride;
    a.select = r.big ? 0 : 1;
    a.k = k;
    a.kreq = (uint32_t)(n < k ? n : k);
    a.fo = fo;
    a.gate = r.gate;
    // room in LDS for twice the candidates expected, and for the sort of k
    a.kp2 = next_pow2(k);
    uint32_t cap = FUSE_CAP_MIN;
    while (cap < FUSE_CAP_MAX && (cap < 2 * a.kp2 || cap < 2 * sp.expect)) cap += FUSE_CAP_MIN;
    a.cap = cap;
    a.polls = r.polls ? r.polls : (g < SAMPLE_WGS ? 1u : SAMPLE_POLLS);
    CandSet &cs = a.cs;
    cs.keys = r.cand;
    cs.counts = r.counts;
    cs.nblk = g;
    cs.pre = pre;
    cs.spill = r.spill;
    cs.spill_cap = r.spill_cap;
    cs.slot = pl.slot;
    if (g) {
        const size_t lds = sizeof(uint64_t) * ((size_t)cap + std::max((g + 3) / 2, cap));
        hipEvent_t ev0 = nullptr;
        if (r.timed) timing_begin(r.timed, s, ev0);
#define TK_STREAM(MM, VPT) \
    hipLaunchKernelGGL((fte_stream_kernel<stream_unroll(MM, VPT), VPT>), dim3(g), dim3(STREAM_BS), lds, s, q, a)
#define TK_STREAM1(MM) TK_STREAM(MM, 1)
#define TK_STREAM2(MM) TK_STREAM(MM, 2)
#define TK_STREAM4(MM) TK_STREAM(MM, 4)
#define TK_STREAM8(MM) TK_STREAM(MM, 8)
        switch (pl.vpt) {
            case 1: TK_SWITCH_M(msw, TK_STREAM1); break;
            case 2: TK_SWITCH_M(msw, TK_STREAM2); break;
            case 4: TK_SWITCH_M(msw, TK_STREAM4); break;
            default: TK_SWITCH_M(msw, TK_STREAM8); break;
        }
#undef TK_STREAM
#undef TK_STREAM1
#undef TK_STREAM2
#undef TK_STREAM4
#undef TK_STREAM8
        if (r.timed) timing_end(r.timed, s, "fte_stream", ev0);
    } else if (!r.big) {
        hipLaunchKernelGGL(fte_final_kernel, dim3(1), dim3(FINAL_BS), 0, s, r.st, cs, k, a.kreq, fo, r.gate);
    }
    return cs;
}

// The select of a run with an n-entry candidate buffer (FteRun::big).
static void final_enqueue(topk_ctx *ctx, Lane &L, const CandSet &cs, uint32_t k, uint32_t kreq, const FinalOut &fo) {
    hipStream_t s = L.stream;
    hipLaunchKernelGGL(cand_offsets_kernel, dim3(1), dim3(FLAT_BS), 0, s, L.st, cs, ctx->offsets, ctx->flat);
    if (cs.nblk)
        hipLaunchKernelGGL(cand_compact_kernel, dim3(cs.nblk), dim3(256), 0, s, cs, ctx->offsets, ctx->flat);
    hipLaunchKernelGGL(fte_final_flat_kernel, dim3(1), dim3(FLAT_BS), 0, s, L.st, ctx->flat, k, kreq, fo);
}

int fte_enqueue(topk_ctx *ctx, Lane &L, uint32_t k, const QCols &q, const FinalOut &fo, int mode, uint64_t n) {
    if (!n) n = ctx->n;
    if (n >= ID_LIMIT) return TOPK_ERR_UNSUPPORTED;  // a run's ids are 32-bit: callers split larger stores
    FteRun r{};
    r.s = L.stream;
    r.n = n;
    r.st = L.st;
    r.blk = L.blk;
    r.pre = L.pre;
    r.counts = L.counts;
    r.big = mode == FTE_EXACT_BIG;
    r.cand = r.big ? ctx->cand_big : L.cand;
    r.cand_cap = ctx->cand_cap;
    r.spill = L.spill;
    r.spill_cap = ctx->spill_cap;
    r.vpt = ctx->tune.stream_vpt;
    r.grid_cap = ctx->tune.stream_grid;
    r.polls = ctx->tune.sample_polls;
    r.timed = ctx;
    const uint32_t kreq = (uint32_t)(n < k ? n : k);
    const CandSet cs = fte_launch(r, k, q, fo, mode);
    if (r.big) final_enqueue(ctx, L, cs, k, kreq, fo);
    TK_HIP(hipGetLastError());
    return TOPK_OK;
}

// ---------------------------------------------------------------------------
// id shards: top k of the union of per-shard top-k lists
// ---------------------------------------------------------------------------
// Entry j of shard s's list (best first) lands at output position j plus,
// for every other shard, the number of its entries that rank above it -- a
// binary search, since each list is sorted.  Ranking is by score (monotone
// key) and then global id; shard t < s holds only lower ids, so on equal
// scores shard t's entries rank above shard s's.  Positions past k are
// dropped; the k-th entry's score is the threshold.
constexpr int MERGE_BS = 1024;
struct ShardCounts {
    uint32_t shards;
    uint32_t cnt[MAX_ID_SHARDS];  // entries of each shard's list: min(k, objects of the shard)
};

__global__ __launch_bounds__(MERGE_BS) void shard_merge_kernel(const uint64_t *__restrict__ sh_ids,
                                                               const float *__restrict__ sh_scores, ShardCounts c,
                                                               uint32_t k, uint32_t kreq, FinalOut fo) {
    const uint32_t S = c.shards;
    for (uint32_t e = threadIdx.x; e < S * k; e += MERGE_BS) {
        const uint32_t s = e / k, j = e % k;
        if (j >= c.cnt[s]) continue;
        const float sc = sh_scores[(uint64_t)s * TOPK_MAX_K + j];
        const uint32_t ok = okey(sc);
        uint32_t r = j;
        for (uint32_t t = 0; t < S && r < k; t++) {
            if (t == s) continue;
            const float *ts = sh_scores + (uint64_t)t * TOPK_MAX_K;
            uint32_t lo = 0, hi = c.cnt[t];  // entries [0, lo) rank above, [hi, cnt) below
            while (lo < hi) {
                const uint32_t mid = (lo + hi) / 2;
                const uint32_t om = okey(ts[mid]);
                if (om > ok || (om == ok && t < s)) lo = mid + 1;
                else hi = mid;
            }
            r += lo;
        }
        if (r < k) {  // positions are distinct: global ids are
            fo.ids[r] = (uint64_t)s * ID_SHARD + sh_ids[(uint64_t)s * TOPK_MAX_K + j];
            fo.scores[r] = sc;
            if (r == kreq - 1 && fo.thr) *fo.thr = sc;
        }
    }
    for (uint32_t i = kreq + threadIdx.x; i < k; i += MERGE_BS) {
        fo.ids[i] = ~0ull;
        fo.scores[i] = -INFINITY;
    }
    if (threadIdx.x == 0 && fo.status) *fo.status = 0;
}

void shard_merge_enqueue(hipStream_t s, const uint64_t *sh_ids, const float *sh_scores, uint64_t n, uint32_t shards,
                         uint32_t k, const FinalOut &fo) {
    ShardCounts c{};
    c.shards = shards;
    for (uint32_t i = 0; i < shards; i++) {
        const uint64_t ns = n - (uint64_t)i * ID_SHARD < ID_SHARD ? n - (uint64_t)i * ID_SHARD : ID_SHARD;
        c.cnt[i] = (uint32_t)(ns < k ? ns : k);
    }
    const uint32_t kreq = (uint32_t)(n < k ? n : k);
    hipLaunchKernelGGL(shard_merge_kernel, dim3(1), dim3(MERGE_BS), 0, s, sh_ids, sh_scores, c, k, kreq, fo);
}

// ---------------------------------------------------------------------------
// allocation-free FTE over a caller's device store (topk_fte_noalloc)
// ---------------------------------------------------------------------------
// The per-query scratch lives in one file-scope device array per GPU, held
// until the process ends: FTE state, the two passes' status words, seed
// winners, prefix keys, per-block counts, candidate slots and spill region.
// A query is at most two pipeline runs, both enqueued up front: the first
// (sample-seeded above 2^19 objects, exact-prefix-seeded below) and an
// exact-prefix run whose kernels exit at once unless the first reported a
// failure.  Nothing waits on the host, so the call can be captured in a graph.
constexpr uint64_t NA_CAND = 1ull << 20;   // candidate slots (8 MiB)
constexpr uint32_t NA_SPILL = 1u << 18;    // spill region (2 MiB)
constexpr uint64_t NA_BLK = (uint64_t)SAMPLE_CHUNKS * TOPK_MAX_K;  // seed winners, any plan (1 MiB)
struct NoAllocScratch {
    FteState st;
    uint32_t pass[2];  // final-select status of the first and the second run (0: settled)
    uint32_t counts[MAX_STREAM_GRID];
    uint64_t pre[TOPK_MAX_K];
    uint64_t blk[NA_BLK];
    uint64_t cand[NA_CAND];
    uint64_t spill[NA_SPILL];
};
static_assert(offsetof(NoAllocScratch, pre) % 8 == 0 && offsetof(NoAllocScratch, blk) % 8 == 0 &&
                  offsetof(NoAllocScratch, cand) % 8 == 0 && offsetof(NoAllocScratch, spill) % 8 == 0,
              "key arrays stay 8-byte aligned");
constexpr size_t NA_SCRATCH_BYTES = sizeof(NoAllocScratch);

static __device__ __align__(256) unsigned char scratch[NA_SCRATCH_BYTES];

// Device address of `scratch` per GPU (the array's name on the host is only
// a stand-in for the symbol), looked up once per device.
constexpr int NA_MAX_DEVICES = 64;
static std::mutex na_mu;
static NoAllocScratch *na_ptr[NA_MAX_DEVICES];

static int noalloc_scratch(NoAllocScratch **out) {
    int dev = 0;
    TK_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= NA_MAX_DEVICES) return TOPK_ERR_UNSUPPORTED;
    std::lock_guard<std::mutex> lock(na_mu);
    if (!na_ptr[dev]) {
        void *p = nullptr;
        TK_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) return TOPK_ERR_HIP;
        na_ptr[dev] = static_cast<NoAllocScratch *>(p);
    }
    *out = na_ptr[dev];
    return TOPK_OK;
}

// Clears what the pipeline expects at zero (a kernel, not a memset node).
__global__ void noalloc_clear_kernel(NoAllocScratch *__restrict__ sc) {
    static_assert(sizeof(FteState) % 8 == 0, "cleared by words");
    uint64_t *w = reinterpret_cast<uint64_t *>(&sc->st);
    for (uint32_t i = threadIdx.x; i < sizeof(FteState) / 8; i += blockDim.x) w[i] = 0;
    if (threadIdx.x < 2) sc->pass[threadIdx.x] = 0;
}

// Caller-visible status: TOPK_OK when either run settled the query.
__global__ void noalloc_status_kernel(const NoAllocScratch *__restrict__ sc, bool second,
                                      uint32_t *__restrict__ status) {
    if (threadIdx.x != 0) return;
    const uint32_t last = second && sc->pass[0] ? sc->pass[1] : sc->pass[0];
    *status = last == 0 ? (uint32_t)TOPK_OK : (uint32_t)TOPK_ERR_OVERFLOW;
}

}  // namespace topk

using namespace topk;

extern "C" int topk_fte_noalloc(const float *d_cols, uint64_t n, uint32_t d, uint64_t ld, uint32_t k, uint8_t qq,
                                const float *weights, const uint8_t *attr, uint64_t *d_ids, float *d_scores,
                                float *d_threshold, uint32_t *d_status, void *stream) {
    if (!d_cols || !weights || !attr || !d_ids || !d_scores || !d_status) return TOPK_ERR_INVALID;
    if (n < 1 || d < 1 || d > TOPK_MAX_DIMS || ld < n || ld % 4 || k < 1) return TOPK_ERR_INVALID;
    if (reinterpret_cast<uintptr_t>(d_cols) % 16) return TOPK_ERR_INVALID;
    if (n >= 0xFFFFFFFFull || k > TOPK_MAX_K) return TOPK_ERR_UNSUPPORTED;
    if (qq < 1 || qq > d) return TOPK_ERR_INVALID;
    QCols q;
    memset(&q, 0, sizeof(q));
    for (uint32_t j = 0; j < qq; j++) {
        if (attr[j] >= d) return TOPK_ERR_INVALID;
        const float wj = weights[attr[j]];
        if (!std::isfinite(wj)) return TOPK_ERR_INVALID;
        q.col[j] = d_cols + (uint64_t)attr[j] * ld;
        q.w[j] = wj;
    }
    q.m = qq;
    NoAllocScratch *sc = nullptr;
    int rc = noalloc_scratch(&sc);
    if (rc) return rc;

    FteRun r{};
    r.s = static_cast<hipStream_t>(stream);
    r.n = n;
    r.st = &sc->st;
    r.blk = sc->blk;
    r.pre = sc->pre;
    r.counts = sc->counts;
    r.cand = sc->cand;
    r.cand_cap = NA_CAND;
    r.spill = sc->spill;
    r.spill_cap = NA_SPILL;
    hipLaunchKernelGGL(noalloc_clear_kernel, dim3(1), dim3(256), 0, r.s, sc);
    const bool sampled = seed_plan(n, k, FTE_QUEUED).tau != TAU_STATE;
    fte_launch(r, k, q, FinalOut{d_ids, d_scores, d_threshold, &sc->pass[0]}, FTE_QUEUED);
    if (sampled) {
        // too few candidates (the sample guessed high) or a full buffer: the
        // exact-prefix run, skipped on the device when the first one settled
        r.gate = &sc->pass[0];
        fte_launch(r, k, q, FinalOut{d_ids, d_scores, d_threshold, &sc->pass[1]}, FTE_EXACT);
    }
    hipLaunchKernelGGL(noalloc_status_kernel, dim3(1), dim3(64), 0, r.s, sc, sampled, d_status);
    TK_HIP(hipGetLastError());
    return TOPK_OK;
}
