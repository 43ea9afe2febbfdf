// PTA: partitioned threshold top-k on gfx950.
//
// Reference: cpu/PTA.h:88-267 (partition build: polar angles, sorted lists,
// per-block threshold vectors) and cpu/PTA.h:357-422, 569-671 (scan with a
// per-block bound, stop once the heap top beats it).  This file keeps the
// idea -- group similar objects, bound each group, skip groups that cannot
// reach the running k-th score -- with its own partitioning and bound:
//
//  * layout (pta_build.hip): the leaves of a k-d tree, objects ordered by
//    attribute sum inside each; per partition max/min per attribute, the max
//    of its objects' attribute sums and the sum of its minima, and each
//    256-object chunk the same statistics over itself and every later chunk
//    of its partition (suffix rows).
//  * bound: the largest weighted sum any point of the partition's box can
//    reach under the attribute-sum limit (a fractional-knapsack LP, solved
//    greedily in FP64), plus a margin covering binary32 rounding of a score,
//    rounded up to binary32.  It is never below an object's score.
//  * query: bound keys for all partitions; the exact k-th key among the best
//    partitions' objects (seed) is a proven lower bound tau of the global
//    k-th key; the cut pass finds the partitions whose bound reaches tau's
//    score (skip iff bound < tau strictly), each up to its first suffix row
//    whose bound falls below tau, as chunk ranges; the scoring pass spreads
//    those chunks evenly over every wave of the GPU and keeps keys >= tau;
//    its last workgroup selects the exact top k, as the plain stream's does,
//    straight into pinned host memory.  Results equal topk_fte's.
#include <string.h>

#include <algorithm>

#include "bound.hpp"
#include "device.hpp"
#include "internal.hpp"
#include "select.hpp"

namespace topk {

constexpr int PTA_BS = 256;
constexpr uint32_t PTA_SEED_OBJS = 1024;     // leading objects (largest attribute sums) of a seed partition
constexpr uint32_t PTA_MIN_SEED = 16;        // seed partitions at least
constexpr uint32_t PTA_SEED_RANK = 1024;     // keys the seed kernel ranks at most
static_assert(PTA_MAX_PARTS <= PTA_SEED_RANK * PTA_BS, "block maxima of any layout fit the ranking");
constexpr uint32_t PTA_MAX_SEED = 64;
constexpr int PTA_SEED_REG = 16;             // seed winners per thread the merge reads at once
constexpr uint32_t PTA_SEED_LDS = PTA_SEED_REG * PTA_BS;  // seed winners the merge ranks in LDS

// ---------------------------------------------------------------------------
// query kernels
// ---------------------------------------------------------------------------
template <int NB>
__global__ __launch_bounds__(PTA_BS) void pta_bound_kernel(BoundArgs b, uint32_t L,
                                                           const uint32_t *__restrict__ psz,
                                                           const float *__restrict__ pmax,
                                                           const float *__restrict__ pmin,
                                                           const float *__restrict__ psum,
                                                           const float *__restrict__ pminsum,
                                                           uint64_t *__restrict__ pbound, uint64_t *__restrict__ bmax) {
    __shared__ uint64_t wm[PTA_BS / 64];
    const uint32_t p = blockIdx.x * PTA_BS + threadIdx.x;
    uint64_t key = 0;
    if (p < L && psz[p]) {
        const float ub = lp_bound<NB>(b, pmax + (uint64_t)p * b.d, pmin + (uint64_t)p * b.d, psum[p], pminsum[p]);
        key = rkey(ub, p);
    }
    if (p < L) pbound[p] = key;
    const uint64_t m = wave_max_u64(key);
    if (lane_id() == 0) wm[threadIdx.x / 64] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint64_t r = wm[0];
        for (int j = 1; j < PTA_BS / 64; j++) r = wm[j] > r ? wm[j] : r;
        bmax[blockIdx.x] = r;
    }
}

// Seed winners blk[0..cnt) as a key source: KPT loads per thread issued
// together, the same trip count on every thread (ballots inside).
template <int KPT>
struct SeedKeys {
    const uint64_t *p;
    uint32_t cnt;
    template <class F>
    __device__ __forceinline__ void for_each(F f) const {
        uint64_t v[KPT];
#pragma unroll
        for (int j = 0; j < KPT; j++) {
            const uint32_t i = j * PTA_BS + threadIdx.x;
            v[j] = i < cnt ? p[i] : 0ull;
        }
#pragma unroll
        for (int j = 0; j < KPT; j++) f(v[j]);
    }
};

// Key array written with agent-scope (write-through) stores.
struct AgentOut {
    uint64_t *p;
    struct Ref {
        uint64_t *p;
        __device__ __forceinline__ void operator=(uint64_t v) const { store_agent(p, v); }
    };
    __device__ __forceinline__ Ref operator[](uint32_t i) const { return Ref{p + i}; }
};

// Block t scores the leading PTA_SEED_OBJS objects (largest attribute sums)
// of the partition whose bound key is the (t+1)-th largest of bmax[0..nb)
// (the partitions' own bound keys on small layouts, else the maxima of
// blocks of PTA_BS partitions) and keeps its top k; the last block to
// finish takes the k-th largest of all seed keys as tau.
template <int M>
__global__ __launch_bounds__(PTA_BS) void pta_seed_kernel(QCols q, const uint64_t *__restrict__ bmax, uint32_t nb,
                                                          const uint32_t *__restrict__ poff,
                                                          const uint32_t *__restrict__ psz,
                                                          const uint32_t *__restrict__ pid, uint32_t k,
                                                          uint64_t *__restrict__ blk, uint64_t *__restrict__ bthr,
                                                          FteState *__restrict__ st) {
    __shared__ SelectScratch ss;
    __shared__ uint64_t pick;
    __shared__ uint32_t is_last, nvalid;
    __shared__ uint64_t bm[PTA_BS];
    __shared__ uint64_t cands[PTA_SEED_LDS];
    __shared__ uint64_t kth;
    const uint32_t tid = threadIdx.x;
    if (tid == 0) pick = 0;
    // the (t+1)-th largest of the keys (they carry partition ids, so nonzero
    // keys are distinct): up to one a thread, the key with exactly t larger
    // ones; above, where that took 45 us at 1024 keys, a radix select
    if (nb <= PTA_BS) {
        const uint64_t v = tid < nb ? bmax[tid] : 0ull;
        bm[tid] = v;
        __syncthreads();
        uint32_t r = 0, unused = 0;
        rank2_lds(bm, nb, v, v, r, unused);
        if (v && r == blockIdx.x) pick = v;
    } else {
        RegKeys<PTA_SEED_RANK / PTA_BS> bk;
        uint32_t mine = 0;
#pragma unroll
        for (uint32_t j = 0; j < PTA_SEED_RANK / PTA_BS; j++) {
            const uint32_t i = j * PTA_BS + tid;
            bk.k[j] = i < nb ? bmax[i] : 0ull;
            mine += bk.k[j] ? 1u : 0u;
        }
        if (tid == 0) nvalid = 0;
        __syncthreads();
        mine = wave_sum_u32(mine);
        if (lane_id() == 0) atomicAdd(&nvalid, mine);
        __syncthreads();
        const uint32_t valid = nvalid;
        __syncthreads();
        if (blockIdx.x < valid) {  // uniform
            const uint64_t v =
                block_kth_largest<PTA_BS, RegKeys<PTA_SEED_RANK / PTA_BS>, 11>(bk, valid, blockIdx.x + 1, ss);
            if (tid == 0) pick = v;
        }
    }
    __syncthreads();
    const uint64_t pk = pick;
    const uint32_t p = rkey_id(pk);
    const uint32_t start = pk ? poff[p] : 0u;
    const uint32_t size = pk ? (psz[p] < PTA_SEED_OBJS ? psz[p] : PTA_SEED_OBJS) : 0u;
    RegKeys<PTA_SEED_OBJS / PTA_BS> rk;
#pragma unroll
    for (int j = 0; j < (int)(PTA_SEED_OBJS / (4 * PTA_BS)); j++) {
        const uint32_t lo = j * 4 * PTA_BS + tid * 4;
        f4 sc = {0.0f, 0.0f, 0.0f, 0.0f};
        if (lo < size) {
            const uint64_t v = (start + lo) / 4;
            if constexpr (M > 0) {
#pragma unroll
                for (int c = 0; c < M; c++) {
                    f4 pr = ld_stream(q.col[c] + v * 4) * q.w[c];
                    sc = sc + pr;
                }
            } else {
                for (uint32_t c = 0; c < q.m; c++) {
                    f4 pr = ld_stream(q.col[c] + v * 4) * q.w[c];
                    sc = sc + pr;
                }
            }
        }
#pragma unroll
        for (int e = 0; e < 4; e++) rk.k[j * 4 + e] = lo + e < size ? rkey(sc[e], pid[start + lo + e]) : 0ull;
    }
    uint64_t thr = 1;
    if (size > k) thr = block_kth_largest<PTA_BS, RegKeys<PTA_SEED_OBJS / PTA_BS>, 11>(rk, size, k, ss);
    // written through to where the last block reads them: no cache write-back
    const AgentOut out{blk + (uint64_t)blockIdx.x * k};
    const uint32_t got = block_gather_ge<PTA_BS>(rk, thr, out, ss);
    for (uint32_t i = got + tid; i < k; i += PTA_BS) out[i] = 0;
    // this block's k-th key (k keys at or above it), or 0 with fewer than k
    if (tid == 0) store_agent(bthr + blockIdx.x, got >= k ? thr : 0ull);

    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's keys have reached memory
    __syncthreads();
    if (tid == 0)
        is_last = __hip_atomic_fetch_add(&st->arrive, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
    __syncthreads();
    if (!is_last) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    const uint32_t nk = gridDim.x * k;
    if (tid == 0) nvalid = 0;
    __syncthreads();
    uint64_t tau = 1;
    if (nk <= PTA_SEED_LDS) {
        // The union's k-th key is at least the largest block k-th key (that
        // block alone has k keys at or above it): only keys at or above it
        // compete.  They are gathered into LDS and the one with exactly k-1
        // larger keys is the k-th (keys are distinct).
        static_assert(PTA_MAX_SEED <= 64, "a lane per seed block");
        const uint64_t floor_key = wave_max_u64(lane_id() < gridDim.x ? bthr[lane_id()] : 0ull);
        const SeedKeys<PTA_SEED_REG> wk{blk, nk};
        const uint32_t nc = block_gather_ge<PTA_BS>(wk, floor_key ? floor_key : 1ull, cands, ss);
        if (nc > k && nc <= 2 * PTA_BS) {
            // two keys per thread, each ranked against all nc
            const uint64_t x = tid < nc ? cands[tid] : 0ull, y = tid + PTA_BS < nc ? cands[tid + PTA_BS] : 0ull;
            uint32_t rx = 0, ry = 0;
            rank2_lds(cands, nc, x, y, rx, ry);
            if (x && rx == k - 1) kth = x;
            if (y && ry == k - 1) kth = y;
            __syncthreads();
            tau = kth;
        } else if (nc > k) {
            tau = block_kth_largest<PTA_BS, SeedKeys<PTA_SEED_REG>, 11>(SeedKeys<PTA_SEED_REG>{cands, nc}, nc, k, ss);
        } else if (nc == k && floor_key) {
            tau = floor_key;  // exactly the largest block's k keys: its k-th is the union's
        }
    } else {
        uint32_t mine = 0;
        for (uint32_t i = tid; i < nk; i += PTA_BS) mine += blk[i] != 0;
        atomicAdd(&nvalid, mine);
        __syncthreads();
        if (nvalid > k) tau = block_kth_largest<PTA_BS>(MemKeys<PTA_BS>{blk, nk}, nvalid, k, ss);
    }
    if (tid == 0) {
        st->tau = tau;
        st->pre_count = 0;
        st->arrive = 0;
    }
}

// Cut per partition, as the number of its leading objects to score: 0 when
// its bound is below tau's score (skip iff bound < tau strictly), else the
// objects before its first chunk whose suffix-row bound falls below tau
// (every later object of the partition scores below tau too).
//
// A wave takes group g: the R <= 64 partitions g, g + G, g + 2 G, ... (the
// ones that survive are neighbours, so they spread over the waves), a lane
// each for the bounds.  The survivors are then cut four at a time, 16 lanes
// each, one chunk row per lane (a 4096-object partition in one round).  The
// group's cuts, chunk total and report go out without atomics; the scoring
// pass scans the totals.  Bound by the chain of one wave's loads.  One
// workgroup per 16 partitions, most of which did not survive, took 12.2 us on
// average at 65536 partitions (9.2 at the least), this 11.0 (7.1).
template <int NB>
__global__ __launch_bounds__(PTA_BS) void pta_cut_kernel(BoundArgs b, uint32_t L, uint32_t R, uint32_t G,
                                                         const uint64_t *__restrict__ pbound,
                                                         const uint32_t *__restrict__ poff,
                                                         const uint32_t *__restrict__ psz,
                                                         const float *__restrict__ cstat, uint64_t nchunks,
                                                         const FteState *__restrict__ st, uint32_t *__restrict__ cut,
                                                         uint32_t *__restrict__ wchunks, uint2 *__restrict__ wstat) {
    const uint32_t lane = lane_id(), part = lane / 16, gl = lane % 16;
    const uint32_t g = blockIdx.x * (PTA_BS / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    if (g >= G) return;
    const uint32_t tau_hi = (uint32_t)(st->tau >> 32);
    const uint32_t d = b.d;
    const uint32_t p = lane < R ? lane * G + g : L;
    const uint64_t pb = p < L ? pbound[p] : 0ull;  // key 0: an empty partition
    const bool alive = pb != 0 && (uint32_t)(pb >> 32) >= tau_hi;
    const uint32_t psz_ = alive ? psz[p] : 0u, poff_ = alive ? poff[p] : 0u;
    if (lane < R && !alive) cut[g * R + lane] = 0;
    const uint64_t mask = __ballot(alive);
    const uint32_t na = (uint32_t)__popcll(mask);
    // lane i: the owner of the i-th survivor (the other lanes push past them)
    const uint32_t below = (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
    const uint32_t owner = (uint32_t)__builtin_amdgcn_ds_permute((int)(4u * (alive ? below : na + lane - below)), (int)lane);
    uint32_t ch = 0, parts = 0, objs = 0;  // this lane's partitions (lanes gl == 0)
    for (uint32_t i0 = 0; i0 < na; i0 += 4) {
        const bool on = i0 + part < na;
        const uint32_t src = (uint32_t)__shfl((int)owner, (int)((i0 + part) & 63u), 64);
        const uint32_t szs = (uint32_t)__shfl((int)psz_, (int)src, 64), offs = (uint32_t)__shfl((int)poff_, (int)src, 64);
        const uint32_t sz = on ? szs : 0u;
        const uint32_t c0 = offs / PTA_CHUNK;
        const uint32_t nc = (sz + PTA_CHUNK - 1) / PTA_CHUNK;
        uint32_t first = nc;  // this partition's answer, settled once `done`
        bool done = !on;
        for (uint32_t cb = 0; __ballot(!done); cb += 16) {
            const uint32_t c = cb + gl;
            bool fail = false;
            if (!done && c < nc) {
                const float *row = cstat + (c0 + c);  // element e at row[e * nchunks]
                fail = okey(lp_bound<NB>(b, row, row + d * nchunks, row[2 * d * nchunks],
                                         row[(2 * d + 1) * nchunks], nchunks)) < tau_hi;
            }
            const uint32_t m = (uint32_t)(__ballot(fail) >> (16 * part)) & 0xFFFFu;
            if (!done) {
                if (m) {
                    first = cb + (uint32_t)__builtin_ctz(m);
                    done = true;
                } else if (cb + 16 >= nc) {
                    done = true;
                }
            }
        }
        // objects to score: the chunks before the cut, the last one partial
        const uint32_t o = min(sz, first * PTA_CHUNK);
        if (gl == 0 && on) {
            cut[g * R + src] = o;
            ch += (o + PTA_CHUNK - 1) / PTA_CHUNK;
            parts += o ? 1u : 0u;
            objs += o;
        }
    }
    ch = wave_sum_u32(ch);
    parts = wave_sum_u32(parts);
    objs = wave_sum_u32(objs);
    if (lane == 0) {
        wchunks[g] = ch;
        wstat[g] = make_uint2(parts, objs);
    }
}

// Scores the chunks of the partitions the cut pass kept.  Every workgroup
// first scans the G groups' chunk totals into LDS (E[g]: chunks before group
// g).  The waves split the chunks into equal contiguous ranges; a wave finds
// its group by a binary search of E, holds the group's cuts (lane j:
// partition g + j * G) and their chunk prefix in registers, and walks on,
// one chunk per step: 4 objects per lane, the queried columns loaded
// together.  Keys >= tau go to the workgroup's own slot region of the
// candidate buffer (an LDS counter; past the slot, the shared spill region),
// its count to cs.counts[workgroup]; the last workgroup selects, as the
// plain stream's does.  One workgroup of 16 waves per CU keeps the arrivals
// few and gives the select its threads: 22.6 us on average at N = 2^28 (17.5 at
// the least), select included; with four of 4 waves scoring alone took 15.1
// (12.7), and a select launch followed.
// Workgroup 0 also reports the partitions and objects scored.
struct ScoreSelect {
    uint32_t cap, kp2, k, kreq;
    FinalOut fo;
};
template <int M>
__global__ __launch_bounds__(STREAM_BS) void pta_score_kernel(QCols q, uint32_t L, uint32_t R, uint32_t G,
                                                              const uint32_t *__restrict__ cut,
                                                              const uint32_t *__restrict__ wchunks,
                                                              const uint2 *__restrict__ wstat,
                                                              const uint32_t *__restrict__ poff,
                                                              const uint32_t *__restrict__ pid,
                                                              FteState *__restrict__ st, CandSet cs,
                                                              uint32_t *__restrict__ report, ScoreSelect a) {
    extern __shared__ uint64_t dyn[];  // cap keys | workgroup offsets, later cap keys
    constexpr uint32_t GPT = PTA_CUT_GROUPS / STREAM_BS;
    __shared__ union {
        uint32_t E[PTA_CUT_GROUPS + 1];
        FuseScratch sel;
    } sh;
    uint32_t *E = sh.E;
    __shared__ uint32_t wtot[STREAM_NW];
    __shared__ uint32_t wrep[STREAM_NW][2];
    __shared__ uint32_t lcount, is_last;
    // the wave index made visibly uniform: the chunk cursor and its loads
    // (group offsets, cuts, partition offsets) are then scalar
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(tid / 64);
    // exclusive scan of the group totals, GPT consecutive groups a thread
    {
        uint32_t v[GPT], sum = 0, pp = 0, oo = 0;
#pragma unroll
        for (uint32_t j = 0; j < GPT; j++) {
            const uint32_t gi = tid * GPT + j;
            v[j] = gi < G ? wchunks[gi] : 0u;
            sum += v[j];
        }
        if (blockIdx.x == 0) {
            // partitions and objects scored, for the report (fit 32 bits: positions do)
#pragma unroll
            for (uint32_t j = 0; j < GPT; j++) {
                const uint32_t gi = tid * GPT + j;
                const uint2 w = gi < G ? wstat[gi] : make_uint2(0u, 0u);
                pp += w.x;
                oo += w.y;
            }
            pp = wave_sum_u32(pp);
            oo = wave_sum_u32(oo);
            if (lane == 0) {
                wrep[wave][0] = pp;
                wrep[wave][1] = oo;
            }
        }
        const uint32_t incl = wave_incl_scan(sum);
        if (lane == 63) wtot[wave] = incl;
        if (tid == 0) lcount = 0;
        __syncthreads();
        uint32_t run = incl - sum, all = 0;
#pragma unroll
        for (uint32_t w = 0; w < STREAM_NW; w++) {
            run += w < wave ? wtot[w] : 0u;
            all += wtot[w];
        }
#pragma unroll
        for (uint32_t j = 0; j < GPT; j++) {
            const uint32_t gi = tid * GPT + j;
            if (gi < G) E[gi] = run;
            run += v[j];
        }
        if (tid == 0) E[G] = all;  // the total
        if (blockIdx.x == 0 && tid == 0) {
            uint32_t parts = 0, o = 0;
            for (uint32_t w = 0; w < STREAM_NW; w++) {
                parts += wrep[w][0];
                o += wrep[w][1];
            }
            report[1] = parts;
            report[2] = o;
            report[3] = 0;
        }
        __syncthreads();
    }
    const uint32_t total = E[G];
    const uint32_t nw = gridDim.x * STREAM_NW, gw = blockIdx.x * STREAM_NW + wave;
    const uint64_t tau = st->tau;
    const uint32_t tau_hi = (uint32_t)(tau >> 32);
    const uint32_t per = (total + nw - 1) / nw;
    uint32_t c = gw * per;
    const uint32_t c_end = c + per < total ? c + per : total;
    uint64_t *my = cs.keys + (uint64_t)blockIdx.x * cs.slot;
    if (c < c_end) {
        // group of chunk c: the last g with E[g] <= c (E non-decreasing, E[0] = 0)
        uint32_t lo = 0, hi = G;
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) / 2;
            if (E[mid] <= c) lo = mid;
            else hi = mid;
        }
        uint32_t grp = lo;
        uint32_t gbase = 0, lch = 0, lincl = 0;  // lane j: chunks of partition grp + j * G, inclusive prefix
        uint32_t lobj = 0, loff = 0;             // its objects to score and first position
        auto load_group = [&]() {
            gbase = E[grp];
            lobj = lane < R ? cut[grp * R + lane] : 0u;
            loff = lobj ? poff[lane * G + grp] : 0u;
            const uint32_t o = lobj;
            lch = (o + PTA_CHUNK - 1) / PTA_CHUNK;
            lincl = wave_incl_scan(lch);
        };
        load_group();
        for (; c < c_end; c++) {
            while (c >= E[grp + 1]) {
                grp++;
                if (c < E[grp + 1]) load_group();
            }
            // partition: the first lane whose inclusive prefix passes c
            const uint64_t pm = __ballot(gbase + lincl > c);
            const uint32_t j = (uint32_t)__builtin_ctzll(pm);
            const uint32_t pincl = (uint32_t)__shfl(lincl, (int)j, 64), pch = (uint32_t)__shfl(lch, (int)j, 64);
            const uint32_t lc = c - (gbase + pincl - pch);
            const uint32_t objs_p = (uint32_t)__shfl((int)lobj, (int)j, 64);
            const uint32_t first = lc * PTA_CHUNK + 4 * lane;
            const uint64_t pos = (uint64_t)(uint32_t)__shfl((int)loff, (int)j, 64) + first;
            f4 sc = {0.0f, 0.0f, 0.0f, 0.0f};
            if constexpr (M > 0) {
                f4 x[M];
#pragma unroll
                for (int jj = 0; jj < M; jj++) x[jj] = ld_stream(q.col[jj] + pos);
#pragma unroll
                for (int jj = 0; jj < M; jj++) {
                    f4 pr = x[jj] * q.w[jj];
                    sc = sc + pr;
                }
            } else {
                for (uint32_t jj = 0; jj < q.m; jj++) {
                    f4 pr = ld_stream(q.col[jj] + pos) * q.w[jj];
                    sc = sc + pr;
                }
            }
            const uint32_t nvalid = first < objs_p ? (objs_p - first < 4u ? objs_p - first : 4u) : 0u;
            uint64_t kk[4];
            uint32_t npass = 0;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t ok = okey(sc[e]);
                uint64_t key = 0;
                if ((uint32_t)e < nvalid && ok >= tau_hi) {
                    key = rkey_from_okey(ok, pid[pos + e]);
                    if (key < tau) key = 0;
                }
                kk[e] = key;
                npass += key ? 1u : 0u;
            }
            if (__ballot(npass != 0)) {
                const uint32_t incl = wave_incl_scan(npass);
                const uint32_t wt = __shfl(incl, 63, 64);
                uint32_t cnt = 0;
                if (lane == 63) cnt = atomicAdd(&lcount, wt);
                cnt = __shfl(cnt, 63, 64);
                const uint32_t first_spill = cnt > cs.slot ? cnt : cs.slot;
                const uint32_t nspill = cnt + wt > first_spill ? cnt + wt - first_spill : 0u;
                uint32_t sbase = 0;
                if (nspill) {
                    if (lane == 63) sbase = atomicAdd(&st->spill, nspill);
                    sbase = __shfl(sbase, 63, 64);
                }
                uint32_t pos_k = cnt + incl - npass;
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (kk[e]) {
                        if (pos_k < cs.slot) {
                            store_agent(my + pos_k, kk[e]);
                        } else {
                            const uint32_t sp = sbase + (pos_k - first_spill);
                            if (sp < cs.spill_cap) store_agent(cs.spill + sp, kk[e]);
                        }
                        pos_k++;
                    }
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's candidates have reached memory
    __syncthreads();
    if (tid == 0) {
        __hip_atomic_store(&cs.counts[blockIdx.x], lcount < cs.slot ? lcount : cs.slot, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        is_last = last_to_arrive(st);
    }
    __syncthreads();
    if (!is_last) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    fused_select<STREAM_BS>(st, cs, a.k, a.kreq, a.cap, a.kp2, a.fo, dyn, dyn + a.cap, sh.sel);
}

// ---------------------------------------------------------------------------
// host: query
// ---------------------------------------------------------------------------
// Four launches on the context's stream: bound, seed, cut, and scoring, whose
// last workgroup selects; fo points at pinned host memory, so the caller only
// synchronises.
int pta_query(topk_ctx *ctx, uint32_t k, uint8_t qq, const float *weights, const uint8_t *attr, const FinalOut &fo) {
    PtaLayout &P = ctx->pta;
    if (!P.built) return TOPK_ERR_STATE;
    QCols q;
    int rc = build_qcols(ctx, P.pcols, P.ld, qq, weights, attr, q);
    if (rc) return rc;
    const BoundArgs b = make_bound_args(ctx->d, qq, weights, attr);

    Lane &Ln = ctx->lane[0];
    hipStream_t s = Ln.stream;
    const uint32_t L = P.nparts;
    const uint32_t nb = (L + PTA_BS - 1) / PTA_BS;
    const int NB = ctx->d <= 8 ? 8 : (ctx->d <= 16 ? 16 : TOPK_MAX_DIMS);
    auto bound = NB == 8 ? pta_bound_kernel<8> : (NB == 16 ? pta_bound_kernel<16> : pta_bound_kernel<TOPK_MAX_DIMS>);
    hipLaunchKernelGGL(bound, dim3(nb), dim3(PTA_BS), 0, s, b, L, P.psz, P.pmax, P.pmin, P.psum, P.pminsum, P.pbound,
                       P.bmax);
    // seed partitions are ranked by their own bounds when there are few of
    // them (so a small layout still seeds from several partitions), else by
    // the block maxima
    const bool own = L <= PTA_SEED_RANK;
    const uint64_t *rkeys = own ? P.pbound : P.bmax;
    const uint32_t nr = own ? L : nb;
    uint32_t T = (4 * k + PTA_SEED_OBJS - 1) / PTA_SEED_OBJS;
    if (T < PTA_MIN_SEED) T = PTA_MIN_SEED;
    if (T > PTA_MAX_SEED) T = PTA_MAX_SEED;
    if (T > nr) T = nr;
#define TK_SEED(MM)                                                                                              \
    hipLaunchKernelGGL(pta_seed_kernel<MM>, dim3(T), dim3(PTA_BS), 0, s, q, rkeys, nr, P.poff, P.psz, P.pid, k, \
                       Ln.blk, Ln.pre, Ln.st)
    TK_SWITCH_M(q.m, TK_SEED);
#undef TK_SEED
    hipEvent_t ev0 = nullptr;
    timing_begin(ctx, s, ev0);
    // cut pass: R partitions a wave, four (one round) on small layouts, at
    // most 64 (a lane each) and PTA_CUT_GROUPS waves
    const uint32_t R = std::min(64u, std::max(4u, (L + 1023) / 1024));
    const uint32_t G = (L + R - 1) / R;
    if (G > PTA_CUT_GROUPS) return TOPK_ERR_UNSUPPORTED;
    auto cutk = NB == 8 ? pta_cut_kernel<8> : (NB == 16 ? pta_cut_kernel<16> : pta_cut_kernel<TOPK_MAX_DIMS>);
    hipLaunchKernelGGL(cutk, dim3((G + PTA_BS / 64 - 1) / (PTA_BS / 64)), dim3(PTA_BS), 0, s, b, L, R, G, P.pbound,
                       P.poff, P.psz, P.cstat, (uint64_t)P.nchunks, Ln.st, P.pcut, P.wchunks, P.wstat);
    // scoring and select: one 16-wave workgroup per CU, one slot region each
    const uint32_t sg = std::min((uint32_t)P.cus, MAX_STREAM_GRID);
    CandSet cs;
    cs.keys = Ln.cand;
    cs.counts = Ln.counts;
    cs.nblk = sg;
    cs.slot = (uint32_t)(ctx->cand_cap / cs.nblk);
    cs.pre = nullptr;
    cs.spill = Ln.spill;
    cs.spill_cap = ctx->spill_cap;
    ScoreSelect sel{};
    sel.k = k;
    sel.kreq = (uint32_t)(ctx->n < k ? ctx->n : k);
    sel.kp2 = next_pow2(k);
    sel.cap = std::min(FUSE_CAP_MAX, std::max(FUSE_CAP_MIN, 4 * sel.kp2));
    sel.fo = fo;
    sel.fo.cand = P.h_report;  // report[0]
    const size_t lds = sizeof(uint64_t) * ((size_t)sel.cap + std::max((sg + 3) / 2, sel.cap));
#define TK_SCORE(MM)                                                                                                \
    hipLaunchKernelGGL(pta_score_kernel<MM>, dim3(sg), dim3(STREAM_BS), lds, s, q, L, R, G, P.pcut, P.wchunks, P.wstat, \
                       P.poff, P.pid, Ln.st, cs, P.h_report, sel)
    TK_SWITCH_M(q.m, TK_SCORE);
#undef TK_SCORE
    timing_end(ctx, s, "pta_stream", ev0);
    TK_HIP(hipGetLastError());
    return TOPK_OK;
}

}  // namespace topk
