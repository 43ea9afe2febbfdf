// Wave64 and workgroup primitives for gfx950: scans and reductions, an exact
// workgroup radix select over 64-bit ranking keys, key gathering and a rank
// sort in LDS.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "keys.hpp"

namespace topk {

typedef float f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t lane_id() { return __lane_id(); }

// Wave-wide scans and reductions by DPP: four row shifts inside the 16-lane
// rows, then two row broadcasts across them (about 60 cycles; the same steps
// as LDS permutes take about 130 cycles each).  All 64 lanes take part.
// Lane l's value of the next step; zero where the pattern has no source.
#define TK_DPP(v, ctrl, rows) ((uint32_t)__builtin_amdgcn_update_dpp(0, (int)(v), ctrl, rows, 0xF, false))
#define TK_DPP_STEPS(STEP)                                                    \
    STEP(0x111, 0xF) /* row_shr 1 */ STEP(0x112, 0xF) /* row_shr 2 */         \
    STEP(0x114, 0xF) /* row_shr 4 */ STEP(0x118, 0xF) /* row_shr 8 */         \
    STEP(0x142, 0xA) /* row_bcast 15 into rows 1, 3 */                        \
    STEP(0x143, 0xC) /* row_bcast 31 into rows 2, 3 */

// Orders a wave's own LDS accesses: what its lanes wrote before is what any of
// them reads after (no instruction beyond the waits the compiler inserts).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Inclusive prefix sum across the 64 lanes of a wave.
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v) {
#define TK_STEP(ctrl, rows) v += TK_DPP(v, ctrl, rows);
    TK_DPP_STEPS(TK_STEP)
#undef TK_STEP
    return v;
}

__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
#define TK_STEP(ctrl, rows)                       \
    {                                             \
        const uint32_t t = TK_DPP(v, ctrl, rows); \
        v = t > v ? t : v;                        \
    }
    TK_DPP_STEPS(TK_STEP)
#undef TK_STEP
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// The high halves' maximum, then the largest low half among its holders.
__device__ __forceinline__ uint64_t wave_max_u64(uint64_t v) {
    const uint32_t hi = wave_max_u32((uint32_t)(v >> 32));
    const uint32_t lo = wave_max_u32((uint32_t)(v >> 32) == hi ? (uint32_t)v : 0u);
    return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ uint64_t wave_min_u64(uint64_t v) { return ~wave_max_u64(~v); }

__device__ __forceinline__ uint32_t wave_sum_u32(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_readlane((int)wave_incl_scan(v), 63);
}

// The last index i in [lo, hi) with key(i) <= t (key non-decreasing, key(lo)
// <= t), found by the wave: 64 probes per round narrow the range 64-fold.
template <class Key>
__device__ __forceinline__ uint32_t wave_last_le(Key key, uint32_t lo, uint32_t hi, uint32_t t) {
    const uint32_t lane = lane_id();
    while (hi - lo > 1) {
        const uint32_t step = (hi - lo + 63) / 64;
        const uint32_t i = lo + lane * step;
        const bool le = i < hi && key(i) <= t;
        const uint64_t m = __ballot(le);  // lanes 0..j (keys are non-decreasing)
        const uint32_t j = 63u - (uint32_t)__builtin_clzll(m);
        lo = lo + j * step;
        hi = lo + step < hi ? lo + step : hi;
    }
    return lo;
}

// Removes the largest of the ranking keys the wave's lanes hold (NPL per
// lane, score half in hi, id half in lo; hi = 0: none) and returns it on
// every lane; 0 once none is left.  Keys are distinct.
template <int NPL>
__device__ __forceinline__ uint64_t wave_pop_max(uint32_t (&hi)[NPL], const uint32_t (&lo)[NPL]) {
    uint32_t m = 0;
#pragma unroll
    for (int j = 0; j < NPL; j++) m = hi[j] > m ? hi[j] : m;
    const uint32_t M = wave_max_u32(m);
    if (M == 0) return 0;
    uint32_t l = 0;
#pragma unroll
    for (int j = 0; j < NPL; j++) l = hi[j] == M && lo[j] > l ? lo[j] : l;
    uint64_t b = __ballot(m == M);
    if (b & (b - 1)) {  // several lanes hold the score: the largest id half
        const uint32_t L = wave_max_u32(m == M ? l : 0u);
        b = __ballot(m == M && l == L);
    }
    const uint32_t leader = (uint32_t)__builtin_ctzll(b);
    const uint32_t L = (uint32_t)__builtin_amdgcn_readlane((int)l, (int)leader);
#pragma unroll
    for (int j = 0; j < NPL; j++) hi[j] = hi[j] == M && lo[j] == L && lane_id() == leader ? 0u : hi[j];
    return ((uint64_t)M << 32) | L;
}

// Streaming 128-bit load that bypasses cache residency (data read once).
__device__ __forceinline__ f4 ld_stream(const float *p) {
    return __builtin_nontemporal_load(reinterpret_cast<const f4 *>(p));
}

// LDS scratch of the workgroup selection: a histogram of BINS digits, one
// word of padding per lane's bins so that the lanes of the scan, BINS / 64
// bins apart, read different banks; also the last 64 keys of a selection.
template <int BINS>
struct SelectScratchT {
    alignas(8) uint32_t hist[BINS + 64];
    uint32_t digit, need, bcnt, counter;
    unsigned long long kmin, kmax;
};
using SelectScratch = SelectScratchT<2048>;  // up to 11-bit digits

// How many of the n keys a[0..n) (LDS, every lane reading the same word)
// are above x and above y: eight reads in flight per step, so the loop
// runs at LDS throughput rather than latency.
__device__ __forceinline__ void rank2_lds(const uint64_t *a, uint32_t n, uint64_t x, uint64_t y, uint32_t &rx,
                                          uint32_t &ry) {
    uint32_t j = 0;
    for (; j + 8 <= n; j += 8) {
        uint64_t v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = a[j + u];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            rx += v[u] > x ? 1u : 0u;
            ry += v[u] > y ? 1u : 0u;
        }
    }
    for (; j < n; j++) {
        const uint64_t v = a[j];
        rx += v > x ? 1u : 0u;
        ry += v > y ? 1u : 0u;
    }
}

// Key sources: the keys a thread owns, visited by for_each.  Key 0 marks an
// empty slot and is never selected.
template <int KPT>
struct RegKeys {
    uint64_t k[KPT];
    template <class F>
    __device__ __forceinline__ void for_each(F f) const {
#pragma unroll
        for (int i = 0; i < KPT; i++) f(k[i]);
    }
};

template <int BS>
struct MemKeys {
    const uint64_t *p;
    uint32_t cnt;
    template <class F>
    __device__ __forceinline__ void for_each(F f) const {
        uint32_t i = threadIdx.x;
        for (; i + 7 * BS < cnt; i += 8 * BS) {  // 8 independent loads in flight
            uint64_t v[8];
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = p[i + j * BS];
#pragma unroll
            for (int j = 0; j < 8; j++) f(v[j]);
        }
        for (; i < cnt; i += BS) f(p[i]);
    }
};

// Block-wide min / max of u64 (all threads call; result on every thread).
template <int BS, class Scratch>
__device__ __forceinline__ void block_minmax(uint64_t &lo, uint64_t &hi, Scratch &s) {
    lo = wave_min_u64(lo);
    hi = wave_max_u64(hi);
    if (BS == 64) return;
    if (threadIdx.x == 0) { s.kmin = ~0ull; s.kmax = 0; }
    __syncthreads();
    if (lane_id() == 0) {
        atomicMin(&s.kmin, (unsigned long long)lo);
        atomicMax(&s.kmax, (unsigned long long)hi);
    }
    __syncthreads();
    lo = s.kmin;
    hi = s.kmax;
    __syncthreads();
}

// Exact k-th largest non-zero key of the block's key source, where setcnt
// (>= k >= 1) is the number of non-zero keys.  Every thread of the block
// (BS = blockDim.x, a multiple of 64) must call it and gets the result.
//
// MSD radix select that never spends a pass on bits all remaining
// candidates share: each round takes the min / max of the candidate set,
// starts its 8-bit digit just below their common prefix, builds the digit
// histogram in LDS, and one wave finds the digit holding the k-th key with
// a lane prefix scan.  Rounds stop when the candidate set is one value, when
// the k-th is its maximum, or when the whole set is inside the top k (then
// the k-th is its minimum), or when at most 64 candidates are left: these are
// ranked against each other in one wave (0.7 us; a round costs 2.5 us, and
// ids below equal or close scores took two or three more).  Inlined always: as
// a call its keys and scratch are reached by flat addresses, and the exact
// seed's merge of 17500 keys took 4 us more (67.6, 64.0).
template <int BS, class Src, int DB = 8, class Scratch = SelectScratch>
__device__ __forceinline__ uint64_t block_kth_largest(const Src &src, uint32_t setcnt, uint32_t k, Scratch &s) {
    static_assert(DB >= 6 && DB <= 11, "digit width");
    static_assert(sizeof(s.hist) >= sizeof(uint32_t) * ((1u << DB) + 64), "one bin per digit, padded");
    constexpr uint32_t NB = 1u << DB, PER = NB / 64;
    auto bin = [](uint32_t b) { return b + b / PER; };
    const uint32_t tid = threadIdx.x;
    uint64_t prefix = 0, mask = 0;
    uint32_t need = k;
    for (;;) {
        if (setcnt <= 64) {
            uint64_t *last = reinterpret_cast<uint64_t *>(s.hist);
            if (tid == 0) s.counter = 0;
            __syncthreads();
            src.for_each([&](uint64_t key) {
                if (key && (key & mask) == prefix) {
                    const uint32_t i = atomicAdd(&s.counter, 1u);
                    if (i < 64) last[i] = key;
                }
            });
            __syncthreads();
            const uint32_t n = s.counter < 64 ? s.counter : 64u;
            if (tid < n) {
                // the key with fewer than `need` larger ones and at least
                // `need` no smaller (equal keys write the same value)
                const uint64_t x = last[tid];
                uint32_t above = 0, from = 0;
                rank2_lds(last, n, x, x - 1, above, from);
                if (above < need && need <= from) s.kmax = x;
            }
            __syncthreads();
            const uint64_t kth = s.kmax;
            __syncthreads();
            return kth;
        }
        uint64_t lo = ~0ull, hi = 0;
        src.for_each([&](uint64_t key) {
            if (key && (key & mask) == prefix) {
                lo = key < lo ? key : lo;
                hi = key > hi ? key : hi;
            }
        });
        block_minmax<BS>(lo, hi, s);
        if (need == setcnt) return lo;
        if (need == 1 || lo == hi) return hi;
        const int db = 63 - __clzll(lo ^ hi);          // highest differing bit
        const uint64_t above = db == 63 ? 0ull : (~0ull << (db + 1));
        prefix = hi & above;
        mask = above;
        const int width = db + 1 < DB ? db + 1 : DB;
        const int shift = db + 1 - width;
        const uint32_t dmask = (1u << width) - 1u;
        for (uint32_t i = tid; i < NB + 64; i += BS) s.hist[i] = 0;
        __syncthreads();
        src.for_each([&](uint64_t key) {
            if (key && (key & mask) == prefix) atomicAdd(&s.hist[bin((uint32_t)(key >> shift) & dmask)], 1u);
        });
        __syncthreads();
        if (tid < 64) {
            // lane l owns bins NB-1-PER*l .. NB-PER*(l+1), highest first
            const uint32_t top = NB - 1 - PER * tid;
            uint32_t tot = 0;
            for (uint32_t j = 0; j < PER; j++) tot += s.hist[bin(top - j)];
            const uint32_t incl = wave_incl_scan(tot);
            const uint32_t excl = incl - tot;
            if (excl < need && need <= incl) {
                uint32_t r = need - excl, acc = 0;
                for (uint32_t j = 0; j < PER; j++) {
                    const uint32_t cj = s.hist[bin(top - j)];
                    if (r <= acc + cj) {
                        s.digit = top - j;
                        s.need = r - acc;
                        s.bcnt = cj;
                        break;
                    }
                    acc += cj;
                }
            }
        }
        __syncthreads();
        const uint32_t digit = s.digit;
        need = s.need;
        setcnt = s.bcnt;
        __syncthreads();
        prefix |= (uint64_t)digit << shift;
        mask |= (uint64_t)dmask << shift;
    }
}

// Writes every non-zero key >= thr of the source to out[] (order
// unspecified) with a wave-aggregated LDS counter; returns the count.  All
// threads of the block must call.
template <int BS, class Src, class Out, class Scratch>
__device__ uint32_t block_gather_ge(const Src &src, uint64_t thr, Out out, Scratch &s) {
    if (threadIdx.x == 0) s.counter = 0;
    __syncthreads();
    src.for_each([&](uint64_t key) {
        const bool p = key && key >= thr;
        const uint64_t bal = __ballot(p);
        if (bal) {
            const uint32_t rank = __popcll(bal & ((1ull << lane_id()) - 1ull));
            uint32_t base = 0;
            if (lane_id() == 0) base = atomicAdd(&s.counter, (uint32_t)__popcll(bal));
            base = __shfl(base, 0, 64);
            if (p) out[base + rank] = key;
        }
    });
    __syncthreads();
    const uint32_t r = s.counter;
    __syncthreads();
    return r;
}

// Memory key source for block_gather_ge: every lane of a wave must take
// part in the ballot, so the trip count is uniform across the block.
template <int BS>
struct MemKeysUniform {
    const uint64_t *p;
    uint32_t cnt;
    template <class F>
    __device__ __forceinline__ void for_each(F f) const {
        for (uint32_t i0 = 0; i0 < cnt; i0 += BS) {
            const uint32_t i = i0 + threadIdx.x;
            f(i < cnt ? p[i] : 0ull);
        }
    }
};

// Key source over a flat index space [0, cnt) resolved by a view's get(p);
// Uniform=true keeps the trip count uniform across the block (for ballots).
template <int BS, class View, bool Uniform>
struct ViewKeys {
    View v;
    uint32_t cnt;
    template <class F>
    __device__ __forceinline__ void for_each(F f) const {
        if constexpr (Uniform) {
            for (uint32_t i0 = 0; i0 < cnt; i0 += BS) {
                const uint32_t i = i0 + threadIdx.x;
                f(i < cnt ? v.get(i) : 0ull);
            }
        } else {
            for (uint32_t i = threadIdx.x; i < cnt; i += BS) f(v.get(i));
        }
    }
};

// Block-wide exclusive prefix sum of one value per thread; returns the
// thread's exclusive prefix and writes the block total to *total.
template <int BS>
__device__ uint32_t block_excl_scan(uint32_t v, uint32_t *wave_sums, uint32_t *total) {
    constexpr int NW = BS / 64;
    const uint32_t w = threadIdx.x / 64;
    const uint32_t incl = wave_incl_scan(v);
    if (lane_id() == 63) wave_sums[w] = incl;
    __syncthreads();
    if (threadIdx.x < 64) {
        const uint32_t ws = threadIdx.x < NW ? wave_sums[threadIdx.x] : 0u;
        const uint32_t wi = wave_incl_scan(ws);
        if (threadIdx.x < NW) wave_sums[threadIdx.x] = wi - ws;
        if (threadIdx.x == NW - 1) *total = wi;
    }
    __syncthreads();
    const uint32_t r = wave_sums[w] + incl - v;
    __syncthreads();
    return r;
}

// Sorts the got distinct keys in[0..got) descending into out[] by rank
// counting (one pass, no barrier inside): out[#{j: in[j] > in[i]}] = in[i].
template <int BS>
__device__ void block_rank_sort_desc(const uint64_t *in, uint32_t got, uint64_t *out) {
    for (uint32_t i = threadIdx.x; i < got; i += BS) {
        const uint64_t x = in[i];
        uint32_t r = 0, unused = 0;
        rank2_lds(in, got, x, x, r, unused);
        out[r] = x;
    }
    __syncthreads();
}

// Sorts a[0..n2) descending in LDS (n2 a power of two); all threads call.
template <int BS>
__device__ void bitonic_sort_desc(uint64_t *a, uint32_t n2) {
    for (uint32_t size = 2; size <= n2; size <<= 1) {
        for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
            for (uint32_t t = threadIdx.x; t < n2 / 2; t += BS) {
                uint32_t lo = 2 * stride * (t / stride) + (t & (stride - 1));
                uint32_t hi = lo + stride;
                bool desc = (lo & size) == 0;
                uint64_t x = a[lo], y = a[hi];
                if ((x < y) == desc) { a[lo] = y; a[hi] = x; }
            }
            __syncthreads();
        }
    }
}

__host__ __device__ __forceinline__ uint32_t next_pow2(uint32_t v) {
    uint32_t p = 1;
    while (p < v) p <<= 1;
    return p;
}

}  // namespace topk
