// The final select of a streaming pass, in its last workgroup: arrival
// counting across XCDs, and the exact top k of the candidates the workgroups
// published (fte.hip, pta.hip).
#pragma once
#include "device.hpp"
#include "internal.hpp"

namespace topk {

constexpr int STREAM_NW = STREAM_BS / 64;

__device__ __forceinline__ void store_agent(uint64_t *p, uint64_t v) {
    __hip_atomic_store(reinterpret_cast<unsigned long long *>(p), (unsigned long long)v, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}

// Flat index -> key over pre[0..npre) followed by the blocks' slot regions;
// off[] (LDS) holds the exclusive prefix of the per-block counts.
struct SlotView {
    const uint64_t *pre;
    uint32_t npre;
    const uint64_t *keys;
    uint32_t slot;
    const uint32_t *off;
    uint32_t nblk, total;  // keys in slots; the spill region's follow
    const uint64_t *spill;
    __device__ __forceinline__ uint64_t get(uint32_t p) const {
        if (p < npre) return pre[p];
        const uint32_t q = p - npre;
        if (q >= total) return spill[q - total];
        uint32_t lo = 0, hi = nblk;  // largest b with off[b] <= q
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (off[mid] <= q) lo = mid;
            else hi = mid;
        }
        return keys[(uint64_t)lo * slot + (q - off[lo])];
    }
};

// Called by one thread of each workgroup once its results are in memory:
// true in the last one.  Group g counts workgroups g, g + ARRIVE_GROUPS, ...
__device__ __forceinline__ bool last_to_arrive(FteState *__restrict__ st) {
    const uint32_t G = gridDim.x, g = blockIdx.x % ARRIVE_GROUPS;
    const uint32_t members = (G - g + ARRIVE_GROUPS - 1) / ARRIVE_GROUPS;
    if (__hip_atomic_fetch_add(&st->group[g * ARRIVE_STRIDE], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) !=
        members - 1)
        return false;
    return __hip_atomic_fetch_add(&st->arrive, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
           (G < ARRIVE_GROUPS ? G : ARRIVE_GROUPS) - 1;
}

constexpr uint32_t FUSE_BINS = 1024;
constexpr uint32_t FUSE_BIN_MAX = 128;  // keys of one bin ranked against each other
struct FuseScratch {
    uint32_t bins[FUSE_BINS];
    SelectScratchT<256> rs;
    uint64_t wlo[STREAM_NW], whi[STREAM_NW];
    uint32_t crowded;     // an interval too full to rank by pairs
    uint32_t cut, ncut;   // the interval holding the k-th key, and the keys up to its end
};

// f on every candidate, c of them.  Spread thin over the workgroups' slots they
// are taken by flat index, four at a time; else a workgroup's slots by a wave,
// eight loads in flight, without a search for each.
template <int BS, class F>
__device__ __forceinline__ void for_candidates(const SlotView &v, uint32_t c, F f) {
    const uint32_t tid = threadIdx.x;
    if (c < 64 * v.nblk) {
        for (uint32_t i0 = tid; i0 < c; i0 += 4 * BS) {
            uint64_t x[4];
#pragma unroll
            for (int j = 0; j < 4; j++) x[j] = i0 + j * BS < c ? v.get(i0 + j * BS) : 0ull;
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (x[j]) f(x[j]);
        }
        return;
    }
    auto range = [&](const uint64_t *p, uint32_t n, uint32_t first, uint32_t step) __attribute__((always_inline)) {
        for (uint32_t i0 = first; i0 < n; i0 += 8 * step) {
            uint64_t x[8];
#pragma unroll
            for (int j = 0; j < 8; j++) x[j] = i0 + j * step < n ? p[i0 + j * step] : 0ull;
#pragma unroll
            for (int j = 0; j < 8; j++)
                if (x[j]) f(x[j]);
        }
    };
    range(v.pre, v.npre, tid, BS);
    for (uint32_t b = tid / 64; b < v.nblk; b += BS / 64) {
        const uint32_t at = v.off[b], end = b + 1 < v.nblk ? v.off[b + 1] : v.total;
        range(v.keys + (uint64_t)b * v.slot, end - at, lane_id(), 64);
    }
    range(v.spill, c - v.npre - v.total, tid, BS);
}

// Writes the first want keys, best first, and sentinels up to k.
template <int BS>
__device__ __forceinline__ void emit_sorted(const uint64_t *sorted, uint32_t want, uint32_t k, const FinalOut &fo) {
    for (uint32_t i = threadIdx.x; i < k; i += BS) {
        const uint64_t x = i < want ? sorted[i] : 0ull;
        fo.ids[i] = i < want ? (uint64_t)rkey_id(x) : ~0ull;
        fo.scores[i] = i < want ? rkey_score(x) : -INFINITY;
    }
    if (threadIdx.x == 0 && fo.thr) *fo.thr = rkey_score(sorted[want - 1]);
}

// Exact top k of the candidates the stream's workgroups published, by the
// last of them to finish.  The counts' offsets are scanned, the candidates
// gathered into LDS (lkeys, cap keys), counting-sorted by 1024 equal
// intervals of their key range -- only as far as the interval that holds the
// k-th -- and each key is ranked inside its interval; results go out best
// first.  Of more candidates than cap, the intervals that hold the first want
// of them are gathered (three passes; the radix select of 90000 candidates
// took 500 us and 11 passes, a binary search a key).  Ties crowding one
// interval, or past cap, take a radix select.  lkeys and regb hold cap keys
// each (2 * kp2 at least).
template <int BS>
__device__ __forceinline__ void fused_select(FteState *__restrict__ st, const CandSet &cs, uint32_t k, uint32_t kreq, uint32_t cap,
                             uint32_t kp2, const FinalOut &fo, uint64_t *lkeys, uint64_t *regb, FuseScratch &fs) {
    __shared__ uint32_t wsum[BS / 64];
    __shared__ uint32_t total, s_spill, s_pre;
    uint32_t *off = reinterpret_cast<uint32_t *>(regb);
    const uint32_t tid = threadIdx.x, wave = tid / 64;
    if (cs.nblk <= 256) {
        // wave 0 scans four counts per lane, the other waves clear
        if (wave == 0) {
            uint32_t n_[4], sum = 0;
#pragma unroll
            for (int j = 0; j < 4; j++) n_[j] = 4 * tid + j < cs.nblk ? cs.counts[4 * tid + j] : 0u;
            if (tid == 0) {
                s_spill = st->spill;
                s_pre = cs.pre ? st->pre_count : 0u;
            }
#pragma unroll
            for (int j = 0; j < 4; j++) sum += n_[j];
            uint32_t at = wave_incl_scan(sum) - sum;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if (4 * tid + j < cs.nblk) off[4 * tid + j] = at;
                at += n_[j];
            }
            if (tid == 63) total = at;
        } else {
            for (uint32_t b = tid - 64; b < FUSE_BINS; b += BS - 64) fs.bins[b] = 0;
            if (tid == 64) fs.crowded = 0;
        }
    } else {
        for (uint32_t b = tid; b < cs.nblk; b += BS) off[b] = cs.counts[b];
        for (uint32_t b = tid; b < FUSE_BINS; b += BS) fs.bins[b] = 0;
        if (tid == 0) {
            fs.crowded = 0;
            s_spill = st->spill;
            s_pre = cs.pre ? st->pre_count : 0u;
        }
        __syncthreads();
        const uint32_t per = (cs.nblk + BS - 1) / BS;
        const uint32_t b0 = tid * per < cs.nblk ? tid * per : cs.nblk;
        const uint32_t b1 = b0 + per < cs.nblk ? b0 + per : cs.nblk;
        uint32_t mine = 0;
        for (uint32_t b = b0; b < b1; b++) mine += off[b];
        uint32_t run = block_excl_scan<BS>(mine, wsum, &total);
        for (uint32_t b = b0; b < b1; b++) {
            const uint32_t c = off[b];
            off[b] = run;
            run += c;
        }
    }
    __syncthreads();
    const uint32_t spilled = s_spill, npre = s_pre;
    const uint32_t nspill = spilled < cs.spill_cap ? spilled : cs.spill_cap;
    const uint32_t ntotal = total, c = npre + ntotal + nspill;
    const uint32_t bad = spilled > cs.spill_cap ? STATUS_OVERFLOW : (c < kreq ? STATUS_RETRY : 0u);
    if (tid == 0) {
        // ready for the next query
        st->spill = 0;
        st->arrive = 0;
        st->ticket = 0;
        if (bad) st->status |= bad;
        else st->cand_last = c;
        if (!bad && fo.cand) *fo.cand = c;
        if (fo.status) *fo.status = bad;
    }
    if (tid < ARRIVE_GROUPS) st->group[tid * ARRIVE_STRIDE] = 0;
    static_assert(SAMPLE_WIN <= BS, "a winner a thread");
    if (tid < SAMPLE_WIN) st->win[tid] = 0;
    if (bad) return;
    const SlotView v{cs.pre, npre, cs.keys, cs.slot, off, cs.nblk, ntotal, cs.spill};
    const uint32_t want = c < k ? c : k;  // results
    uint64_t *sorted;
    if (c <= BS / 4) {
        // few: each key's rank counted by four threads, a quarter of the keys each
        const uint32_t i = tid % (BS / 4), part = tid / (BS / 4), q4 = (c + 3) / 4;
        uint64_t x = 0;
        if (part == 0 && i < c) lkeys[i] = x = v.get(i);
        if (part == 1) fs.bins[i] = 0;  // the ranks
        __syncthreads();
        if (i < c) {
            x = lkeys[i];
            const uint32_t j1 = (part + 1) * q4 < c ? (part + 1) * q4 : c;
            uint32_t r = 0;
            for (uint32_t j = part * q4; j < j1; j++) r += lkeys[j] > x ? 1u : 0u;
            if (r) atomicAdd(&fs.bins[i], r);
        }
        __syncthreads();
        if (tid < c) regb[fs.bins[tid]] = x;  // the offsets are used up
        __syncthreads();
        emit_sorted<BS>(regb, want, k, fo);
        return;
    }
    // the interval of a key, and the cut: the interval that holds the want-th
    // (bins[] counts, then starts)
    uint64_t lo = ~0ull, hi = 0;
    int shift = 0;
    auto interval = [&](uint64_t x) __attribute__((always_inline)) { return (uint32_t)((hi - x) >> shift); };
    auto range = [&]() __attribute__((always_inline)) {
        lo = wave_min_u64(lo);
        hi = wave_max_u64(hi);
        if (lane_id() == 0) {
            fs.wlo[wave] = lo;
            fs.whi[wave] = hi;
        }
        __syncthreads();
#pragma unroll
        for (int w = 0; w < BS / 64; w++) {
            lo = fs.wlo[w] < lo ? fs.wlo[w] : lo;
            hi = fs.whi[w] > hi ? fs.whi[w] : hi;
        }
        const int width = 64 - (hi > lo ? __builtin_clzll(hi - lo) : 63);
        shift = width > 10 ? width - 10 : 0;  // interval 0 holds the largest keys
    };
    constexpr int BPT = FUSE_BINS / BS;
    auto starts = [&](uint32_t most) __attribute__((always_inline)) {
        uint32_t n_[BPT], sum = 0;
#pragma unroll
        for (int j = 0; j < BPT; j++) {
            n_[j] = fs.bins[tid * BPT + j];
            sum += n_[j];
        }
        uint32_t at = block_excl_scan<BS>(sum, wsum, &total);
#pragma unroll
        for (int j = 0; j < BPT; j++) {
            fs.bins[tid * BPT + j] = at;
            if (at < want) {
                if (n_[j] > most) fs.crowded = 1;
                if (at + n_[j] >= want) {  // holds the last result
                    fs.cut = tid * BPT + j;
                    fs.ncut = at + n_[j];
                }
            }
            at += n_[j];
        }
        __syncthreads();
    };
    uint32_t held = c;  // keys in lkeys
    bool few = c <= cap;
    if (!few) {
        for_candidates<BS>(v, c, [&](uint64_t x) __attribute__((always_inline)) {
            lo = x < lo ? x : lo;
            hi = x > hi ? x : hi;
        });
        range();
        for_candidates<BS>(v, c, [&](uint64_t x) __attribute__((always_inline)) { atomicAdd(&fs.bins[interval(x)], 1u); });
        __syncthreads();
        starts(0xFFFFFFFFu);
        if (fs.ncut <= cap) {
            held = fs.ncut;
            const uint32_t cut = fs.cut;
            if (tid == 0) s_spill = 0;  // used up: the next free place in lkeys
            __syncthreads();
            for_candidates<BS>(v, c, [&](uint64_t x) __attribute__((always_inline)) {
                if (interval(x) <= cut) lkeys[atomicAdd(&s_spill, 1u)] = x;
            });
            for (uint32_t b = tid; b < FUSE_BINS; b += BS) fs.bins[b] = 0;
            few = true;
            lo = ~0ull;
            hi = 0;
        }
        __syncthreads();
    }
    if (few) {
        for (uint32_t i = tid; i < held; i += BS) {
            const uint64_t x = c <= cap ? v.get(i) : lkeys[i];
            if (c <= cap) lkeys[i] = x;
            lo = x < lo ? x : lo;
            hi = x > hi ? x : hi;
        }
        range();
        for (uint32_t i = tid; i < held; i += BS) atomicAdd(&fs.bins[interval(lkeys[i])], 1u);
        __syncthreads();
        starts(FUSE_BIN_MAX);
        if (!fs.crowded) {
            // the intervals up to the cut, in order; bins[] turns from an
            // interval's start into its end (the offsets in regb are used up)
            for (uint32_t i = tid; i < held; i += BS) {
                const uint64_t x = lkeys[i];
                const uint32_t b = interval(x);
                if (b <= fs.cut) regb[atomicAdd(&fs.bins[b], 1u)] = x;
            }
            __syncthreads();
            sorted = lkeys;
            for (uint32_t i = tid; i < fs.ncut; i += BS) {
                const uint64_t x = regb[i];
                const uint32_t b = interval(x);
                const uint32_t s0 = b ? fs.bins[b - 1] : 0u, s1 = fs.bins[b];
                uint32_t r = s0;
                for (uint32_t j = s0; j < s1; j++) r += regb[j] > x ? 1u : 0u;
                if (r < want) sorted[r] = x;
            }
            __syncthreads();
        }
    }
    if (!few || fs.crowded) {
        uint32_t got;
        if (few) {
            const uint64_t thr =
                held > k ? block_kth_largest<BS, MemKeys<BS>, 8>(MemKeys<BS>{lkeys, held}, held, k, fs.rs) : 1ull;
            got = block_gather_ge<BS>(MemKeysUniform<BS>{lkeys, held}, thr, regb, fs.rs);
            sorted = regb;
        } else {
            const uint64_t thr = block_kth_largest<BS, ViewKeys<BS, SlotView, false>, 8>(
                ViewKeys<BS, SlotView, false>{v, c}, c, k, fs.rs);
            got = block_gather_ge<BS>(ViewKeys<BS, SlotView, true>{v, c}, thr, lkeys, fs.rs);
            sorted = lkeys;
        }
        if (got <= (uint32_t)BS) {  // a rank pass, else a bitonic sort (got^2 compares grow past it)
            const uint64_t x = tid < got ? sorted[tid] : 0ull;
            uint32_t r = 0, unused = 0;
            rank2_lds(sorted, got, x, x, r, unused);
            __syncthreads();
            if (tid < got) sorted[r] = x;
            __syncthreads();
        } else {
            for (uint32_t i = got + tid; i < kp2; i += BS) sorted[i] = 0;
            __syncthreads();
            bitonic_sort_desc<BS>(sorted, kp2);
        }
    }
    emit_sorted<BS>(sorted, want, k, fo);
}

}  // namespace topk
