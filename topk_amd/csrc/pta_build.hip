// Partition layout of the PTA path on gfx950 (topk_init with TOPK_INIT_PTA).
//
// Reference: cpu/PTA.h:88-267 (partition build: polar angles, sorted lists,
// per-block threshold vectors); the grouping here is this engine's own: a
// k-d tree over a deterministic sample of the store, whose leaves are the
// partitions; objects are counting-sorted by leaf, then ordered inside each
// partition by attribute sum (largest first, ties by id); every partition
// keeps its box, its largest attribute sum and the sum of its minima, every
// 256-object chunk the same over itself and the later chunks of its
// partition (suffix rows), and a bound tree aggregates the partitions.
//
// Everything runs on the device; the host only deals out the tree's segments,
// whose sizes depend on the counts alone, and learns the padded size:
//
//  1. sample rows (row-major, so that a node's objects stay one load each).
//  2. tree: a level splits every segment of the sample at the exact median
//     of its widest axis -- column extremes, three radix passes over the
//     axis values, a stable partition -- and segments of at most KD_SUB rows
//     finish their whole subtree in one workgroup.  Order among equal values
//     is the row index, so the tree is a function of the store.
//  3. assign: each object walks the tree (its copy in LDS); its workgroup
//     writes the rows of its range, counts leaves in LDS, reserves its share
//     of each leaf with one global atomic and lists its range in leaf order.
//  4. scatter: each workgroup's rows and their ordering keys go to the
//     partitions in that order, in runs of neighbouring rows.  (Object by
//     object, 16M random 32-byte writes took 1.1 ms; a gather of columns by
//     sorted id would fetch a 64-byte line for every 4 bytes.)
//  5. one workgroup per partition sorts the keys in LDS by one counting pass
//     and ranks, writes the columns and ids in that order, and reduces every
//     statistic from the staged columns.
//  6. bound tree, level by level.
//
// At N = 2^24, d = 8 (4096 partitions) a rebuild takes 3.0 ms: scatter 0.87,
// assign 0.65, partitions 0.51, the tree 0.7 (device-wide levels 65 us each,
// subtrees 0.17), sample 0.14.  The tree on the host, with the columns
// gathered and sorted by separate passes, took 71 ms, 53 of them the host's.
//
// Steps 4 and 5 in this form need every partition inside PTA_SORT_MAX objects:
// a single larger one sends the whole store through separate passes (below),
// where the gather of single words leads (2^28 x 8: 54 of 120 ms).
#include <string.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <vector>

#include "bound.hpp"
#include "device.hpp"
#include "internal.hpp"

namespace topk {

constexpr uint32_t PTA_SORT_MAX = 8192;  // objects of a partition that is sorted (larger: scatter order)

// Split of the node between leaves i and i + 1: objects below go left.  The
// shape is implied: the subtree of leaves [lo, lo + nl) has its root between
// leaves lo + nl / 2 - 1 and lo + nl / 2.
struct KdNode {
    float split;
    uint32_t axis;
};

// ---------------------------------------------------------------------------
// 1. sample
// ---------------------------------------------------------------------------
// Row j of the sample is object j * n / s; rows have dp floats (d rounded up
// to 4, zero filled).
__global__ __launch_bounds__(256) void kd_sample_kernel(const float *__restrict__ cols, uint64_t ld, uint32_t d,
                                                        uint32_t dp, uint64_t n, uint64_t s, float *__restrict__ rows,
                                                        uint32_t *__restrict__ idx) {
    const uint64_t j = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (j >= s) return;
    const uint64_t i = j * n / s;
    for (uint32_t m = 0; m < dp; m += 4) {
        f4 v;
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = m + e < d ? cols[(uint64_t)(m + e) * ld + i] : 0.0f;
        *reinterpret_cast<f4 *>(rows + j * dp + m) = v;
    }
    idx[j] = (uint32_t)j;
}

// ---------------------------------------------------------------------------
// 2. k-d tree
// ---------------------------------------------------------------------------
// The subtree of leaves [leaf_lo, leaf_lo + nl) over sample positions
// [lo, hi); its root splits at position lo + (hi - lo) * (nl / 2) / nl and is
// node leaf_lo + nl / 2 - 1.
struct KdSeg {
    uint32_t lo, hi, leaf_lo, nl;
    __host__ __device__ uint32_t nleft() const { return nl / 2; }
    __host__ __device__ uint32_t mid() const { return lo + (uint32_t)((uint64_t)(hi - lo) * nleft() / nl); }
    __host__ __device__ uint32_t node() const { return leaf_lo + nleft() - 1; }
};
// A workgroup's share [b, e) of segment seg; its segment's shares start at first.
struct KdShare {
    uint32_t seg, b, e, first;
};
constexpr uint32_t KD_SHARE = 4096, KD_BS = 256, KD_EPT = KD_SHARE / KD_BS;
constexpr uint32_t KD_SUB = 4096, KD_SUB_LEAVES = 64;  // rows and leaves of a subtree one workgroup builds
constexpr int KD_PASSES = 3;
constexpr uint32_t KD_BINS = 2048;
constexpr int KD_SHIFT[KD_PASSES] = {21, 10, 0};
constexpr int KD_WIDTH[KD_PASSES] = {11, 11, 10};
// Scratch of one segment of a level, cleared before it.
struct KdState {
    uint32_t ext[2 * TOPK_MAX_DIMS];   // okey maxima, then maxima of ~okey
    uint32_t hist[KD_PASSES][KD_BINS];
    uint32_t prefix[KD_PASSES], rank[KD_PASSES];  // after pass p: key bits found, rank left among the keys that share them
};

// Ordering key of an axis value: -0 and +0 are one value to the comparisons.
__device__ __forceinline__ uint32_t kd_key(float v) { return okey(v + 0.0f); }

// Widest axis of a node from its extremes (ext as in KdState, stride apart):
// the lowest axis among equals.
__device__ __forceinline__ uint32_t kd_axis(const uint32_t *ext, uint32_t d) {
    uint32_t axis = 0;
    float best = -1.0f;
    for (uint32_t m = 0; m < d; m++) {
        const float w = okey_inv(ext[m]) - okey_inv(~ext[TOPK_MAX_DIMS + m]);
        if (w > best) {
            best = w;
            axis = m;
        }
    }
    return axis;
}

__global__ __launch_bounds__(KD_BS) void kd_extremes_kernel(const KdShare *__restrict__ shares,
                                                            const uint32_t *__restrict__ idx,
                                                            const float *__restrict__ rows, uint32_t d, uint32_t dp,
                                                            KdState *__restrict__ st) {
    __shared__ uint32_t ext[2 * TOPK_MAX_DIMS];
    const KdShare sh = shares[blockIdx.x];
    if (threadIdx.x < 2 * TOPK_MAX_DIMS) ext[threadIdx.x] = 0;
    __syncthreads();
    uint32_t id[KD_EPT];
#pragma unroll
    for (uint32_t j = 0; j < KD_EPT; j++) {
        const uint32_t p = sh.b + j * KD_BS + threadIdx.x;
        id[j] = idx[p < sh.e ? p : sh.b];  // past the end: the first row again
    }
    for (uint32_t m = 0; m < dp; m += 4) {
        uint32_t mx[4] = {0, 0, 0, 0}, mn[4] = {0, 0, 0, 0};
#pragma unroll
        for (uint32_t j = 0; j < KD_EPT; j++) {
            const f4 v = *reinterpret_cast<const f4 *>(rows + (uint64_t)id[j] * dp + m);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t k = okey(v[e]);
                mx[e] = k > mx[e] ? k : mx[e];
                mn[e] = ~k > mn[e] ? ~k : mn[e];
            }
        }
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t a = wave_max_u32(mx[e]), b = wave_max_u32(mn[e]);
            if (lane_id() == 0 && m + e < d) {
                atomicMax(&ext[m + e], a);
                atomicMax(&ext[TOPK_MAX_DIMS + m + e], b);
            }
        }
    }
    __syncthreads();
    uint32_t *out = st[sh.seg].ext;
    if (threadIdx.x < d) atomicMax(&out[threadIdx.x], ext[threadIdx.x]);
    else if (threadIdx.x >= TOPK_MAX_DIMS && threadIdx.x < TOPK_MAX_DIMS + d)
        atomicMax(&out[threadIdx.x], ext[threadIdx.x]);
}

// The digit of pass P's finished histogram that holds the wanted rank, found
// by every workgroup of the segment; prefix and rank of the pass on return.
template <int P>
__device__ __forceinline__ void kd_pick(const KdSeg &sg, const KdState &st, uint32_t &prefix, uint32_t &rank) {
    __shared__ uint32_t wsum[KD_BS / 64], total, s_digit, s_rank;
    constexpr uint32_t PER = KD_BINS / KD_BS;
    const uint32_t want = P ? st.rank[P > 0 ? P - 1 : 0] : sg.mid() - sg.lo;
    uint32_t c[PER], sum = 0;
#pragma unroll
    for (uint32_t j = 0; j < PER; j++) {
        c[j] = st.hist[P][threadIdx.x * PER + j];
        sum += c[j];
    }
    uint32_t at = block_excl_scan<KD_BS>(sum, wsum, &total);
#pragma unroll
    for (uint32_t j = 0; j < PER; j++) {
        if (at <= want && want < at + c[j]) {
            s_digit = threadIdx.x * PER + j;
            s_rank = want - at;
        }
        at += c[j];
    }
    __syncthreads();
    prefix = (P ? st.prefix[P > 0 ? P - 1 : 0] : 0u) | (s_digit << KD_SHIFT[P]);
    rank = s_rank;
    __syncthreads();
}

// Pass P of the radix select of each segment's median: the first pass takes
// the axis values from the rows and keeps their keys in val[].  The first
// workgroup of a segment records what the pass before found.
template <int P>
__global__ __launch_bounds__(KD_BS) void kd_hist_kernel(const KdShare *__restrict__ shares,
                                                        const KdSeg *__restrict__ segs,
                                                        const uint32_t *__restrict__ idx,
                                                        const float *__restrict__ rows, uint32_t d, uint32_t dp,
                                                        uint32_t *__restrict__ val, KdState *__restrict__ states) {
    __shared__ uint32_t h[KD_BINS];
    __shared__ uint32_t s_axis;
    const KdShare sh = shares[blockIdx.x];
    KdState &st = states[sh.seg];
    uint32_t prefix = 0, rank = 0;
    for (uint32_t i = threadIdx.x; i < KD_BINS; i += KD_BS) h[i] = 0;
    if constexpr (P == 0) {
        if (threadIdx.x == 0) s_axis = kd_axis(st.ext, d);
    } else {
        kd_pick<P - 1>(segs[sh.seg], st, prefix, rank);
        if (blockIdx.x == sh.first && threadIdx.x == 0) {
            st.prefix[P - 1] = prefix;
            st.rank[P - 1] = rank;
        }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < KD_EPT; j++) {
        const uint32_t p = sh.b + j * KD_BS + threadIdx.x;
        if (p >= sh.e) break;
        uint32_t k;
        if constexpr (P == 0) {
            k = kd_key(rows[(uint64_t)idx[p] * dp + s_axis]);
            val[p] = k;
        } else {
            k = val[p];
            constexpr int above = KD_SHIFT[P > 0 ? P - 1 : 0];
            if ((k >> above) != (prefix >> above)) continue;
        }
        atomicAdd(&h[(k >> KD_SHIFT[P]) & ((1u << KD_WIDTH[P]) - 1u)], 1u);
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < KD_BINS; i += KD_BS)
        if (h[i]) atomicAdd(&st.hist[P][i], h[i]);
}

// Rows of each share below the median value, and equal to it; the segment's
// node.  rank is then the number of equal rows (lowest indexes) that go left.
__global__ __launch_bounds__(KD_BS) void kd_count_kernel(const KdShare *__restrict__ shares,
                                                         const KdSeg *__restrict__ segs, uint32_t d,
                                                         const uint32_t *__restrict__ val,
                                                         KdState *__restrict__ states, uint2 *__restrict__ cnt,
                                                         KdNode *__restrict__ nodes) {
    __shared__ uint32_t wc[KD_BS / 64][2];
    const KdShare sh = shares[blockIdx.x];
    const KdSeg sg = segs[sh.seg];
    KdState &st = states[sh.seg];
    uint32_t key, rank;
    kd_pick<KD_PASSES - 1>(sg, st, key, rank);
    if (blockIdx.x == sh.first && threadIdx.x == 0) {
        st.prefix[KD_PASSES - 1] = key;
        st.rank[KD_PASSES - 1] = rank;
        nodes[sg.node()] = KdNode{okey_inv(key), kd_axis(st.ext, d)};
    }
    uint32_t less = 0, same = 0;
#pragma unroll
    for (uint32_t j = 0; j < KD_EPT; j++) {
        const uint32_t p = sh.b + j * KD_BS + threadIdx.x;
        const uint32_t k = p < sh.e ? val[p] : 0xFFFFFFFFu;
        less += p < sh.e && k < key ? 1u : 0u;
        same += p < sh.e && k == key ? 1u : 0u;
    }
    less = wave_sum_u32(less);
    same = wave_sum_u32(same);
    if (lane_id() == 0) {
        wc[threadIdx.x / 64][0] = less;
        wc[threadIdx.x / 64][1] = same;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint2 r = make_uint2(0u, 0u);
        for (uint32_t w = 0; w < KD_BS / 64; w++) {
            r.x += wc[w][0];
            r.y += wc[w][1];
        }
        cnt[blockIdx.x] = r;
    }
}

// Stable partition of every segment around its median: each thread takes
// KD_EPT consecutive positions.
__global__ __launch_bounds__(KD_BS) void kd_split_kernel(const KdShare *__restrict__ shares,
                                                         const KdSeg *__restrict__ segs,
                                                         const uint32_t *__restrict__ idx,
                                                         const uint32_t *__restrict__ val,
                                                         const KdState *__restrict__ states,
                                                         const uint2 *__restrict__ cnt, uint32_t *__restrict__ out) {
    __shared__ uint32_t wsum[KD_BS / 64], tot_less, tot_same, tot;
    const KdShare sh = shares[blockIdx.x];
    const KdSeg sg = segs[sh.seg];
    const uint32_t key = states[sh.seg].prefix[KD_PASSES - 1], need = states[sh.seg].rank[KD_PASSES - 1];
    // rows of the segment's earlier shares
    uint32_t a = 0, b = 0;
    for (uint32_t s = sh.first + threadIdx.x; s < blockIdx.x; s += KD_BS) {
        const uint2 c = cnt[s];
        a += c.x;
        b += c.y;
    }
    block_excl_scan<KD_BS>(a, wsum, &tot_less);
    block_excl_scan<KD_BS>(b, wsum, &tot_same);
    uint32_t v[KD_EPT], id[KD_EPT], same = 0;
    const uint32_t p0 = sh.b + threadIdx.x * KD_EPT;
#pragma unroll
    for (uint32_t j = 0; j < KD_EPT; j++) {
        const bool on = p0 + j < sh.e;
        v[j] = on ? val[p0 + j] : 0xFFFFFFFFu;
        id[j] = on ? idx[p0 + j] : 0u;
        same += on && v[j] == key ? 1u : 0u;
    }
    uint32_t eq = tot_same + block_excl_scan<KD_BS>(same, wsum, &tot);  // equal rows before this thread's
    uint32_t left = 0, lm = 0;
#pragma unroll
    for (uint32_t j = 0; j < KD_EPT; j++) {
        const bool on = p0 + j < sh.e, is = on && v[j] == key;
        const bool l = on && (v[j] < key || (is && eq < need));
        eq += is ? 1u : 0u;
        lm |= l ? 1u << j : 0u;
        left += l ? 1u : 0u;
    }
    // rows before this share that went left: the smaller ones, and the equal ones up to `need`
    uint32_t at = tot_less + (tot_same < need ? tot_same : need) + block_excl_scan<KD_BS>(left, wsum, &tot);
    const uint32_t mid = sg.mid();
#pragma unroll
    for (uint32_t j = 0; j < KD_EPT; j++) {
        const bool l = (lm >> j) & 1u;
        if (p0 + j < sh.e) out[l ? sg.lo + at : mid + (p0 + j - sg.lo - at)] = id[j];
        at += l ? 1u : 0u;
    }
}

// One workgroup builds a whole subtree.  Its rows stay in LDS as (axis key,
// row) words, a node's in one run; a level counting-sorts every node's run by
// equal intervals of its axis range, and orders only the interval that holds
// the split position, by pairs: what lies in the intervals around it is on
// its side already.  (A bitonic sort of the words took 72 us a level.)
constexpr uint32_t KD_SUB_BINS = 4096;
struct KdSubScratch {
    uint64_t a[KD_SUB], b[KD_SUB];
    uint32_t bins[KD_SUB_BINS];
    uint8_t of[KD_SUB];  // node of each position
    KdSeg nd[2][KD_SUB_LEAVES];
    uint32_t ext[KD_SUB_LEAVES][2 * TOPK_MAX_DIMS];
    uint32_t axis[KD_SUB_LEAVES], kmin[KD_SUB_LEAVES], shift[KD_SUB_LEAVES], child[KD_SUB_LEAVES];
    uint32_t wsum[16], total, nn, more;
};
static_assert(sizeof(KdSubScratch) <= 150 * 1024, "one workgroup per CU");
__global__ __launch_bounds__(1024) void kd_subtree_kernel(const KdSeg *__restrict__ subs,
                                                          const uint32_t *__restrict__ idx,
                                                          const float *__restrict__ rows, uint32_t d, uint32_t dp,
                                                          KdNode *__restrict__ nodes) {
    __shared__ KdSubScratch S;
    const uint32_t tid = threadIdx.x, lane = lane_id();
    const KdSeg root = subs[blockIdx.x];
    const uint32_t n = root.hi - root.lo;
    for (uint32_t i = tid; i < n; i += 1024) {
        S.a[i] = idx[root.lo + i];
        S.of[i] = 0;
    }
    if (tid == 0) {
        S.nd[0][0] = KdSeg{0, n, root.leaf_lo, root.nl};
        S.nn = 1;
    }
    __syncthreads();
    for (uint32_t cur = 0;; cur ^= 1) {
        const uint32_t nn = S.nn;
        const KdSeg *nd = S.nd[cur];
        uint32_t lb = 12;  // log2 of the intervals of a node
        while (lb > 6 && (nn << lb) > KD_SUB_BINS) lb--;
        for (uint32_t i = tid; i < nn * 2 * TOPK_MAX_DIMS; i += 1024) (&S.ext[0][0])[i] = 0;
        for (uint32_t i = tid; i < KD_SUB_BINS; i += 1024) S.bins[i] = 0;
        __syncthreads();
        // extremes of every node: 64 positions per wave and step, the lanes
        // of one node at a time
        for (uint32_t p0 = tid - lane; p0 < n; p0 += 1024) {
            const uint32_t p = p0 + lane < n ? p0 + lane : p0;
            const uint32_t row = (uint32_t)S.a[p] & 0xFFFFFFu, of = S.of[p];
            for (uint32_t m = 0; m < dp; m += 4) {
                const f4 v = *reinterpret_cast<const f4 *>(rows + (uint64_t)row * dp + m);
                for (uint64_t left = ~0ull; left;) {
                    const uint32_t o = (uint32_t)__builtin_amdgcn_readlane((int)of, (int)__builtin_ctzll(left));
                    const bool mine = of == o;
                    left &= ~__ballot(mine);
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const uint32_t k = okey(v[e]);
                        const uint32_t mx = wave_max_u32(mine ? k : 0u), mn = wave_max_u32(mine ? ~k : 0u);
                        if (lane == 0 && m + e < d) {
                            atomicMax(&S.ext[o][m + e], mx);
                            atomicMax(&S.ext[o][TOPK_MAX_DIMS + m + e], mn);
                        }
                    }
                }
            }
        }
        __syncthreads();
        if (tid < nn) {
            const uint32_t ax = kd_axis(S.ext[tid], d);
            const uint32_t k0 = kd_key(okey_inv(~S.ext[tid][TOPK_MAX_DIMS + ax])), k1 = kd_key(okey_inv(S.ext[tid][ax]));
            const int width = k1 > k0 ? 32 - __builtin_clz(k1 - k0) : 0;
            S.axis[tid] = ax;
            S.kmin[tid] = k0;
            S.shift[tid] = width > (int)lb ? (uint32_t)width - lb : 0u;
        }
        __syncthreads();
        auto bin = [&](uint64_t w, uint32_t of) {
            return (of << lb) + (nd[of].nl > 1 ? ((uint32_t)(w >> 24) - S.kmin[of]) >> S.shift[of] : 0u);
        };
        for (uint32_t i = tid; i < n; i += 1024) {
            const uint32_t row = (uint32_t)S.a[i] & 0xFFFFFFu, of = S.of[i];
            const uint64_t w = ((uint64_t)kd_key(rows[(uint64_t)row * dp + S.axis[of]]) << 24) | row;
            S.a[i] = w;
            atomicAdd(&S.bins[bin(w, of)], 1u);
        }
        __syncthreads();
        {
            constexpr uint32_t PER = KD_SUB_BINS / 1024;
            uint32_t c[PER], sum = 0;
#pragma unroll
            for (uint32_t j = 0; j < PER; j++) {
                c[j] = S.bins[tid * PER + j];
                sum += c[j];
            }
            uint32_t at = block_excl_scan<1024>(sum, S.wsum, &S.total);
#pragma unroll
            for (uint32_t j = 0; j < PER; j++) {
                S.bins[tid * PER + j] = at;
                at += c[j];
            }
        }
        __syncthreads();
        for (uint32_t i = tid; i < n; i += 1024) {
            const uint64_t w = S.a[i];
            S.b[atomicAdd(&S.bins[bin(w, S.of[i])], 1u)] = w;  // a node's intervals fill its run
        }
        __syncthreads();
        for (uint32_t i = tid; i < n; i += 1024) {
            const uint64_t w = S.b[i];
            const uint32_t of = S.of[i], b = bin(w, of), mid = nd[of].mid();
            const uint32_t s0 = b ? S.bins[b - 1] : 0u, s1 = S.bins[b];
            uint32_t r = i;
            if (nd[of].nl > 1 && s0 <= mid && mid < s1) {
                r = s0;
                for (uint32_t j = s0; j < s1; j++) r += S.b[j] < w ? 1u : 0u;
            }
            S.a[r] = w;
        }
        __syncthreads();
        // nodes, and the next level's table in position order
        if (tid < 64) {
            const bool on = tid < nn;
            const KdSeg s = on ? nd[tid] : KdSeg{0, 0, 0, 1};
            const uint32_t kids = on ? (s.nl > 1 ? 2u : 1u) : 0u;
            const uint32_t at = wave_incl_scan(kids) - kids;
            const uint32_t nl = s.nleft(), mid = s.mid();
            if (on) {
                S.child[tid] = at;
                if (s.nl > 1) {
                    nodes[s.node()] = KdNode{okey_inv((uint32_t)(S.a[mid] >> 24)), S.axis[tid]};
                    S.nd[cur ^ 1][at] = KdSeg{s.lo, mid, s.leaf_lo, nl};
                    S.nd[cur ^ 1][at + 1] = KdSeg{mid, s.hi, s.leaf_lo + nl, s.nl - nl};
                } else {
                    S.nd[cur ^ 1][at] = s;
                }
            }
            const uint64_t any = __ballot(on && s.nl >= 3);
            const uint32_t all = wave_sum_u32(kids);
            if (tid == 0) {
                S.nn = all;
                S.more = any != 0;
            }
        }
        __syncthreads();
        if (!S.more) return;
        for (uint32_t i = tid; i < n; i += 1024) {
            const uint32_t of = S.of[i];
            S.of[i] = (uint8_t)(S.child[of] + (nd[of].nl > 1 && i >= nd[of].mid() ? 1u : 0u));
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// 3. assign
// ---------------------------------------------------------------------------
constexpr uint32_t PA_BS = 1024;

struct AssignArgs {
    const float *cols;
    uint64_t ld, n, per;  // workgroup g takes objects [g * per, (g + 1) * per)
    uint32_t d, dp, L;
    const KdNode *nodes;
    int tree_lds;         // the tree fits in LDS
    uint2 *place;         // leaf and rank of each object (null: not kept)
    uint32_t *cnt;        // objects per leaf
    // counted in LDS (else null): per workgroup and leaf, what added to the
    // leaf's offset and an index in leaf order gives the position; the range
    // in leaf order (object, leaf); the objects' rows
    uint32_t *base;
    uint2 *order;
    float *rows;
    // without place: ids to their partitions (cnt then counts them again)
    const uint32_t *poff;
    uint32_t *pid;
};

// Dynamic LDS: d x PA_BS attribute values (a lane reads its own column of
// them, so any axis is free of bank conflicts), the tree (L splits, L axes)
// and L counters as they fit.
__global__ __launch_bounds__(PA_BS) void pta_assign_kernel(AssignArgs a) {
    extern __shared__ float pa_lds[];
    __shared__ uint32_t wsum[PA_BS / 64], total;
    const uint32_t tid = threadIdx.x, L = a.L, d = a.d;
    float *x = pa_lds;
    uint32_t *h = reinterpret_cast<uint32_t *>(x + (size_t)d * PA_BS);
    float *ts = reinterpret_cast<float *>(h + (a.base ? L : 0u));
    uint8_t *ta = reinterpret_cast<uint8_t *>(ts + L);
    if (a.base)
        for (uint32_t l = tid; l < L; l += PA_BS) h[l] = 0;
    if (a.tree_lds)
        for (uint32_t l = tid; l + 1 < L; l += PA_BS) {
            const KdNode nd = a.nodes[l];
            ts[l] = nd.split;
            ta[l] = (uint8_t)nd.axis;
        }
    __syncthreads();
    const uint64_t i0 = (uint64_t)blockIdx.x * a.per, i1 = i0 + a.per < a.n ? i0 + a.per : a.n;
    for (uint64_t i = i0 + tid; i < i1; i += PA_BS) {
        for (uint32_t m = 0; m < a.dp; m += 4) {
            f4 v;
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = m + e < d ? a.cols[(uint64_t)(m + e) * a.ld + i] : 0.0f;
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (m + e < d) x[(m + e) * PA_BS + tid] = v[e];
            if (a.rows) *reinterpret_cast<f4 *>(a.rows + i * a.dp + m) = v;
        }
        uint32_t lo = 0;
        for (uint32_t nl = L; nl > 1;) {
            const uint32_t nleft = nl / 2, c = lo + nleft - 1;
            float split;
            uint32_t axis;
            if (a.tree_lds) {
                split = ts[c];
                axis = ta[c];
            } else {
                const KdNode nd = a.nodes[c];
                split = nd.split;
                axis = nd.axis;
            }
            const bool left = x[axis * PA_BS + tid] < split;
            lo += left ? 0u : nleft;
            nl = left ? nleft : nl - nleft;
        }
        const uint32_t r = a.base ? atomicAdd(&h[lo], 1u) : atomicAdd(&a.cnt[lo], 1u);
        if (a.place) a.place[i] = make_uint2(lo, r);
        else if (a.pid) a.pid[a.poff[lo] + r] = (uint32_t)i;
    }
    if (!a.base) return;
    __syncthreads();
    // the counts' offsets in leaf order, and this workgroup's share of every leaf
    const uint32_t per = (L + PA_BS - 1) / PA_BS, b0 = tid * per < L ? tid * per : L, b1 = b0 + per < L ? b0 + per : L;
    uint32_t sum = 0;
    for (uint32_t l = b0; l < b1; l++) sum += h[l];
    uint32_t at = block_excl_scan<PA_BS>(sum, wsum, &total);
    for (uint32_t l = b0; l < b1; l++) {
        const uint32_t c = h[l];
        h[l] = at;
        a.base[(uint64_t)blockIdx.x * L + l] = (c ? atomicAdd(&a.cnt[l], c) : 0u) - at;
        at += c;
    }
    __syncthreads();
    for (uint64_t i = i0 + tid; i < i1; i += PA_BS) {
        const uint2 pl = a.place[i];
        a.order[i0 + h[pl.x] + pl.y] = make_uint2((uint32_t)i, pl.x);
    }
}

// Partitions past PTA_SORT_MAX objects stay as scattered.  They hold repeated
// values, whose best objects are those of the lowest ids, and a query's seed
// takes a partition's first objects: in the order in which the assign
// workgroups happened to reserve their shares, 512 queries over N = 2^23 equal
// objects (d = 8) all kept more ties than a list holds, 129 ms; in id order
// 0.9 ms.  So the shares are given out again, workgroup by workgroup: recounted
// here, and made prefixes over the workgroups, a thread per leaf, below.
__global__ __launch_bounds__(PA_BS) void pta_recount_kernel(AssignArgs a) {
    extern __shared__ float pa_lds[];
    uint32_t *h = reinterpret_cast<uint32_t *>(pa_lds);
    for (uint32_t l = threadIdx.x; l < a.L; l += PA_BS) h[l] = 0;
    __syncthreads();
    const uint64_t i0 = (uint64_t)blockIdx.x * a.per, i1 = i0 + a.per < a.n ? i0 + a.per : a.n;
    for (uint64_t i = i0 + threadIdx.x; i < i1; i += PA_BS) atomicAdd(&h[a.place[i].x], 1u);
    __syncthreads();
    for (uint32_t l = threadIdx.x; l < a.L; l += PA_BS) a.base[(uint64_t)blockIdx.x * a.L + l] = h[l];
}

__global__ __launch_bounds__(256) void pta_base_kernel(uint32_t *__restrict__ base, uint32_t L, uint32_t groups) {
    const uint32_t l = blockIdx.x * 256 + threadIdx.x;
    if (l >= L) return;
    uint32_t at = 0;
    for (uint32_t g0 = 0; g0 < groups; g0 += 8) {
        uint32_t c[8];
#pragma unroll
        for (uint32_t j = 0; j < 8; j++) c[j] = g0 + j < groups ? base[(uint64_t)(g0 + j) * L + l] : 0u;
#pragma unroll
        for (uint32_t j = 0; j < 8; j++)
            if (g0 + j < groups) {
                base[(uint64_t)(g0 + j) * L + l] = at;
                at += c[j];
            }
    }
}

// Padded offsets of the partitions (one workgroup); rep (pinned): padded
// total (two words), nonempty partitions, largest partition.
__global__ __launch_bounds__(1024) void pta_offsets_kernel(const uint32_t *__restrict__ cnt, uint32_t L,
                                                           uint32_t *__restrict__ poff, uint32_t *__restrict__ psz,
                                                           uint32_t *__restrict__ rep) {
    __shared__ uint64_t wtot[16];
    __shared__ uint32_t wne[16], wmx[16];
    const uint32_t tid = threadIdx.x, per = (L + 1023) / 1024;
    const uint32_t b = tid * per < L ? tid * per : L, e = b + per < L ? b + per : L;
    uint64_t sum = 0;
    uint32_t ne = 0, mx = 0;
    for (uint32_t p = b; p < e; p++) {
        const uint32_t c = cnt[p];
        sum += (c + PART_ALIGN - 1) / PART_ALIGN;
        ne += c ? 1u : 0u;
        mx = c > mx ? c : mx;
    }
    // aligned units: a store of fewer than 2^32 objects has fewer than 2^25 of them
    const uint32_t incl = wave_incl_scan((uint32_t)sum);
    ne = wave_sum_u32(ne);
    mx = wave_max_u32(mx);
    if (lane_id() == 63) wtot[tid / 64] = incl;
    if (lane_id() == 0) {
        wne[tid / 64] = ne;
        wmx[tid / 64] = mx;
    }
    __syncthreads();
    uint64_t at = incl - sum, all = 0;
    ne = mx = 0;
    for (uint32_t w = 0; w < 16; w++) {
        at += w < tid / 64 ? wtot[w] : 0ull;
        all += wtot[w];
        ne += wne[w];
        mx = wmx[w] > mx ? wmx[w] : mx;
    }
    for (uint32_t p = b; p < e; p++) {
        const uint32_t c = cnt[p];
        poff[p] = (uint32_t)(at * PART_ALIGN);
        psz[p] = c;
        at += (c + PART_ALIGN - 1) / PART_ALIGN;
    }
    if (tid == 0) {
        poff[L] = (uint32_t)(all * PART_ALIGN);
        *reinterpret_cast<uint64_t *>(rep) = all * PART_ALIGN;
        rep[2] = ne;
        rep[3] = mx;
    }
}

// ---------------------------------------------------------------------------
// 4. scatter
// ---------------------------------------------------------------------------
// Ordering keys, and rows (if out != null), of assign workgroup blockIdx.y's
// objects to their places in the partition order (unordered inside a
// partition): in leaf order, so that a leaf's rows follow each other, or
// (order null, bases by pta_base_kernel) in id order.
__global__ __launch_bounds__(256) void pta_scatter_kernel(AssignArgs a, const uint32_t *__restrict__ poff,
                                                          uint64_t *__restrict__ keys, float *__restrict__ out) {
    const uint64_t i0 = (uint64_t)blockIdx.y * a.per, i1 = i0 + a.per < a.n ? i0 + a.per : a.n;
    const uint32_t *base = a.base ? a.base + (uint64_t)blockIdx.y * a.L : nullptr;
    for (uint64_t q = i0 + blockIdx.x * 256 + threadIdx.x; q < i1; q += gridDim.x * 256) {
        uint32_t i, pos;
        if (a.order) {
            const uint2 o = a.order[q];
            i = o.x;
            pos = poff[o.y] + base[o.y] + (uint32_t)(q - i0);
        } else {
            const uint2 pl = a.place[q];
            i = (uint32_t)q;
            pos = poff[pl.x] + (base ? base[pl.x] : 0u) + pl.y;
        }
        float s = 0.0f;  // attribute sum, in attribute order
        for (uint32_t m = 0; m < a.dp; m += 4) {
            f4 v;
            if (a.rows) {
                v = *reinterpret_cast<const f4 *>(a.rows + (uint64_t)i * a.dp + m);
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = m + e < a.d ? a.cols[(uint64_t)(m + e) * a.ld + i] : 0.0f;
            }
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (m + e < a.d) s += v[e];
            if (out) *reinterpret_cast<f4 *>(out + (uint64_t)pos * a.dp + m) = v;
        }
        keys[pos] = rkey(s, i);
    }
}

// ---------------------------------------------------------------------------
// 5. partitions
// ---------------------------------------------------------------------------
struct PartOut {
    float *pcols;
    uint64_t ldp;
    uint32_t *pid;
    uint64_t nchunks;
    float *cstat;
    uint32_t *cminid;
    float *pmax, *pmin, *psum, *pminsum;
};
constexpr uint32_t PP_BS = 1024, PP_EPT = PTA_SORT_MAX / PP_BS, PP_BINS = 2048;
constexpr uint32_t PP_CHUNKS = PTA_SORT_MAX / PTA_CHUNK;

__device__ __forceinline__ float wave_max_f32(float v) { return okey_inv(wave_max_u32(okey(v))); }
__device__ __forceinline__ float wave_min_f32(float v) { return okey_inv(~wave_max_u32(~okey(v))); }

// One workgroup per partition of at most `cap` objects (cap <= PTA_SORT_MAX).
// The position of an object is the number of larger keys: a counting sort
// over 2048 equal intervals of the key range, then ranks inside an interval.
// The rows are then read once, in their scattered (contiguous) order, two
// columns at a time go through LDS into position order, and a wave writes
// and reduces one chunk of 256.  Dynamic LDS: cap keys -- later two columns,
// or the attribute sums -- and cap list entries.
__global__ __launch_bounds__(PP_BS) void pta_part_kernel(const uint64_t *__restrict__ keys,
                                                         const float *__restrict__ rows, uint32_t d, uint32_t dp,
                                                         const uint32_t *__restrict__ poff,
                                                         const uint32_t *__restrict__ psz, uint32_t cap, PartOut o) {
    extern __shared__ uint64_t pp_lds[];
    uint64_t *lk = pp_lds;
    uint16_t *order = reinterpret_cast<uint16_t *>(pp_lds + cap);
    __shared__ uint32_t bins[PP_BINS];
    __shared__ uint32_t wsum[PP_BS / 64], total;
    __shared__ uint64_t wlo[PP_BS / 64], whi[PP_BS / 64];
    __shared__ float cmx[TOPK_MAX_DIMS][PP_CHUNKS], cmn[TOPK_MAX_DIMS][PP_CHUNKS];
    __shared__ float csum[PP_CHUNKS];
    const uint32_t p = blockIdx.x, tid = threadIdx.x, lane = lane_id(), wave = tid / 64;
    const uint32_t s = psz[p], start = poff[p];
    if (s == 0) {
        if (tid < d) {
            o.pmax[(uint64_t)p * d + tid] = 0.0f;
            o.pmin[(uint64_t)p * d + tid] = 0.0f;
        }
        if (tid == 0) {
            o.psum[p] = -INFINITY;
            o.pminsum[p] = 0.0f;
        }
        return;
    }
    const uint32_t nch = (s + PTA_CHUNK - 1) / PTA_CHUNK;
    uint64_t lo = ~0ull, hi = 0;
    uint64_t key[PP_EPT];
#pragma unroll
    for (uint32_t j = 0; j < PP_EPT; j++) {
        const uint32_t i = j * PP_BS + tid;
        key[j] = i < s ? keys[start + i] : 0ull;
        if (i < s) {
            lk[i] = key[j];
            lo = key[j] < lo ? key[j] : lo;
            hi = key[j] > hi ? key[j] : hi;
        }
    }
    for (uint32_t b = tid; b < PP_BINS; b += PP_BS) bins[b] = 0;
    lo = wave_min_u64(lo);
    hi = wave_max_u64(hi);
    if (lane == 0) {
        wlo[wave] = lo;
        whi[wave] = hi;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t w = 0; w < PP_BS / 64; w++) {
        lo = wlo[w] < lo ? wlo[w] : lo;
        hi = whi[w] > hi ? whi[w] : hi;
    }
    const int width = hi > lo ? 64 - __builtin_clzll(hi - lo) : 1;
    const int shift = width > 11 ? width - 11 : 0;
#pragma unroll
    for (uint32_t j = 0; j < PP_EPT; j++)
        if (j * PP_BS + tid < s) atomicAdd(&bins[(uint32_t)((hi - key[j]) >> shift)], 1u);
    __syncthreads();
    {
        const uint32_t a = bins[2 * tid], b = bins[2 * tid + 1];
        const uint32_t at = block_excl_scan<PP_BS>(a + b, wsum, &total);
        bins[2 * tid] = at;
        bins[2 * tid + 1] = at + a;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < PP_EPT; j++) {
        const uint32_t i = j * PP_BS + tid;
        if (i < s) order[atomicAdd(&bins[(uint32_t)((hi - key[j]) >> shift)], 1u)] = (uint16_t)i;
    }
    __syncthreads();
    // bins[] holds the intervals' ends now
    uint32_t r[PP_EPT];
#pragma unroll
    for (uint32_t j = 0; j < PP_EPT; j++) {
        r[j] = 0;
        if (j * PP_BS + tid < s) {
            const uint32_t b = (uint32_t)((hi - key[j]) >> shift);
            const uint32_t s0 = b ? bins[b - 1] : 0u, s1 = bins[b];
            r[j] = s0;
            for (uint32_t t = s0; t < s1; t++) r[j] += lk[order[t]] > key[j] ? 1u : 0u;
        }
    }
    __syncthreads();  // the keys are used up
    uint32_t *su = reinterpret_cast<uint32_t *>(pp_lds);
#pragma unroll
    for (uint32_t j = 0; j < PP_EPT; j++)
        if (j * PP_BS + tid < s) su[r[j]] = rkey_id(key[j]);
    __syncthreads();
    for (uint32_t c = wave; c < nch; c += PP_BS / 64) {
        const uint32_t q = c * PTA_CHUNK + 4 * lane;
        uint4 v = *reinterpret_cast<const uint4 *>(su + q);
        v.x = q < s ? v.x : 0xFFFFFFFFu;
        v.y = q + 1 < s ? v.y : 0xFFFFFFFFu;
        v.z = q + 2 < s ? v.z : 0xFFFFFFFFu;
        v.w = q + 3 < s ? v.w : 0xFFFFFFFFu;
        *reinterpret_cast<uint4 *>(o.pid + start + q) = v;
        const uint32_t m01 = v.x < v.y ? v.x : v.y, m23 = v.z < v.w ? v.z : v.w;
        const uint32_t mn = ~wave_max_u32(~(m01 < m23 ? m01 : m23));
        if (lane == 0) o.cminid[start / PTA_CHUNK + c] = mn;
    }
    double sums[PP_EPT];
#pragma unroll
    for (uint32_t j = 0; j < PP_EPT; j++) sums[j] = 0.0;
    float *st0 = reinterpret_cast<float *>(pp_lds), *st1 = st0 + cap;
    for (uint32_t m0 = 0; m0 < d; m0 += 4) {
        f4 x[PP_EPT];
#pragma unroll
        for (uint32_t j = 0; j < PP_EPT; j++) {
            const uint32_t i = j * PP_BS + tid;
            if (i < s) x[j] = ld_stream(rows + ((uint64_t)start + i) * dp + m0);
        }
#pragma unroll
        for (uint32_t e = 0; e < 4; e += 2) {
            if (m0 + e >= d) break;
            __syncthreads();  // the stage is free
#pragma unroll
            for (uint32_t j = 0; j < PP_EPT; j++)
                if (j * PP_BS + tid < s) {
                    st0[r[j]] = x[j][e];
                    st1[r[j]] = x[j][e + 1];
                    sums[j] += (double)x[j][e];
                    if (m0 + e + 1 < d) sums[j] += (double)x[j][e + 1];
                }
            __syncthreads();
            for (uint32_t t = wave; t < 2 * nch; t += PP_BS / 64) {
                const uint32_t m = m0 + e + (t & 1), c = t >> 1, q = c * PTA_CHUNK + 4 * lane;
                if (m >= d) continue;
                f4 v = *reinterpret_cast<const f4 *>((t & 1 ? st1 : st0) + q);
                float mx = -INFINITY, mn = INFINITY;
#pragma unroll
                for (uint32_t u = 0; u < 4; u++) {
                    const bool on = q + u < s;
                    mx = on && v[u] > mx ? v[u] : mx;
                    mn = on && v[u] < mn ? v[u] : mn;
                    v[u] = on ? v[u] : 0.0f;
                }
                *reinterpret_cast<f4 *>(o.pcols + (uint64_t)m * o.ldp + start + q) = v;
                mx = wave_max_f32(mx);
                mn = wave_min_f32(mn);
                if (lane == 0) {
                    cmx[m][c] = mx;
                    cmn[m][c] = mn;
                }
            }
        }
    }
    __syncthreads();
    double *sd = reinterpret_cast<double *>(pp_lds);
#pragma unroll
    for (uint32_t j = 0; j < PP_EPT; j++)
        if (j * PP_BS + tid < s) sd[r[j]] = sums[j];
    __syncthreads();
    for (uint32_t c = wave; c < nch; c += PP_BS / 64) {
        double best = -INFINITY;
#pragma unroll
        for (uint32_t u = 0; u < 4; u++) {
            const uint32_t q = c * PTA_CHUNK + 64 * u + lane;
            const double v = q < s ? sd[q] : -INFINITY;
            best = v > best ? v : best;
        }
        for (int x = 32; x > 0; x >>= 1) {
            const double t = __shfl_xor(best, x, 64);
            best = t > best ? t : best;
        }
        if (lane == 0) csum[c] = f32_round_up(best);
    }
    __syncthreads();
    // suffix rows: element e of chunk c over chunks c, c + 1, ...
    const uint64_t S = o.nchunks, c0 = start / PTA_CHUNK;
    if (tid < 2 * d) {
        const bool top = tid < d;
        const uint32_t m = top ? tid : tid - d;
        float *col = top ? cmx[m] : cmn[m];
        float a = top ? -INFINITY : INFINITY;
        for (uint32_t c = nch; c-- > 0;) {
            a = top ? fmaxf(a, col[c]) : fminf(a, col[c]);
            col[c] = a;
            o.cstat[(uint64_t)tid * S + c0 + c] = a;
        }
        (top ? o.pmax : o.pmin)[(uint64_t)p * d + m] = a;
    } else if (tid >= 2 * TOPK_MAX_DIMS && tid < 2 * TOPK_MAX_DIMS + 1) {
        float a = -INFINITY;
        for (uint32_t c = nch; c-- > 0;) {
            a = fmaxf(a, csum[c]);
            o.cstat[2ull * d * S + c0 + c] = a;
        }
        o.psum[p] = a;
    }
    __syncthreads();
    if (tid < nch) {
        double ms = 0.0;
        for (uint32_t m = 0; m < d; m++) ms += (double)cmn[m][tid];
        const float v = f32_round_down(ms);
        o.cstat[(2ull * d + 1) * S + c0 + tid] = v;
        if (tid == 0) o.pminsum[p] = v;
    }
}

// The positions past the last partition: no object, zero values.
__global__ __launch_bounds__(256) void pta_tail_kernel(uint64_t npos, uint64_t ld, uint32_t d, float *__restrict__ pcols,
                                                       uint32_t *__restrict__ pid) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (npos + i < ld) {
        pid[npos + i] = 0xFFFFFFFFu;
        for (uint32_t m = 0; m < d; m++) pcols[(uint64_t)m * ld + npos + i] = 0.0f;
    }
    if (i < 8192) pcols[(uint64_t)d * ld + i] = 0.0f;  // the last column's padding tile
}

// ---- stores with a partition past PTA_SORT_MAX objects, or no room for the
//      scattered rows or for anything per object: the same layout by separate
//      passes ----

// Sorts each partition's keys, largest first (over PTA_SORT_MAX: as scattered).
__global__ __launch_bounds__(1024) void pta_sort_kernel(const uint32_t *__restrict__ poff,
                                                        const uint32_t *__restrict__ psz,
                                                        uint64_t *__restrict__ keys) {
    __shared__ uint64_t a[PTA_SORT_MAX];
    const uint32_t p = blockIdx.x, s = psz[p];
    if (s < 2 || s > PTA_SORT_MAX) return;
    uint64_t *seg = keys + poff[p];
    uint32_t n2 = 1;
    while (n2 < s) n2 <<= 1;
    for (uint32_t i = threadIdx.x; i < n2; i += 1024) a[i] = i < s ? seg[i] : 0ull;
    __syncthreads();
    bitonic_sort_desc<1024>(a, n2);
    for (uint32_t i = threadIdx.x; i < s; i += 1024) seg[i] = a[i];
}

// The same for ids without their keys: the attribute sums are gathered.
__global__ __launch_bounds__(1024) void pta_sort_ids_kernel(const float *__restrict__ cols, uint64_t ld, uint32_t d,
                                                            const uint32_t *__restrict__ poff,
                                                            const uint32_t *__restrict__ psz,
                                                            uint32_t *__restrict__ pid) {
    __shared__ uint64_t a[PTA_SORT_MAX];
    const uint32_t p = blockIdx.x, s = psz[p];
    if (s < 2 || s > PTA_SORT_MAX) return;
    uint32_t *seg = pid + poff[p];
    uint32_t n2 = 1;
    while (n2 < s) n2 <<= 1;
    for (uint32_t i = threadIdx.x; i < n2; i += 1024) {
        uint64_t key = 0;
        if (i < s) {
            const uint32_t id = seg[i];
            float sum = 0.0f;  // attribute sum, in attribute order
            for (uint32_t m = 0; m < d; m++) sum += cols[(uint64_t)m * ld + id];
            key = rkey(sum, id);
        }
        a[i] = key;
    }
    __syncthreads();
    bitonic_sort_desc<1024>(a, n2);
    for (uint32_t i = threadIdx.x; i < s; i += 1024) seg[i] = rkey_id(a[i]);
}

// keys null: the ids are in pid[].
__global__ void pta_gather_kernel(const float *__restrict__ cols, uint64_t ld, uint32_t d, uint64_t npos,
                                  const uint64_t *__restrict__ keys, float *__restrict__ pcols, uint64_t ldp,
                                  uint32_t *__restrict__ pid) {
    const uint64_t pos = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (pos >= npos) return;
    const uint32_t id = keys ? rkey_id(keys[pos]) : pid[pos];  // key 0: no object, id 0xFFFFFFFF
    if (keys) pid[pos] = id;
    for (uint32_t m = 0; m < d; m++) pcols[(uint64_t)m * ldp + pos] = id != 0xFFFFFFFFu ? cols[(uint64_t)m * ld + id] : 0.0f;
}

constexpr int PB_BS = 256;
// One block per partition: per-attribute max/min, the max attribute sum
// (FP64, rounded up) and the sum of the minima (FP64, rounded down).
__global__ __launch_bounds__(PB_BS) void pta_bounds_kernel(const float *__restrict__ pcols, uint64_t ldp, uint32_t d,
                                                            const uint32_t *__restrict__ poff,
                                                            const uint32_t *__restrict__ psz,
                                                            float *__restrict__ pmax, float *__restrict__ pmin,
                                                            float *__restrict__ psum, float *__restrict__ pminsum) {
    __shared__ float smax[PB_BS / 64], smin[PB_BS / 64];
    __shared__ double ssum[PB_BS / 64];
    __shared__ float colmin[TOPK_MAX_DIMS];
    const uint32_t p = blockIdx.x, start = poff[p], s = psz[p];
    const uint32_t w = threadIdx.x / 64;
    for (uint32_t m = 0; m < d; m++) {
        float mx = -INFINITY, mn = INFINITY;
        for (uint32_t i = threadIdx.x; i < s; i += PB_BS) {
            const float v = pcols[(uint64_t)m * ldp + start + i];
            mx = v > mx ? v : mx;
            mn = v < mn ? v : mn;
        }
        for (int o = 32; o > 0; o >>= 1) {
            mx = fmaxf(mx, __shfl_xor(mx, o, 64));
            mn = fminf(mn, __shfl_xor(mn, o, 64));
        }
        if (lane_id() == 0) { smax[w] = mx; smin[w] = mn; }
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int j = 1; j < PB_BS / 64; j++) { mx = fmaxf(mx, smax[j]); mn = fminf(mn, smin[j]); }
            pmax[(uint64_t)p * d + m] = s ? mx : 0.0f;
            pmin[(uint64_t)p * d + m] = s ? mn : 0.0f;
            colmin[m] = s ? mn : 0.0f;
        }
        __syncthreads();
    }
    double best = -INFINITY;
    for (uint32_t i = threadIdx.x; i < s; i += PB_BS) {
        double t = 0;
        for (uint32_t m = 0; m < d; m++) t += (double)pcols[(uint64_t)m * ldp + start + i];
        best = t > best ? t : best;
    }
    for (int o = 32; o > 0; o >>= 1) {
        const double t = __shfl_xor(best, o, 64);
        best = t > best ? t : best;
    }
    if (lane_id() == 0) ssum[w] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int j = 1; j < PB_BS / 64; j++) best = ssum[j] > best ? ssum[j] : best;
        double ms = 0;
        for (uint32_t m = 0; m < d; m++) ms += (double)colmin[m];
        psum[p] = s ? f32_round_up(best) : -INFINITY;
        pminsum[p] = s ? f32_round_down(ms) : 0.0f;
    }
}

// One wave per chunk of PTA_CHUNK positions: element e of chunk c (at
// cstat[e * nchunks + c]) holds the chunk's per-attribute maxima (e in
// [0, d)) and minima ([d, 2d)), the largest attribute sum of its objects
// (FP64, rounded up) at 2d and the sum of its minima (FP64, rounded down)
// at 2d + 1.  A chunk without objects has sum -inf.  cminid[c] gets the
// chunk's smallest object id (0xFFFFFFFF: none).
__global__ __launch_bounds__(256) void pta_chunk_kernel(const float *__restrict__ pcols, uint64_t ldp, uint32_t d,
                                                        const uint32_t *__restrict__ pid, uint64_t nchunks,
                                                        float *__restrict__ cstat, uint32_t *__restrict__ cminid) {
    const uint64_t c = (uint64_t)blockIdx.x * 4 + threadIdx.x / 64;
    if (c >= nchunks) return;
    const uint32_t lane = lane_id();
    constexpr uint32_t PER = PTA_CHUNK / 64;
    const uint64_t pos0 = c * PTA_CHUNK + lane * PER;
    bool ok[PER];
    bool any = false;
    uint32_t idmin = 0xFFFFFFFFu;  // padding positions hold id 0xFFFFFFFF
#pragma unroll
    for (uint32_t j = 0; j < PER; j++) {
        const uint32_t id = pid[pos0 + j];
        ok[j] = id != 0xFFFFFFFFu;
        any |= ok[j];
        idmin = id < idmin ? id : idmin;
    }
    const bool nonempty = __ballot(any) != 0;
    for (int o = 32; o > 0; o >>= 1) {
        const uint32_t t = (uint32_t)__shfl_xor((int)idmin, o, 64);
        idmin = t < idmin ? t : idmin;
    }
    if (lane == 0) cminid[c] = idmin;
    float *row = cstat + c;  // element e at row[e * nchunks]
    double best = -INFINITY, minsum = 0.0;
    double sums[PER];
#pragma unroll
    for (uint32_t j = 0; j < PER; j++) sums[j] = 0.0;
    for (uint32_t m = 0; m < d; m++) {
        float mx = -INFINITY, mn = INFINITY;
#pragma unroll
        for (uint32_t j = 0; j < PER; j++) {
            const float v = pcols[(uint64_t)m * ldp + pos0 + j];
            if (ok[j]) {
                mx = v > mx ? v : mx;
                mn = v < mn ? v : mn;
                sums[j] += (double)v;
            }
        }
        for (int o = 32; o > 0; o >>= 1) {
            mx = fmaxf(mx, __shfl_xor(mx, o, 64));
            mn = fminf(mn, __shfl_xor(mn, o, 64));
        }
        minsum += (double)mn;
        if (lane == 0) {
            row[m * nchunks] = nonempty ? mx : 0.0f;
            row[(d + m) * nchunks] = nonempty ? mn : 0.0f;
        }
    }
#pragma unroll
    for (uint32_t j = 0; j < PER; j++) best = ok[j] && sums[j] > best ? sums[j] : best;
    for (int o = 32; o > 0; o >>= 1) {
        const double t = __shfl_xor(best, o, 64);
        best = t > best ? t : best;
    }
    if (lane == 0) {
        row[2 * d * nchunks] = nonempty ? f32_round_up(best) : -INFINITY;
        row[(2 * d + 1) * nchunks] = nonempty ? f32_round_down(minsum) : 0.0f;
    }
}

// One thread per partition turns its chunk rows into suffix rows: row c
// then bounds chunks c, c + 1, ... of the partition (per-attribute maxima and
// minima, the largest attribute sum, and the sum of the union's minima in
// FP64 rounded down), so a partition's row bounds never increase with c.
__global__ __launch_bounds__(256) void pta_chunk_suffix_kernel(uint32_t L, uint32_t d,
                                                               const uint32_t *__restrict__ poff,
                                                               const uint32_t *__restrict__ psz, uint64_t nchunks,
                                                               float *__restrict__ cstat) {
    const uint32_t p = blockIdx.x * 256 + threadIdx.x;
    if (p >= L || psz[p] == 0) return;
    const uint32_t c0 = poff[p] / PTA_CHUNK, n = (psz[p] + PTA_CHUNK - 1) / PTA_CHUNK;
    const uint64_t S = nchunks;  // element stride
    for (uint32_t i = n - 1; i > 0; i--) {
        const float *nx = cstat + (c0 + i);
        float *row = cstat + (c0 + i - 1);
        double ms = 0.0;
        for (uint32_t m = 0; m < d; m++) {
            row[m * S] = fmaxf(row[m * S], nx[m * S]);
            row[(d + m) * S] = fminf(row[(d + m) * S], nx[(d + m) * S]);
            ms += (double)row[(d + m) * S];
        }
        row[2 * d * S] = fmaxf(row[2 * d * S], nx[2 * d * S]);
        row[(2 * d + 1) * S] = f32_round_down(ms);
    }
}

// ---------------------------------------------------------------------------
// 6. bound tree
// ---------------------------------------------------------------------------
struct TreeOut {
    uint32_t p2, L, d;
    float *tmax, *tmin, *tsum, *tminsum;
    uint32_t *tminid;
};

// Leaves (one thread each, p2 of them): partitions, and empty nodes past them;
// node 0 is never read.
__global__ __launch_bounds__(256) void pta_tree_leaf_kernel(TreeOut t, const uint32_t *__restrict__ poff,
                                                            const uint32_t *__restrict__ psz,
                                                            const float *__restrict__ pmax,
                                                            const float *__restrict__ pmin,
                                                            const float *__restrict__ psum,
                                                            const float *__restrict__ pminsum,
                                                            const uint32_t *__restrict__ cminid) {
    const uint32_t p = blockIdx.x * 256 + threadIdx.x;
    if (p >= t.p2) return;
    const uint64_t nn = 2ull * t.p2, v = t.p2 + p;
    const uint32_t s = p < t.L ? psz[p] : 0u;
    for (uint32_t m = 0; m < t.d; m++) {
        t.tmax[m * nn + v] = s ? pmax[(uint64_t)p * t.d + m] : -INFINITY;
        t.tmin[m * nn + v] = s ? pmin[(uint64_t)p * t.d + m] : INFINITY;
    }
    t.tsum[v] = s ? psum[p] : -INFINITY;
    t.tminsum[v] = s ? pminsum[p] : 0.0f;
    uint32_t id = 0xFFFFFFFFu;
    if (s)
        for (uint32_t c = poff[p] / PTA_CHUNK, e = c + (s + PTA_CHUNK - 1) / PTA_CHUNK; c < e; c++)
            id = cminid[c] < id ? cminid[c] : id;
    t.tminid[v] = id;
    if (p == 0) {
        for (uint32_t m = 0; m < t.d; m++) {
            t.tmax[m * nn] = -INFINITY;
            t.tmin[m * nn] = INFINITY;
        }
        t.tsum[0] = -INFINITY;
        t.tminsum[0] = 0.0f;
        t.tminid[0] = 0xFFFFFFFFu;
    }
}

// Nodes [v0, 2 * v0) from their children, then (one workgroup) the levels
// above them down to `last`.
__global__ __launch_bounds__(1024) void pta_tree_kernel(TreeOut t, uint32_t v0, uint32_t last) {
    const uint64_t nn = 2ull * t.p2;
    for (;; v0 >>= 1) {
        for (uint32_t v = v0 + blockIdx.x * 1024 + threadIdx.x; v < 2 * v0; v += gridDim.x * 1024) {
            const uint64_t a = 2ull * v, b = a + 1;
            const float sm = fmaxf(t.tsum[a], t.tsum[b]);
            const bool any = sm > -INFINITY;
            double ms = 0.0;
            for (uint32_t m = 0; m < t.d; m++) {
                t.tmax[m * nn + v] = fmaxf(t.tmax[m * nn + a], t.tmax[m * nn + b]);
                const float mn = fminf(t.tmin[m * nn + a], t.tmin[m * nn + b]);
                t.tmin[m * nn + v] = mn;
                ms += any ? (double)mn : 0.0;
            }
            t.tsum[v] = sm;
            t.tminsum[v] = any ? f32_round_down(ms) : 0.0f;
            t.tminid[v] = t.tminid[a] < t.tminid[b] ? t.tminid[a] : t.tminid[b];
        }
        if (v0 <= last) return;
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------
static double now_ms() {
    return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

// Forgets the layout; its memory goes too unless it is about to be rebuilt.
static void pta_forget(PtaLayout &P, bool keep_memory) {
    PtaLayout N;
    N.psize = P.psize;
    N.generation = P.generation + 1;
    N.h_report = P.h_report;
    N.cus = P.cus;
    hipFree(P.xbits);
    if (keep_memory) {
        N.arena = P.arena;
        N.arena_cap = P.arena_cap;
        N.pcols = P.pcols;
        N.pcols_cap = P.pcols_cap;
        N.scratch = P.scratch;
        N.scratch_cap = P.scratch_cap;
    } else {
        hipFree(P.arena);
        hipFree(P.pcols);
        hipFree(P.scratch);
    }
    P = N;
}

void pta_release(topk_ctx *ctx) {
    batch_quiesce(ctx);  // batches in flight read the layout
    pta_forget(ctx->pta, false);
}

// The same before a rebuild: the memory stays for it.
void pta_stale(topk_ctx *ctx) {
    batch_quiesce(ctx);
    pta_forget(ctx->pta, true);
}

// Gives back the scratch a build left for the next one.
void pta_trim(topk_ctx *ctx) {
    hipFree(ctx->pta.scratch);
    ctx->pta.scratch = nullptr;
    ctx->pta.scratch_cap = 0;
}

// Room for `need` bytes at p (cap bytes so far), whose contents may go.
static int pta_room(unsigned char *&p, size_t &cap, size_t need) {
    if (need <= cap) return TOPK_OK;
    hipFree(p);
    p = nullptr;
    cap = 0;
    if (hipMalloc(&p, need) != hipSuccess) {
        (void)hipGetLastError();
        p = nullptr;
        return TOPK_ERR_NOMEM;
    }
    cap = need;
    return TOPK_OK;
}

namespace {

// Hands out 256-byte aligned pieces of one allocation; measures when base is null.
struct Carve {
    unsigned char *base = nullptr;
    size_t at = 0;
    template <class T>
    void take(T *&p, size_t count) {
        at = (at + 255) & ~(size_t)255;
        p = base ? reinterpret_cast<T *>(base + at) : nullptr;
        at += sizeof(T) * count;
    }
};

// The levels of the tree over ns sample rows and L leaves: the segments that
// take a device-wide level (with their workgroups' shares), and the subtrees
// one workgroup builds.
struct KdPlan {
    std::vector<KdSeg> segs, subs;
    std::vector<KdShare> shares;
    struct Level {
        uint32_t seg0, nseg, share0, nshare;
        bool carry;  // subtrees dealt out already: their rows move along
    };
    std::vector<Level> levels;
    uint32_t max_seg = 0, max_share = 0;

    KdPlan(uint32_t ns, uint32_t L) {
        std::vector<KdSeg> cur{KdSeg{0, ns, 0, L}}, next;
        while (!cur.empty()) {
            Level lv{(uint32_t)segs.size(), 0, (uint32_t)shares.size(), 0, false};
            next.clear();
            for (const KdSeg &s : cur) {
                if (s.nl < 2) continue;
                if (s.hi - s.lo <= KD_SUB && s.nl <= KD_SUB_LEAVES) {
                    subs.push_back(s);
                    continue;
                }
                const uint32_t first = lv.nshare;
                for (uint32_t b = s.lo; b < s.hi; b += KD_SHARE, lv.nshare++)
                    shares.push_back(KdShare{lv.nseg, b, std::min(s.hi, b + KD_SHARE), first});
                segs.push_back(s);
                lv.nseg++;
                const uint32_t nl = s.nleft(), mid = s.mid();
                next.push_back(KdSeg{s.lo, mid, s.leaf_lo, nl});
                next.push_back(KdSeg{mid, s.hi, s.leaf_lo + nl, s.nl - nl});
            }
            lv.carry = !subs.empty();
            if (lv.nseg) levels.push_back(lv);
            max_seg = std::max(max_seg, lv.nseg);
            max_share = std::max(max_share, lv.nshare);
            cur.swap(next);
        }
    }
};

}  // namespace

// Enqueues the tree over the sample; idx holds 0 .. ns-1 on entry.
static int kd_enqueue(const KdPlan &plan, hipStream_t s, const KdSeg *d_segs, const KdShare *d_shares,
                      const KdSeg *d_subs, uint32_t *idx, uint32_t *idx2, uint32_t *val, KdState *states, uint2 *cnt,
                      const float *rows, uint32_t d, uint32_t dp, KdNode *nodes) {
    for (size_t l = 0; l < plan.levels.size(); l++) {
        const KdPlan::Level &lv = plan.levels[l];
        const KdSeg *sg = d_segs + lv.seg0;
        const KdShare *sh = d_shares + lv.share0;
        TK_HIP(hipMemsetAsync(states, 0, sizeof(KdState) * lv.nseg, s));
        const dim3 g(lv.nshare), b(KD_BS);
        hipLaunchKernelGGL(kd_extremes_kernel, g, b, 0, s, sh, idx, rows, d, dp, states);
        hipLaunchKernelGGL(kd_hist_kernel<0>, g, b, 0, s, sh, sg, idx, rows, d, dp, val, states);
        hipLaunchKernelGGL(kd_hist_kernel<1>, g, b, 0, s, sh, sg, idx, rows, d, dp, val, states);
        hipLaunchKernelGGL(kd_hist_kernel<2>, g, b, 0, s, sh, sg, idx, rows, d, dp, val, states);
        hipLaunchKernelGGL(kd_count_kernel, g, b, 0, s, sh, sg, d, val, states, cnt, nodes);
        if (lv.carry) TK_HIP(hipMemcpyAsync(idx2, idx, sizeof(uint32_t) * plan.segs[0].hi, hipMemcpyDeviceToDevice, s));
        hipLaunchKernelGGL(kd_split_kernel, g, b, 0, s, sh, sg, idx, val, states, cnt, idx2);
        std::swap(idx, idx2);
    }
    if (!plan.subs.empty())
        hipLaunchKernelGGL(kd_subtree_kernel, dim3((uint32_t)plan.subs.size()), dim3(1024), 0, s, d_subs, idx, rows, d,
                           dp, nodes);
    TK_HIP(hipGetLastError());
    return TOPK_OK;
}

// A rebuild reuses the memory of the layout it replaces, and the scratch of
// the build before if that is at most PTA_KEEP_SCRATCH: device memory freed
// and allocated again at the pace of the build (1.5 GB in 3 ms) ends in the
// driver's clearing of freed pages, which stalled builds for up to seconds.  An
// allocation of the context that finds no room takes the scratch back
// (ctx_malloc).
constexpr size_t PTA_KEEP_SCRATCH = 4ull << 30;

int pta_build(topk_ctx *ctx) {
    const double t0 = now_ms();
    PtaLayout &P = ctx->pta;
    pta_stale(ctx);
    const uint64_t n = ctx->n;
    const uint32_t d = ctx->d, dp = (d + 3) & ~3u;
    hipStream_t s = ctx->stream;
    if (n >= ID_LIMIT) return TOPK_ERR_UNSUPPORTED;  // positions and partition ids are 32-bit
    const uint64_t want = (n + P.psize - 1) / P.psize;
    const uint32_t L = (uint32_t)(want < PTA_MAX_PARTS ? want : PTA_MAX_PARTS);
    uint64_t ns = (uint64_t)L * 64;
    if (ns < (1u << 20)) ns = 1u << 20;
    if (ns > n) ns = n;
    const KdPlan plan((uint32_t)ns, L);
    if (!P.cus) TK_HIP(hipDeviceGetAttribute(&P.cus, hipDeviceAttributeMultiprocessorCount, ctx->device));
    if (P.cus < 1) P.cus = 1;
    if (!P.h_report) TK_HIP(hipHostMalloc(&P.h_report, sizeof(uint32_t) * 4, hipHostMallocDefault));

    // assign: as many workgroups as are resident at once.  Beside the
    // attribute values LDS holds the leaf counters, else every object takes a
    // global atomic (past 2^15 leaves a workgroup meets most of its leaves
    // once, and counting would save nothing), and the tree if that fits too.
    constexpr size_t LDS_MAX = 150u * 1024;
    AssignArgs as{};
    size_t lds = sizeof(float) * d * PA_BS;
    const bool counted = lds + sizeof(uint32_t) * L <= LDS_MAX;
    if (counted) lds += sizeof(uint32_t) * L;
    as.tree_lds = lds + (sizeof(float) + 1) * L <= LDS_MAX ? 1 : 0;
    if (as.tree_lds) lds += (sizeof(float) + 1) * L;
    const uint32_t groups =
        (uint32_t)std::min<uint64_t>((n + PA_BS - 1) / PA_BS, (uint64_t)P.cus * (lds <= 78u * 1024 ? 2 : 1));
    as.cols = ctx->cols;
    as.ld = ctx->ld;
    as.n = n;
    as.per = (n + groups - 1) / groups;
    as.d = d;
    as.dp = dp;
    as.L = L;

    // the layout's own arrays, for npos positions (before they are counted: the
    // most padding)
    uint64_t npos_room = (n + (uint64_t)(PART_ALIGN - 1) * L + 8191) / 8192 * 8192;
    uint32_t p2 = 1;
    while (p2 < L) p2 <<= 1;
    const size_t nn = 2 * (size_t)p2;
    P.crow = 2 * d + 2;
    auto own = [&](unsigned char *p) {
        const size_t nchunks = npos_room / PTA_CHUNK;
        Carve c;
        c.base = p;
        c.take(P.pid, npos_room);
        c.take(P.cstat, nchunks * P.crow);
        c.take(P.cminid, nchunks);
        c.take(P.poff, L + 1);
        c.take(P.psz, L);
        c.take(P.pmax, (size_t)L * d);
        c.take(P.pmin, (size_t)L * d);
        c.take(P.psum, L);
        c.take(P.pminsum, L);
        c.take(P.pbound, L);
        c.take(P.bmax, (L + 255) / 256);
        c.take(P.pcut, L + 64);  // by group: R L/R rounded up
        c.take(P.wchunks, PTA_CUT_GROUPS);
        c.take(P.wstat, PTA_CUT_GROUPS);
        c.take(P.tmax, nn * d);
        c.take(P.tmin, nn * d);
        c.take(P.tsum, nn);
        c.take(P.tminsum, nn);
        c.take(P.tminid, nn);
        return c.at;
    };
    auto room = [&]() {
        int rc = pta_room(P.arena, P.arena_cap, own(nullptr));
        unsigned char *pc = reinterpret_cast<unsigned char *>(P.pcols);
        if (!rc) rc = pta_room(pc, P.pcols_cap, sizeof(float) * (npos_room * d + 8192));
        P.pcols = reinterpret_cast<float *>(pc);
        if (!rc) own(P.arena);
        return rc;
    };
    // scratch of the build in one piece.  The rows in object order may lie in
    // the columns' memory, which is written after their last use; without
    // room for the scattered rows the columns are gathered by id instead, and
    // without room for anything per object (24 bytes of it) the tree is walked
    // twice, the arrays are sized after the first walk has counted, and the
    // columns are read once more for the sums: no more memory at any time than
    // the store, the layout and the sample.
    const bool rows_in_pcols = n * dp <= npos_room * d + 8192;
    float *rows = nullptr, *own_rows = nullptr, *srows = nullptr;
    uint32_t *idx = nullptr, *idx2 = nullptr, *val = nullptr, *off = nullptr, *sz = nullptr;
    KdState *states = nullptr;
    uint2 *share_cnt = nullptr;
    KdNode *nodes = nullptr;
    KdSeg *segs = nullptr, *subs = nullptr;
    KdShare *shares = nullptr;
    uint64_t *keys = nullptr;
    bool with_rows = true, lean = ctx->tune.init_lean != 0;
    auto carve = [&](unsigned char *p) {
        Carve c;
        c.base = p;
        c.take(rows, ns * dp);
        c.take(idx, ns);
        c.take(idx2, ns);
        c.take(val, ns);
        c.take(states, plan.max_seg);
        c.take(share_cnt, plan.max_share);
        c.take(segs, plan.segs.size());
        c.take(shares, plan.shares.size());
        c.take(subs, plan.subs.size());
        c.take(nodes, L);
        c.take(as.cnt, L);
        c.take(off, lean ? L + 1 : 0);
        c.take(sz, lean ? L : 0);
        c.take(as.place, lean ? 0 : n);
        c.take(as.base, counted && !lean ? (size_t)groups * L : 0);
        c.take(as.order, counted && !lean ? n : 0);
        c.take(keys, lean ? 0 : npos_room);
        c.take(own_rows, with_rows && counted && !lean && !rows_in_pcols ? n * dp : 0);
        c.take(srows, with_rows && !lean ? npos_room * dp : 0);
        return c.at;
    };
    int rc = lean ? TOPK_ERR_NOMEM : room();
    if (!rc && pta_room(P.scratch, P.scratch_cap, carve(nullptr))) {
        with_rows = false;
        rc = pta_room(P.scratch, P.scratch_cap, carve(nullptr));
    }
    if (rc) {
        pta_forget(P, false);
        P.crow = 2 * d + 2;
        lean = true;
        with_rows = false;
        rc = pta_room(P.scratch, P.scratch_cap, carve(nullptr));
    }
    if (rc) {
        pta_forget(P, false);
        return rc;
    }
    carve(P.scratch);
    if (!counted || lean) {
        as.base = nullptr;
        as.order = nullptr;
    }
    if (lean) as.place = nullptr;
    as.nodes = nodes;
    as.rows = !with_rows || !counted ? nullptr : (rows_in_pcols ? P.pcols : own_rows);
#define TK_TRY(call)                                              \
    do {                                                          \
        hipError_t e_ = (call);                                   \
        if (e_ != hipSuccess) { rc = hip_status(e_); goto fail; } \
    } while (0)
    {
        // 1, 2: sample and tree
        if (!plan.segs.empty()) {
            TK_TRY(hipMemcpyAsync(segs, plan.segs.data(), sizeof(KdSeg) * plan.segs.size(), hipMemcpyHostToDevice, s));
            TK_TRY(hipMemcpyAsync(shares, plan.shares.data(), sizeof(KdShare) * plan.shares.size(),
                                  hipMemcpyHostToDevice, s));
        }
        if (!plan.subs.empty())
            TK_TRY(hipMemcpyAsync(subs, plan.subs.data(), sizeof(KdSeg) * plan.subs.size(), hipMemcpyHostToDevice, s));
        hipLaunchKernelGGL(kd_sample_kernel, dim3((uint32_t)((ns + 255) / 256)), dim3(256), 0, s, ctx->cols, ctx->ld,
                           d, dp, n, ns, rows, idx);
        rc = kd_enqueue(plan, s, segs, shares, subs, idx, idx2, val, states, share_cnt, rows, d, dp, nodes);
        if (rc) goto fail;
        // 3: leaves
        TK_TRY(hipMemsetAsync(as.cnt, 0, sizeof(uint32_t) * L, s));
        hipLaunchKernelGGL(pta_assign_kernel, dim3(groups), dim3(PA_BS), lds, s, as);
        hipLaunchKernelGGL(pta_offsets_kernel, dim3(1), dim3(1024), 0, s, as.cnt, L, lean ? off : P.poff,
                           lean ? sz : P.psz, P.h_report);
        TK_TRY(hipGetLastError());
        TK_TRY(hipStreamSynchronize(s));
        const uint64_t npos = *reinterpret_cast<volatile uint64_t *>(P.h_report);
        P.nonempty = reinterpret_cast<volatile uint32_t *>(P.h_report)[2];
        P.maxsz = reinterpret_cast<volatile uint32_t *>(P.h_report)[3];
        if (npos >= 0xFFFFFFFFull) { rc = TOPK_ERR_UNSUPPORTED; goto fail; }
        P.nparts = L;
        P.npos = npos;
        P.ld = (npos + 8191) / 8192 * 8192;
        P.nchunks = npos / PTA_CHUNK;
        P.p2 = p2;
        if (lean) {
            npos_room = P.ld;
            rc = room();
            if (rc) goto fail;
            TK_TRY(hipMemcpyAsync(P.poff, off, sizeof(uint32_t) * (L + 1), hipMemcpyDeviceToDevice, s));
            TK_TRY(hipMemcpyAsync(P.psz, sz, sizeof(uint32_t) * L, hipMemcpyDeviceToDevice, s));
        }
        // 4, 5: objects to their partitions, the partitions in order
        const bool fused = with_rows && P.maxsz <= PTA_SORT_MAX;
        if (!fused && !lean) TK_TRY(hipMemsetAsync(keys, 0, sizeof(uint64_t) * P.ld, s));
        if (P.maxsz > PTA_SORT_MAX && as.base) {
            hipLaunchKernelGGL(pta_recount_kernel, dim3(groups), dim3(PA_BS), sizeof(uint32_t) * L, s, as);
            hipLaunchKernelGGL(pta_base_kernel, dim3((L + 255) / 256), dim3(256), 0, s, as.base, L, groups);
            as.order = nullptr;
        }
        if (lean) {
            TK_TRY(hipMemsetAsync(as.cnt, 0, sizeof(uint32_t) * L, s));
            TK_TRY(hipMemsetAsync(P.pid, 0xFF, sizeof(uint32_t) * P.ld, s));
            as.poff = P.poff;
            as.pid = P.pid;
            hipLaunchKernelGGL(pta_assign_kernel, dim3(groups), dim3(PA_BS), lds, s, as);
        } else {
            hipLaunchKernelGGL(pta_scatter_kernel, dim3((uint32_t)std::min<uint64_t>(16, (as.per + 255) / 256), groups),
                               dim3(256), 0, s, as, P.poff, keys, fused ? srows : (float *)nullptr);
        }
        if (fused) {
            const uint32_t cap = (std::max(P.maxsz, 1u) + 255) / 256 * 256;
            const PartOut po{P.pcols, P.ld, P.pid, P.nchunks, P.cstat, P.cminid, P.pmax, P.pmin, P.psum, P.pminsum};
            hipLaunchKernelGGL(pta_part_kernel, dim3(L), dim3(PP_BS), (sizeof(uint64_t) + sizeof(uint16_t)) * cap, s,
                               keys, srows, d, dp, P.poff, P.psz, cap, po);
            hipLaunchKernelGGL(pta_tail_kernel, dim3(32), dim3(256), 0, s, P.npos, P.ld, d, P.pcols, P.pid);
        } else {
            if (lean)
                hipLaunchKernelGGL(pta_sort_ids_kernel, dim3(L), dim3(1024), 0, s, ctx->cols, ctx->ld, d, P.poff, P.psz,
                                   P.pid);
            else hipLaunchKernelGGL(pta_sort_kernel, dim3(L), dim3(1024), 0, s, P.poff, P.psz, keys);
            TK_TRY(hipMemsetAsync(P.pcols + P.ld * d, 0, sizeof(float) * 8192, s));
            hipLaunchKernelGGL(pta_gather_kernel, dim3((uint32_t)((P.ld + 255) / 256)), dim3(256), 0, s, ctx->cols,
                               ctx->ld, d, P.ld, lean ? (const uint64_t *)nullptr : keys, P.pcols, P.ld, P.pid);
            hipLaunchKernelGGL(pta_bounds_kernel, dim3(L), dim3(PB_BS), 0, s, P.pcols, P.ld, d, P.poff, P.psz, P.pmax,
                               P.pmin, P.psum, P.pminsum);
            if (P.nchunks) {
                hipLaunchKernelGGL(pta_chunk_kernel, dim3((uint32_t)((P.nchunks + 3) / 4)), dim3(256), 0, s, P.pcols,
                                   P.ld, d, P.pid, (uint64_t)P.nchunks, P.cstat, P.cminid);
                hipLaunchKernelGGL(pta_chunk_suffix_kernel, dim3((L + 255) / 256), dim3(256), 0, s, L, d, P.poff,
                                   P.psz, (uint64_t)P.nchunks, P.cstat);
            }
        }
        // 6: bound tree
        const TreeOut to{p2, L, d, P.tmax, P.tmin, P.tsum, P.tminsum, P.tminid};
        hipLaunchKernelGGL(pta_tree_leaf_kernel, dim3((p2 + 255) / 256), dim3(256), 0, s, to, P.poff, P.psz, P.pmax,
                           P.pmin, P.psum, P.pminsum, P.cminid);
        uint32_t v0 = p2 / 2;
        for (; v0 > 1024; v0 /= 2)
            hipLaunchKernelGGL(pta_tree_kernel, dim3(std::min(v0 / 1024, 256u)), dim3(1024), 0, s, to, v0, v0);
        if (v0) hipLaunchKernelGGL(pta_tree_kernel, dim3(1), dim3(1024), 0, s, to, v0, 1u);
        TK_TRY(hipGetLastError());
        TK_TRY(hipStreamSynchronize(s));
    }
#undef TK_TRY
    if (lean || P.scratch_cap > PTA_KEEP_SCRATCH) pta_trim(ctx);
    P.built = true;
    P.tt_build_ms = now_ms() - t0;
    return TOPK_OK;
fail:
    hipStreamSynchronize(s);  // kernels of the build may still use its memory
    pta_forget(P, false);
    return rc;
}

// ---------------------------------------------------------------------------
// extreme-value bitmaps
// ---------------------------------------------------------------------------
// One wave per (row, word): lane i reads object 64 w + i of the attribute
// and the ballot of "equals the store's largest / smallest value" is the word.
__global__ __launch_bounds__(256) void extreme_bits_kernel(const float *__restrict__ cols, uint64_t ld, uint64_t n,
                                                           uint32_t d, const float *__restrict__ rmax,
                                                           const float *__restrict__ rmin, uint64_t rstride,
                                                           uint64_t nw, uint64_t *__restrict__ bits) {
    const uint32_t lane = lane_id();
    const uint64_t nwaves = (uint64_t)gridDim.x * 4;
    for (uint64_t v = (uint64_t)blockIdx.x * 4 + threadIdx.x / 64; v < (uint64_t)d * nw; v += nwaves) {
        const uint32_t a = (uint32_t)(v / nw);
        const uint64_t w = v - (uint64_t)a * nw, id = 64 * w + lane;
        const float x = id < n ? cols[(uint64_t)a * ld + id] : 0.0f;
        const uint64_t hi = __ballot(id < n && x == rmax[a * rstride]);
        const uint64_t lo = __ballot(id < n && x == rmin[a * rstride]);
        if (lane == 0) {
            bits[(uint64_t)a * nw + w] = hi;
            bits[(uint64_t)(d + a) * nw + w] = lo;
        }
    }
}

int pta_extreme_bits(topk_ctx *ctx) {
    PtaLayout &P = ctx->pta;
    if (!P.built) return TOPK_ERR_STATE;
    if (P.xbits) return TOPK_OK;
    const uint64_t nw = ((ctx->n + 63) / 64 + 15) & ~15ull;  // padding words hold ids >= n: zero
    TK_HIP(ctx_malloc(ctx, &P.xbits, sizeof(uint64_t) * 2 * ctx->d * nw));
    P.nw = nw;
    const uint64_t waves = (uint64_t)ctx->d * nw;
    const uint32_t grid = (uint32_t)std::min<uint64_t>((waves + 3) / 4, 65536);
    hipLaunchKernelGGL(extreme_bits_kernel, dim3(grid), dim3(256), 0, ctx->stream, ctx->cols, ctx->ld, ctx->n, ctx->d,
                       P.tmax + 1, P.tmin + 1, 2 * (uint64_t)P.p2, nw, P.xbits);
    TK_HIP(hipGetLastError());
    TK_HIP(hipStreamSynchronize(ctx->stream));
    return TOPK_OK;
}

}  // namespace topk
