// Launch plans of the plain query (fte.hip): the threshold's source and rank,
// the stream's tiles and the slots of its candidates.  Host arithmetic only,
// so that a CPU program can check how far a plan reads and writes; tile_vec
// is the one the kernels use.
#pragma once

#include <algorithm>
#include <cmath>

#include "keys.hpp"

namespace topk {

// FTE pipeline modes: sample-seeded (the caller re-runs a bad guess),
// exact-prefix-seeded with the regular candidate buffer, exact with an
// n-entry buffer, and queued: sample-seeded above 2^19 objects, exact below
// (nothing re-runs it).
enum { FTE_SAMPLE = 0, FTE_EXACT = 1, FTE_EXACT_BIG = 2, FTE_QUEUED = 3 };

constexpr uint32_t MAX_STREAM_GRID = 4096;
constexpr uint32_t STREAM_BS = 1024;                        // threads of a stream workgroup
constexpr uint32_t STREAM_GRID = 256;                       // stream workgroups at most (one per CU), unless tuned
constexpr uint32_t FUSE_CAP_MIN = 1024, FUSE_CAP_MAX = 4096;  // candidates the last stream workgroup selects in LDS

constexpr uint32_t SEED_TILE = 4096;     // exact mode: objects per seed block (16 per thread)
constexpr uint32_t SAMPLE_TILE = 1024;   // shared sample: objects per chunk
constexpr uint32_t SAMPLE_CHUNKS = 128;  // shared sample: chunks at most, spread over the ids
constexpr uint32_t SAMPLE_WGS = 32;      // shared sample: pieces, each a workgroup's
constexpr uint32_t SAMPLE_WIN = 1024;    // shared sample: winners of all pieces at most
constexpr uint32_t SAMPLE_MAX_W = SAMPLE_WIN / SAMPLE_WGS;  // winners of a piece at most
constexpr uint32_t SAMPLE_POLLS = 32;    // tries before a workgroup takes a missing piece of the sample
constexpr int SAMPLE_VEC = SAMPLE_CHUNKS * SAMPLE_TILE / (SAMPLE_WGS * STREAM_BS * 4);  // float4 per thread
constexpr int OWN_VEC = 4096 / (STREAM_BS * 4);  // own sample: float4 vectors per thread
constexpr uint32_t OWN_OBJS = STREAM_BS * 4 * OWN_VEC;
constexpr uint32_t OWN_SPOTS = OWN_OBJS / 16;   // own sample: 256 runs of 16 objects, one 64-byte line per column each
constexpr uint32_t OWN_MAX_W = 32;              // own sample: keys of a wave at most
constexpr uint64_t OWN_MAX_N = 1ull << 19;      // stores up to this size take their own sample

// A column of n objects is readable to its n-th value rounded up to 16
// bytes, and PAD_REACH values on; the exact seed's whole tiles read that far.
constexpr uint32_t PAD_REACH = 8191;
static_assert(SEED_TILE - 1 <= PAD_REACH, "a seed tile ends inside the padding");

// float4 vector a lane of a stream tile reads: tiles are longer than the
// padding, so what lies past the store's last vector reads that one instead
// (its ids say that it is no object).
TK_HD uint32_t tile_vec(uint32_t v, uint32_t last) { return v < last ? v : last; }

// A run with an n-entry buffer takes tiles of at most BIG_TILE objects: its
// slots hold a workgroup's every object, and hold no more than the rounding
// of ensure_big's buffer allows.
constexpr uint32_t BIG_TILE = 8192;
static inline uint64_t big_slots(uint64_t n) { return n + (uint64_t)MAX_STREAM_GRID * BIG_TILE; }

static inline uint32_t exact_prefix_blocks(uint64_t n, uint32_t k) {
    const uint64_t need = (n + SEED_TILE - 1) / SEED_TILE;
    uint32_t g = 32768u / (k ? k : 1);
    if (g > 256) g = 256;
    if (g < 8) g = 8;
    return (uint32_t)(need < g ? need : g);
}

static inline uint32_t stream_grid(uint32_t grid_cap, uint64_t ntiles) {
    const uint64_t cap = grid_cap ? (uint64_t)grid_cap : STREAM_GRID;
    const uint64_t g = ntiles < cap ? ntiles : cap;
    return (uint32_t)(g < 1 ? 1 : g);
}

// float4 vectors per lane per column of one stream tile: enough loads in
// flight per lane (about 8-16) without exhausting registers.
static inline int stream_vpt(uint32_t m) {
    if (m <= 1) return 8;
    if (m <= 2) return 4;
    if (m <= 4) return 2;
    return 1;
}

// Columns the stream kernel is unrolled for, its first tile's loads all in
// flight while tau is found; 0: the runtime width, eight loads a lane at a
// time.  16 waves a workgroup leave a lane 128 registers, and past 12 loads
// of 16 bytes they spill.  2^25 objects, k = 64, unrolled and runtime width,
// alone / queued: 9 columns 220 / 186 and 216 / 183 us, 12: 271 / 243 and 271
// / 244, 13: 308 / 270 and 295 / 267, 16: 380 / 342 and 355 / 327; 2^22: 9:
// 61 / 39 and 64 / 42, 12: 69 / 47 and 71 / 50, 13: 78 / 54 and 74 / 53, 16:
// 91 / 65 and 83 / 62.
constexpr int stream_unroll(int m, int vpt) { return m * vpt <= 12 ? m : 0; }

// Samples above the ks-th largest of a random sample of s of the n objects
// leave ks * n / s candidates on average, spread like a Gamma(ks) variable.
// The smallest ks that leaves fewer than k with a chance of about 1e-4, from
// q = k * s / n (the expected number of the top k in the sample): ks - 3.7
// sqrt(ks) + 3.6 >= q, e.g. 17 k candidates at ks = 4, 5 k at 8, 2 k at 32.
static inline uint32_t sample_rank(double q) {
    uint32_t ks = 4;
    while (ks < 4096 && ks - 3.7 * std::sqrt((double)ks) + 3.6 < q) ks++;
    return ks;
}

// The same for a query nothing re-runs: fewer than k means that ks of the
// top k fell into the sample, for about Poisson(q) of them less often than
// exp(-q) (e q / ks)^ks (Chernoff, ten times the truth): here 1e-8, and 1e-5
// below q = 1, where every rank adds candidates the most (32 queries of 16M x
// 5, k = 32, q = 0.25: rank 4, 1e-4, 1797 us; rank 6 1820; rank 8 1872).
//
// These chances are for scores that do not depend on the id.  Stores in
// score order, or with their best objects side by side, put whole runs of the
// top k into one chunk: the rank leaves 8 k candidates at least, and k, a proven
// bound, where that takes one (up to 2^20 objects).
static inline uint32_t queued_rank(double q, uint32_t k) {
    const double rare = q < 1.0 ? 11.5 : 18.4;
    uint32_t ks = std::max(4u, (uint32_t)std::min(std::ceil(8.0 * q), 4096.0));
    while (ks < 4096 && (ks <= q || ks * (std::log(ks / q) - 1.0) + q < rare)) ks++;
    return std::min(ks, std::max(k, 4u));
}

// Keys a piece of the shared sample publishes.  Up to 2^20 objects half of a
// rank below k, so that tau lies below the best of at least two pieces: of a
// store in score order one piece holds the whole top ks, and with all of them
// published ks objects would reach tau instead of k (2^20 objects, k = 10: a
// second, exact run, 100 us in all instead of 63).  Larger stores take that
// run, as they always did.  From a rank of 16 on a piece's share, with room: a
// piece that holds more lowers tau.
static inline uint32_t piece_winners(uint32_t ks, uint32_t k, uint64_t n) {
    const uint32_t w = ks < k && n <= 1ull << 20 ? (ks + 1) / 2 : ks;
    return w < 16 ? w : (ks <= 256 ? 16u : SAMPLE_MAX_W);
}

// Keys a wave of the own sample contributes: half, for the same reason (2^19
// objects, k = 64: 100 us in two runs, 40 in one; the exact run alone took
// 80), which also halves its rounds (16k objects, k = 10: 35.4 -> 33.8 us).
static inline uint32_t wave_winners(uint32_t ks) { return std::min({(ks + 1) / 2, 8 + ks / 4, OWN_MAX_W}); }

// Where a stream workgroup takes tau from: every object is a candidate,
// st->tau, the shared sample, the own sample.
enum { TAU_ALL = 0, TAU_STATE = 1, TAU_SHARED = 2, TAU_OWN = 3 };

// How a query gets its threshold.
struct SeedPlan {
    int tau;               // TAU_*
    uint32_t blocks, ks;   // chunks of the sample or blocks of the exact seed; rank of tau (exact: winners per block)
    uint32_t W;            // winners per piece of the shared sample, or per wave of the own one
    uint64_t stride;       // objects between the chunks' first objects
    uint64_t n_eff;        // exact: objects of the prefix
    uint64_t first;        // first object to stream: n_eff where the seed hands on the prefix's top k
    uint32_t total_valid;  // exact: keys the blocks deposit
    double expect;         // candidates expected
};

// FTE_SAMPLE may guess on any store (the caller re-runs a bad guess): every
// object of a store that fits the select, the own sample up to 2^19 objects,
// the shared sample above.  FTE_QUEUED guesses only above 2^19 objects:
// nothing re-runs it; below, tau is the k-th key of the exact prefix.
static inline SeedPlan seed_plan(uint64_t n, uint32_t k, int mode) {
    SeedPlan p{};
    if (mode == FTE_SAMPLE && n <= FUSE_CAP_MAX) {
        p.tau = TAU_ALL;
        p.expect = (double)n;
    } else if (mode == FTE_SAMPLE && n <= OWN_MAX_N) {
        p.tau = TAU_OWN;
        p.ks = sample_rank((double)k * OWN_OBJS / (double)n);
        p.W = wave_winners(p.ks);
        p.expect = (double)p.ks * n / OWN_OBJS;
        if (p.expect >= n) p.tau = TAU_ALL;
    } else if ((mode == FTE_SAMPLE || mode == FTE_QUEUED) && n > OWN_MAX_N) {
        p.tau = TAU_SHARED;
        // As many chunks as make tau the 8th largest of the sample (q =
        // 1.13).  A long list on a small store would leave few of them, large
        // jumps of the id range: below 32 chunks, all 128 and a deeper rank.
        // Queued: all 128.
        const uint64_t c8 = (uint64_t)(1.13 * (double)n / ((double)k * SAMPLE_TILE));
        p.blocks = mode == FTE_SAMPLE && c8 >= SAMPLE_CHUNKS / 4 && c8 < SAMPLE_CHUNKS ? (uint32_t)c8 : SAMPLE_CHUNKS;
        p.stride = (n / p.blocks) & ~15ull;  // a line; the chunks reach to the end of the store
        const double s = (double)p.blocks * SAMPLE_TILE;
        p.ks = mode == FTE_QUEUED ? queued_rank(k * s / (double)n, k) : sample_rank(k * s / (double)n);
        p.W = piece_winners(p.ks, k, n);
        p.expect = (double)p.ks * n / s;
    } else {
        p.tau = TAU_STATE;
        p.blocks = exact_prefix_blocks(n, k);
        p.stride = SEED_TILE;
        const uint64_t pre = (uint64_t)p.blocks * SEED_TILE;
        p.n_eff = n < pre ? n : pre;
        // Queued: past 4096 seed winners or k = 256 the prefix is streamed
        // again, with the select in the last stream workgroup, instead of
        // listed by the seed's last workgroup (a search of all winners) and
        // selected by a launch of its own.  Listed / streamed, us a query:
        // 100,000 objects (25 blocks), k = 16 17.6 / 20.6, 100 21.6 / 23.2, 400
        // 37.7 / 32.5, 1000 70.6 / 45.3; 2^19 (128 blocks), k = 16 29.6 / 34.7,
        // 100 42.6 / 39.8; 5000, k = 1000 36.8 / 24.6.
        p.first = mode != FTE_QUEUED || (k <= 256 && p.blocks * k <= 4096) ? p.n_eff : 0;
        p.ks = k;
        const uint64_t full = p.n_eff / SEED_TILE, rem = p.n_eff % SEED_TILE;
        p.total_valid = (uint32_t)(full * (k < SEED_TILE ? k : SEED_TILE) + (rem < k ? rem : k));
        p.expect = 2.0 * k;
    }
    return p;
}

// The stream pass over objects [first, n).
struct StreamPlan {
    int vpt;
    uint64_t tile, ntiles;  // objects per tile
    uint64_t nstatic;       // tiles dealt out in turn; the rest as workgroups get free
    uint32_t grid;          // 0: nothing to stream
    uint32_t slot;          // candidate slots per workgroup
};

// vpt and grid_cap as tuned (0: chosen here); cand_cap: entries of the
// candidate buffer; big: of at least big_slots(n) entries, a block's every
// object fits its slots.
static inline StreamPlan stream_plan(uint64_t n, uint64_t first, uint32_t m, bool big, int vpt, uint32_t grid_cap,
                                     uint64_t cand_cap) {
    StreamPlan p{};
    p.vpt = vpt ? vpt : stream_vpt(m);
    // smaller tiles where the wide ones would leave workgroups without one
    while (!vpt && p.vpt > 1 && n - first < (uint64_t)STREAM_GRID * STREAM_BS * 4 * p.vpt) p.vpt /= 2;
    if (big) p.vpt = std::min<int>(p.vpt, BIG_TILE / (STREAM_BS * 4));
    p.tile = (uint64_t)STREAM_BS * 4 * p.vpt;
    p.ntiles = n > first ? (n - first + p.tile - 1) / p.tile : 0;
    p.grid = p.ntiles ? stream_grid(grid_cap, p.ntiles) : 0;
    // The last sixth of the tiles by ticket, at least two a workgroup, four
    // where a tile lasts longer (above 8 columns): with a twelfth and two, a
    // workgroup that the query before delays at its start (its last one
    // selects) ended late.  Queued queries, 2^25 objects: 12 columns 251 ->
    // 242 us, 8 columns 171 -> 164 (alone 202 -> 194); 2^24 x 12: 130 with
    // two, 125 with four, 2^24 x 5: 58.3 and 59.7.  Up to four tiles a
    // workgroup are all dealt (2^22 x 8: 37 -> 34 us), and so are those of a
    // run whose slots hold a block's every object.
    const uint64_t g = p.grid;
    p.nstatic = p.ntiles;
    if (!big && p.ntiles > 4 * g)
        p.nstatic = (p.ntiles - std::max<uint64_t>(p.ntiles / 6, (m > 8 ? 4ull : 2ull) * g) + g - 1) / g * g;
    if (g) p.slot = (uint32_t)(big ? (p.ntiles + g - 1) / g * p.tile : cand_cap / g);
    return p;
}

}  // namespace topk
