"""The plain query's launch plans (topk_amd/csrc/fte_plan.hpp) on the CPU:
how far the stream's tiles and the exact seed read a column, and what the
slots of an n-entry run take, over store sizes, widths, modes and the tuned
tile and grid -- the sizes around every tile, pad and plan limit."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HEADER = r"""
#include <cstdint>
#include <cstdio>
#include <initializer_list>
#include <vector>
#include "fte_plan.hpp"
using namespace topk;
static int fails = 0;
#define CHECK(c, ...) do { if (!(c)) { if (fails++ < 10) { std::printf("%s: ", #c); std::printf(__VA_ARGS__); std::printf("\n"); } } } while (0)
"""

REACH = HEADER + r"""
int main() {
    std::vector<uint64_t> sizes;
    for (uint64_t c : {1ull, 4096ull, 8192ull, 32768ull, 1ull << 19, 1ull << 20, 1ull << 21, 3000001ull, 1ull << 23,
                       8388609ull, 10000000ull, 150000000ull, 1ull << 28, (1ull << 32) - 8192})
        for (int64_t o : {-8191, -4097, -4095, -1, 0, 1, 4, 4095, 4097, 8191})
            if ((int64_t)c + o >= 1 && c + o < 0xFFFFFFFFull) sizes.push_back(c + o);
    for (uint64_t n : sizes)
        for (uint32_t m : {1u, 2u, 3u, 5u, 9u, 20u})
            for (uint32_t k : {1u, 200u, 1024u})
                for (int mode : {FTE_SAMPLE, FTE_EXACT, FTE_EXACT_BIG, FTE_QUEUED})
                    for (int vpt : {0, 1, 2, 4, 8})
                        for (uint32_t grid : {0u, 1u, 257u, MAX_STREAM_GRID}) {
                            const SeedPlan s = seed_plan(n, k, mode);
                            const uint64_t first = s.first, pad = (n + 3) / 4 * 4;
                            const bool big = mode == FTE_EXACT_BIG;
                            const StreamPlan p = stream_plan(n, first, m, big, vpt, grid, 1ull << 21);
                            // the stream: every object of [first, n), nothing past the column's last vector
                            CHECK(first == 0 || (s.tau == TAU_STATE && first == s.n_eff), "n %llu", (unsigned long long)n);
                            CHECK(first + p.ntiles * p.tile >= n && (!p.ntiles || first % 4 == 0), "n %llu", (unsigned long long)n);
                            const uint32_t last = (uint32_t)((n - 1) / 4);
                            uint64_t most = 0;
                            for (uint64_t t = p.ntiles > 2 ? p.ntiles - 2 : 0; t < p.ntiles; t++)
                                for (uint64_t v = 0; v < p.tile / 4; v += v + 1 < p.tile / 4 && v ? p.tile / 4 - 1 - v : 1)
                                    most = std::max<uint64_t>(most, 4ull * tile_vec((uint32_t)((first + t * p.tile) / 4 + v), last) + 4);
                            CHECK(most <= pad, "n %llu m %u k %u mode %d vpt %d: reads %llu", (unsigned long long)n, m, k,
                                  mode, vpt, (unsigned long long)most);
                            // samples and the exact seed
                            if (s.tau == TAU_STATE)
                                CHECK(((s.n_eff + SEED_TILE - 1) / SEED_TILE) * SEED_TILE <= n + PAD_REACH, "n %llu",
                                      (unsigned long long)n);
                            if (s.tau == TAU_SHARED)
                                CHECK((s.blocks - 1) * s.stride + SAMPLE_TILE <= n + SAMPLE_TILE - 1, "n %llu",
                                      (unsigned long long)n);
                            // slots: an n-entry run's hold every object of a workgroup's tiles, inside the buffer
                            if (big && p.grid) {
                                CHECK((uint64_t)p.slot >= (p.ntiles + p.grid - 1) / p.grid * p.tile, "n %llu",
                                      (unsigned long long)n);
                                CHECK((uint64_t)p.slot * p.grid <= big_slots(n), "n %llu m %u vpt %d grid %u",
                                      (unsigned long long)n, m, vpt, grid);
                            }
                            CHECK(p.grid <= MAX_STREAM_GRID && p.grid <= std::max<uint64_t>(p.ntiles, 1), "grid %u", p.grid);
                            CHECK(p.nstatic <= p.ntiles && (p.nstatic == p.ntiles || p.nstatic >= p.grid), "n %llu",
                                  (unsigned long long)n);
                        }
    return fails ? 1 : 0;
}
"""

RANKS = HEADER + r"""
int main() {
    // a query nothing re-runs: no threshold above the one that k-th, or 8 k candidates', rank of 128 x 1024
    // sampled objects gives
    for (uint64_t n : {(1ull << 19) + 1, 524289ull, 700001ull, 1ull << 20, (1ull << 20) + 1, 1500000ull, 1ull << 21, 3000001ull,
                       1ull << 23, 16777213ull, 1ull << 26, 1ull << 31})
        for (uint32_t k = 1; k <= 1024; k++) {
            const SeedPlan p = seed_plan(n, k, FTE_QUEUED);
            const uint64_t s = 128 * 1024, want = (8ull * k * s + n - 1) / n;
            const uint32_t floor_ = (uint32_t)(want < 4 ? 4 : (want > k ? k : want));
            CHECK(p.tau == TAU_SHARED && p.blocks == 128 && p.ks >= floor_ && p.ks <= SAMPLE_WGS * p.W && p.W <= SAMPLE_MAX_W,
                  "n %llu k %u: rank %u of %u, %u expected", (unsigned long long)n, k, p.ks, p.blocks, floor_);
            if (n <= 1ull << 20) CHECK(p.ks >= k, "n %llu k %u", (unsigned long long)n, k);
        }
    return fails ? 1 : 0;
}
"""

ORDERED = HEADER + r"""
// Candidates that reach tau in a store whose score falls with the id, from the plan alone: the sample's positions,
// W winners of each piece or wave, the ks-th best of them.
static uint64_t reach(const SeedPlan &p, uint64_t n) {
    std::vector<uint64_t> best;
    if (p.tau == TAU_SHARED) {
        for (uint32_t piece = 0; piece < SAMPLE_WGS; piece++)
            for (uint32_t w = 0, c = piece, i = 0; w < p.W && c < p.blocks; w++) {
                best.push_back(c * p.stride + i);
                if (++i == SAMPLE_TILE) c += SAMPLE_WGS, i = 0;
            }
    } else {
        const uint64_t lines = (n + 15) / 16;
        for (uint32_t wave = 0; wave < STREAM_BS / 64; wave++)
            for (uint32_t w = 0; w < p.W; w++) {
                const uint64_t spot = w / 16 * (STREAM_BS / 64) + wave, id = spot * lines / OWN_SPOTS * 16 + w % 16;
                if (id < n) best.push_back(id);
            }
    }
    std::sort(best.begin(), best.end());
    return best.size() < p.ks ? n : best[p.ks - 1] + 1;
}
int main() {
    for (uint64_t n : {4097ull, 16411ull, 65521ull, 131072ull, 300007ull, 1ull << 19, (1ull << 19) + 1, 700001ull, 1ull << 20})
        for (uint32_t k = 1; k <= 1024; k++) {
            const SeedPlan p = seed_plan(n, k, FTE_SAMPLE);
            if (p.tau == TAU_ALL) continue;
            const uint64_t c = reach(p, n);
            CHECK(c >= k, "n %llu k %u: rank %u, %u winners a piece, %llu candidates", (unsigned long long)n, k, p.ks, p.W,
                  (unsigned long long)c);
        }
    return fails ? 1 : 0;
}
"""


def _run(program, tmp_path):
    if not shutil.which("g++"):
        pytest.skip("no g++")
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text(program)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "topk_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout


def test_reads_and_slots_stay_inside_their_buffers(tmp_path):
    _run(REACH, tmp_path)


def test_queued_ranks_are_as_deep_as_a_proven_bound(tmp_path):
    _run(RANKS, tmp_path)


def test_stores_in_score_order_take_one_run(tmp_path):
    _run(ORDERED, tmp_path)
