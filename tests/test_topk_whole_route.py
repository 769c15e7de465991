"""Which lists go in one launch (csrc/topk_route.h, whole_tiles), compiled and checked on the CPU: never more select blocks
than may wait for each other, in a bucket as many as its counters are laid out for, and groups whose candidates fit."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "topk_route.h"
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>
using namespace mcclhip;
#define REQUIRE(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); std::exit(1); } } while (0)

static TopkCall list(const std::vector<uint64_t>& v, double ratio) {
    const uint64_t longest = *std::max_element(v.begin(), v.end());
    const uint32_t k = (uint32_t)(longest * ratio);
    return {longest * v.size(), longest, (uint32_t)v.size(), v.data(), k ? k : 1, topk_many(longest, ratio)};
}
static uint32_t shift_of(const TopkCall& c) { return c.many ? 8 : topk_group_shift_few(topk_tiles(c.bucket_elems)); }

int main() {
    std::mt19937 rng(1);
    int taken = 0;
    for (int i = 0; i < 20000; i++) {
        const double ratios[] = {0.001, 0.01, 0.02, 0.05, 0.12};
        const double ratio = ratios[rng() % 5];
        std::vector<uint64_t> v(1 + rng() % 64);
        for (auto& n : v) n = 1 + rng() % (1u << (8 + rng() % 16));
        const TopkCall c = list(v, ratio);
        const uint32_t shift = shift_of(c);
        for (const uint64_t limit : {uint64_t(0), uint64_t(32), uint64_t(64), uint64_t(128), uint64_t(256)}) {
            const uint32_t per = whole_tiles(c, shift, limit);
            if (!per) continue;
            taken++;
            REQUIRE(per % 2 == 0 && per >= 8 && per <= kWholeMost);   // a streaming block's two tiles are of one group
            uint64_t groups = 0, tiles = 0;
            for (const uint64_t n : v) {
                const uint32_t t = topk_tiles(n), g = (t + per - 1) / per;
                REQUIRE(g >= 1 && g <= 1u << shift && g <= kMaxGroups);
                groups += g;
                tiles += t;
            }
            REQUIRE(groups <= limit && tiles <= kWholeTiles);
            REQUIRE(per * window_share((double)c.k_full / c.bucket_elems) * kFTile <= kWholeOwn);
        }
        TopkCall one = c;
        one.counts = nullptr;
        REQUIRE(!whole_tiles(one, shift, 256));
    }
    REQUIRE(taken > 10000);
    std::vector<uint64_t> ragged;
    for (int i = 0; i < 24; i++) ragged.push_back(1001 + i * 40000);
    REQUIRE(whole_tiles(list(ragged, 0.01), 6, 256) && !whole_tiles(list(ragged, 0.01), 6, 16));
    REQUIRE(!whole_tiles(list({4000000, 4000001}, 0.01), 7, 256) && whole_tiles(list({2500000, 2500001}, 0.01), 6, 256));
    std::puts("ok");
}
"""


def test_lists_in_one_launch(tmp_path):
    src, exe = tmp_path / "whole.cpp", tmp_path / "whole"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-I", os.path.join(ROOT, "mccl_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)
    assert subprocess.run([str(exe)], capture_output=True, text=True, timeout=120).stdout == "ok\n"


LONG_BUCKETS = r"""
#include "topk_route.h"
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <vector>
using namespace mcclhip;
static bool one(uint64_t others, uint32_t count, uint64_t longest, double ratio) {   // tiles
    std::vector<uint64_t> v(count, others * kFTile);
    v.push_back(longest * kFTile);
    const uint64_t n = std::max(others, longest) * kFTile;
    const uint32_t k = (uint32_t)(n * ratio);
    const TopkCall c = {n * v.size(), n, (uint32_t)v.size(), v.data(), k ? k : 1, topk_many(n, ratio)};
    return whole_tiles(c, c.many ? 8 : topk_group_shift_few(topk_tiles(n)), 256);
}
int main() {
    for (const double ratio : {0.001, 0.005, 0.008, 0.009, 0.01, 0.011, 0.012, 0.02}) {
        const bool dense = ratio > 0.0085 && ratio < 0.0115;   // few slots a tile and many candidates in them
        const bool ok = one(10, 10, 1280, ratio) && one(10, 10, 1281, ratio) != dense &&     // up to 2304 tiles
                        one(198, 10, 320, ratio) && one(198, 10, 324, ratio) &&              // 2300, 2304
                        one(199, 10, 320, ratio) && one(199, 10, 321, ratio) != dense;       // more
        if (!ok) { std::printf("%g\n", ratio); return 1; }
    }
    std::puts("ok");
}
"""


def test_long_buckets_of_dense_tiles_take_two_launches(tmp_path):
    src, exe = tmp_path / "long.cpp", tmp_path / "long"
    src.write_text(LONG_BUCKETS)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-I", os.path.join(ROOT, "mccl_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)
    assert subprocess.run([str(exe)], capture_output=True, text=True, timeout=120).stdout == "ok\n"
