"""Which kernels a top-k call takes, on the CPU: csrc/topk_route.h, which the library decides with,
compiled into a program that checks the rule's bounds for many calls and devices and lets launches
that it admits run against each other in a model of the hardware's dispatch."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "topk_route.h"
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <numeric>
#include <random>
#include <vector>
using namespace mcclhip;
typedef std::vector<uint32_t> Blocks;  // blocks of each bucket of one launch, in grid order

#define REQUIRE(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); std::exit(1); } } while (0)

static uint32_t picks(uint64_t n, double ratio) { const uint32_t k = (uint32_t)(n * ratio); return k ? k : 1; }

static TopkCall uniform(uint64_t n, uint64_t be, double ratio) {
    return {n, be, (uint32_t)((n + be - 1) / be), nullptr, picks(be, ratio)};
}
static TopkCall list(const std::vector<uint64_t>& v, double ratio) {
    const uint64_t longest = *std::max_element(v.begin(), v.end());
    return {longest * v.size(), longest, (uint32_t)v.size(), v.data(), picks(longest, ratio)};
}

// The launches of an admitted call.
static std::vector<Blocks> launches(const TopkCall& c, int vecs, uint64_t limit) {
    const uint64_t per = kRVecElems * vecs;
    std::vector<Blocks> out;
    if (!c.counts) {
        Blocks b(c.nbuckets, (uint32_t)((c.bucket_elems + per - 1) / per));
        b.back() = (uint32_t)((c.n_total - (c.nbuckets - 1) * c.bucket_elems + per - 1) / per);
        return {b};
    }
    std::vector<uint32_t> counts(c.counts, c.counts + c.nbuckets), order(c.nbuckets);
    std::iota(order.begin(), order.end(), 0u);
    std::stable_sort(order.begin(), order.end(), [&](uint32_t p, uint32_t q) { return counts[p] > counts[q]; });
    std::vector<int> seen(c.nbuckets);
    for (uint32_t done = 0; done < c.nbuckets;) {
        const uint32_t taken = next_launch(counts.data(), order.data() + done, c.nbuckets - done, per, limit);
        REQUIRE(taken > 0);
        Blocks b;
        for (uint32_t i = 0; i < taken; i++) {
            const uint32_t bucket = order[done + i];
            REQUIRE(!seen[bucket]++ && (i == 0 || counts[order[done + i - 1]] >= counts[bucket]));
            b.push_back((uint32_t)((counts[bucket] + per - 1) / per));
        }
        out.push_back(b);
        done += taken;
    }
    return out;
}
static uint64_t waiting(const Blocks& b) {
    uint64_t s = 0;
    for (uint32_t n : b) s += n > 1 ? n : 0;
    return s;
}

// Launches under way at the same time on `xcds` dies of `slots` slots.  Every launch deals its blocks to
// the dies in turn; a die dispatches a launch's share in order, and which launch goes next on which
// die is drawn.  A bucket ends when all its blocks are resident.  False when nothing can go on.
static bool all_end(const std::vector<Blocks>& ls, int xcds, int slots, std::mt19937& rng) {
    struct Block { int launch, bucket; };
    std::vector<std::vector<std::vector<Block>>> share(ls.size(), std::vector<std::vector<Block>>(xcds));
    std::vector<std::vector<size_t>> next(ls.size(), std::vector<size_t>(xcds));
    std::vector<std::vector<Block>> resident(xcds);
    std::vector<Blocks> missing = ls;
    size_t left = 0;
    for (size_t l = 0; l < ls.size(); l++) {
        uint32_t i = rng() % xcds;
        for (size_t b = 0; b < ls[l].size(); b++)
            for (uint32_t n = 0; n < ls[l][b]; n++, left++) share[l][i++ % xcds].push_back({(int)l, (int)b});
    }
    while (left) {
        bool moved = false;
        // dies take blocks at speeds of their own: one die as much as it can hold
        std::vector<int> dies(xcds);
        std::iota(dies.begin(), dies.end(), 0);
        std::shuffle(dies.begin(), dies.end(), rng);
        for (int x : dies) {
            const size_t favoured = rng() % ls.size();
            while ((int)resident[x].size() < slots) {
                size_t l = ls.size();
                for (size_t j = 0; j < ls.size() && l == ls.size(); j++) {
                    const size_t c = (favoured + j) % ls.size();
                    if (next[c][x] < share[c][x].size()) l = c;
                }
                if (l == ls.size()) break;
                const Block b = share[l][x][next[l][x]++];
                resident[x].push_back(b);
                missing[l][b.bucket]--;
                moved = true;
            }
        }
        for (auto& r : resident) {
            const size_t before = r.size();
            r.erase(std::remove_if(r.begin(), r.end(), [&](const Block& b) { return missing[b.launch][b.bucket] == 0; }), r.end());
            left -= before - r.size();
            moved |= r.size() != before;
        }
        if (!moved) return false;
    }
    return true;
}

int main() {
    // two blocks per CU, four queues
    REQUIRE(resident_limit(512, 4) == 128 && resident_limit(128, 4) == 32 && resident_limit(64, 4) == 16);
    REQUIRE(resident_limit(512, 32) == 16 && resident_limit(0, 4) == 0);
    // a stream that has part of the GPU, or a priority and with it queues beside the four
    REQUIRE(stream_limit({256, 0}, 256, 2, 4) == 128 && stream_limit({32, 0}, 32, 2, 4) == 16);
    REQUIRE(stream_limit({255, 0}, 256, 2, 4) == 0 && stream_limit({256, -1}, 256, 2, 4) == 0 && stream_limit({256, 1}, 256, 2, 4) == 0);
    const double r1 = 0.01, r5 = 0.05;
    const auto path = [](const TopkCall& c, uint64_t limit) { return choose_path(c, 0, limit).path; };
    const auto vecs = [](const TopkCall& c, uint64_t limit) { return choose_path(c, 0, limit).vecs; };
    // one bucket: as many blocks as the limit, never more
    REQUIRE(vecs(uniform(262144, 262144, r1), 128) == 1 && vecs(uniform(262145, 262145, r1), 128) == 2);
    REQUIRE(vecs(uniform(1048577, 1048577, r1), 128) == 4 && vecs(uniform(kRMaxBucket, kRMaxBucket, r1), 128) == 4);
    REQUIRE(path(uniform(kRMaxBucket + 1, kRMaxBucket + 1, r1), 128) == kPathStream);
    REQUIRE(path(uniform(2000000, 2000000, r1), 32) == kPathStream && path(uniform(2000000, 2000000, r1), 16) == kPathStream);
    REQUIRE(vecs(uniform(262144, 262144, r1), 16) == 4 && path(uniform(262145, 262145, r1), 16) == kPathStream);
    REQUIRE(path(uniform(65537, 65537, r1), 0) == kPathExact && path(uniform(300000, 300000, r1), 0) == kPathStream);
    REQUIRE(vecs(uniform(4096, 4096, r1), 0) == 1 && vecs(uniform(1500 * 16384, 16384, r1), 128) == 4);
    // several: more vectors where that brings the call under the limit, else the other paths
    REQUIRE(vecs(uniform(4 * 65536, 65536, r1), 128) == 1 && vecs(uniform(8 * 262144, 262144, r1), 128) == 4);
    REQUIRE(path(uniform(9 * 262144, 262144, r1), 128) == kPathStream && path(uniform(2 * 2000000, 2000000, r1), 128) == kPathStream);
    REQUIRE(path(uniform(4 * 2000000, 2000000, r5), 128) == kPathExact && path(uniform(14 * 2000000, 2000000, r5), 128) == kPathStream);
    const std::vector<uint64_t> ragged = {1500001, 1000003, 700001, 300007, 4097, 4096, 100001, 17};
    REQUIRE(path(list(ragged, r1), 128) == kPathStream && path(list(ragged, r5), 128) == kPathResident);
    REQUIRE(path(list(ragged, r5), 16) == kPathStream && path(list({5, 4000, 1}, r1), 0) == kPathResident);
    // forced paths are bounded as well
    REQUIRE(choose_path(uniform(300000, 300000, r1), 3, 0).path == kPathStream && choose_path(list(ragged, r1), 3, 128).path == kPathResident);
    REQUIRE(choose_path(uniform(300000, 300000, r1), 1, 128).path == kPathExact && choose_path(uniform(5000, 5000, r1), 2, 128).path == kPathStream);

    std::mt19937 rng(1);
    const auto any = [&](uint64_t hi) { return 1 + (uint64_t)(std::exp(std::log((double)hi) * (rng() / 4294967296.0))); };
    const struct { int cus, xcds; } devices[] = {{32, 1}, {64, 2}, {128, 4}, {256, 8}};
    int admitted = 0;
    for (int i = 0; i < 3000; i++) {
        const auto& d = devices[rng() % 4];
        const uint32_t queues = rng() % 4 ? 4 : 1 + rng() % 8;
        const uint64_t slots = 2ull * d.cus, limit = resident_limit(slots, queues);
        std::vector<Blocks> under_way;
        std::vector<std::vector<uint64_t>> kept;
        for (uint32_t tries = 0; under_way.size() < queues && tries < 50; tries++) {
            TopkCall c;
            const double ratio = rng() % 2 ? r1 : r5;
            if (rng() % 2) {
                const uint64_t be = any(kRMaxBucket + 1000);
                c = uniform(be * (1 + rng() % 20) - rng() % be, be, ratio);
            } else {
                std::vector<uint64_t> v(1 + rng() % 64);
                for (auto& n : v) n = any(kRMaxBucket);
                kept.push_back(v);
                c = list(kept.back(), ratio);
            }
            const Route r = choose_path(c, rng() % 4 ? 0 : 3, limit);
            if (r.path != kPathResident) continue;
            const auto ls = launches(c, r.vecs, limit);
            for (const Blocks& b : ls) {
                REQUIRE(waiting(b) <= limit);
                REQUIRE(*std::max_element(b.begin(), b.end()) <= kRMaxBlocks);
            }
            under_way.push_back(ls[rng() % ls.size()]);
            admitted++;
        }
        if (!under_way.empty()) REQUIRE(all_end(under_way, d.xcds, (int)(slots / d.xcds), rng));
    }
    REQUIRE(admitted > 1000);
    // the model does find launches that hold each other up: four buckets of 128 blocks, twice
    int stuck = 0;
    for (int i = 0; i < 200; i++) stuck += !all_end({Blocks(4, 128), Blocks(4, 128)}, 8, 64, rng);
    REQUIRE(stuck > 0);
    return 0;
}
"""


def test_admitted_launches_always_end(tmp_path):
    src, exe = tmp_path / "route.cpp", tmp_path / "route"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-I", os.path.join(ROOT, "mccl_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)
    p = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True, timeout=100)
    assert p.returncode == 0, p.stdout[:2000]


GROUPS = r"""
#include "topk_route.h"
#include <cstdio>
using namespace mcclhip;
int main() {
    int more = 0;
    for (uint32_t shift = 6; shift <= 8; shift++)
        for (uint32_t tiles = 1; tiles <= 4000; tiles += tiles < 700 ? 1 : 13)
            for (uint32_t last = 1; last <= tiles; last++) {
                const uint32_t launched = topk_launched_groups(tiles, last, shift);
                more += topk_groups(last, shift) > topk_groups(tiles, shift);
                if (launched < topk_groups(tiles, shift) || launched < topk_groups(last, shift) || launched > 1u << shift) {
                    std::printf("%u tiles, the last bucket %u, shift %u: %u\n", tiles, last, shift, launched);
                    return 1;
                }
            }
    return more > 1000 ? 0 : 2;
}
"""


def test_a_shorter_last_bucket_has_all_its_groups(tmp_path):
    src, exe = tmp_path / "groups.cpp", tmp_path / "groups"
    src.write_text(GROUPS)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-I", os.path.join(ROOT, "mccl_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)
    p = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True, timeout=100)
    assert p.returncode == 0, p.stdout[:2000]


FALLBACK = SOURCE[:SOURCE.index("int main()")] + r"""
// Groups of the longest bucket of a call, as the library launches them.
static uint32_t groups_of(const TopkCall& c, uint64_t fits) {
    const uint32_t tiles = topk_tiles(c.bucket_elems), most = c.many ? 8 : topk_group_shift_few(tiles);
    return topk_groups(tiles, topk_shift(tiles, c.nbuckets * (uint64_t)topk_groups(tiles, most), c.many, fits));
}
static TopkCall call(uint64_t n, uint64_t be, double ratio) {
    TopkCall c = uniform(n, be, ratio);
    c.many = topk_many(be, ratio);
    return c;
}

int main() {
    // four blocks of the select launch per CU, four queues: the whole GPU, a half, a quarter, an eighth of it
    const auto fits = [](int cus, uint32_t queues) { return stream_limit({cus, 0}, cus, 4, queues); };
    REQUIRE(fits(256, 4) == 256 && fits(128, 4) == 128 && fits(64, 4) == 64 && fits(32, 4) == 32);
    const TopkCall one = call(10000000, 10000000, 0.01);
    REQUIRE(groups_of(one, fits(256, 4)) == 245 && groups_of(one, fits(128, 4)) <= 128 && groups_of(one, fits(64, 4)) <= 64);
    REQUIRE(groups_of(one, fits(32, 4)) <= 64 && groups_of(one, fits(256, 8)) <= 128 && groups_of(one, fits(256, 16)) <= 64);
    // a stream that has part of the GPU, or queues beside the four
    REQUIRE(groups_of(one, stream_limit({60, 0}, 256, 4, 4)) <= 64 && groups_of(one, stream_limit({256, 1}, 256, 4, 4)) <= 64);
    // large ratios: the exact path, which waits for nobody, where the fewest groups might not be resident together
    for (double r : {0.02, 0.05, 0.12})
        for (uint64_t n : {2200000ull, 6553600ull, 30000000ull}) {
            const TopkCall c = call(n, n, r);
            REQUIRE(choose_path(c, 0, 0, fits(256, 4)).path == kPathStream && choose_path(c, 0, 0, fits(64, 4)).path == kPathStream);
            REQUIRE(choose_path(c, 0, 0, fits(32, 4)).path == kPathExact);
            REQUIRE(choose_path(c, 0, 0, 0).path == kPathExact);
        }
    REQUIRE(choose_path(one, 0, 0, 0).path == kPathStream);
    // the sizes of test_gpu_topk_groups.py: elements, bucket, ratio, groups of a bucket, select launches
    const uint64_t tile = kFTile;
    const struct { uint64_t n, be; double ratio; uint32_t groups, launches; } sizes[] = {
        {64 * 14 * tile, 64 * 14 * tile, 0.01, 64, 1}, {64 * 14 * tile + 1, 64 * 14 * tile + 1, 0.01, 113, 1},
        {64 * 28 * tile, 64 * 28 * tile, 0.01, 128, 1}, {64 * 28 * tile + 1, 64 * 28 * tile + 1, 0.01, 120, 1},
        {128 * 16 * tile, 128 * 16 * tile, 0.01, 128, 1}, {128 * 16 * tile + 3, 128 * 16 * tile + 3, 0.01, 228, 1},
        {256 * 28 * tile + 4097, 256 * 28 * tile + 4097, 0.01, 248, 1},
        {8 * 900 * tile, 900 * tile, 0.01, 113, 1}, {9 * 900 * tile, 900 * tile, 0.01, 113, 1}, {10 * 900 * tile, 900 * tile, 0.01, 60, 1},
        {9 * 1850 * tile, 1850 * tile, 0.01, 124, 2}, {9 * 1850 * tile - 3000001, 1850 * tile, 0.01, 124, 2},
        {1600 * tile, 1600 * tile, 0.05, 229, 1}, {40000000, 8000000, 0.05, 123, 1}, {17 * 1048576 - 3, 1048576, 0.05, 64, 2}};
    for (const auto& s : sizes) {
        const TopkCall c = call(s.n, s.be, s.ratio);
        const uint32_t g = groups_of(c, fits(256, 4)), at_once = 1024 / g;
        if (g != s.groups || (c.nbuckets + at_once - 1) / at_once != s.launches) {
            std::printf("%llu / %llu at %g: %u groups\n", (unsigned long long)s.n, (unsigned long long)s.be, s.ratio, g);
            return 1;
        }
    }
    // buckets that fall back in every queue at once, one each, with whatever groups they have
    std::mt19937 rng(2);
    for (int i = 0; i < 2000; i++) {
        const int cus[] = {64, 128, 256}, c = cus[rng() % 3];
        const uint32_t queues = 1 + rng() % 8;
        const uint64_t f = fits(c, queues);
        std::vector<Blocks> under_way;
        for (uint32_t q = 0; q < queues; q++) {
            const uint64_t be = 300000 + rng() % 40000000;
            under_way.push_back({groups_of(call(be * (1 + rng() % 3), be, rng() % 2 ? 0.01 : 0.05), f)});
            if (f >= kFewestFits) REQUIRE(under_way.back()[0] <= f);
        }
        if (f >= kFewestFits) REQUIRE(all_end(under_way, c / 32, 128, rng));
    }
    // the model does find one bucket of 245 groups on an eighth of the GPU, three of them on a half, stuck
    REQUIRE(!all_end({{245}}, 1, 128, rng));
    int stuck = 0;
    for (int i = 0; i < 200; i++) stuck += !all_end({{245}, {245}, {245}}, 4, 128, rng);
    REQUIRE(stuck > 0);
    return 0;
}
"""


def test_a_bucket_that_falls_back_has_its_blocks_resident(tmp_path):
    src, exe = tmp_path / "fallback.cpp", tmp_path / "fallback"
    src.write_text(FALLBACK)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wno-unused-function", "-Werror", "-I", os.path.join(ROOT, "mccl_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True)
    p = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True, timeout=100)
    assert p.returncode == 0, p.stdout[:2000]
