"""How a list of binary folds is spread over launches (csrc/fold_rows.h), compiled and checked on the
CPU: every fold is in one launch, no large one's blocks stride, and neither the blocks without work
nor the launches are many."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "fold_rows.h"
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>
using namespace mcclhip;

static bool check(const std::vector<uint64_t>& nvec) {
    std::vector<FoldSpan> f(nvec.size());
    uint64_t sum = 0, longest = 0, shortest = ~0ull;
    for (size_t i = 0; i < f.size(); i++) {
        f[i] = FoldSpan{nullptr, nullptr, nvec[i], (uint16_t)i, 0, 0};
        const uint64_t b = fold_blocks(f[i]);
        sum += b;
        longest = std::max(longest, b);
        shortest = std::min(shortest, b);
    }
    std::vector<int> seen(f.size());
    uint64_t launches = 0, surplus = 0;
    bool ok = true;
    fold_rows(f.data(), (uint32_t)f.size(), [&](const FoldSpan* p, uint32_t m, uint64_t blocks) {
        launches++;
        uint64_t work = 0, rounds = 1;
        for (uint32_t i = 0; i < m; i++) {
            seen[p[i].head]++;
            ok = ok && p[i].nvec == nvec[p[i].head];
            work += fold_blocks(p[i]);
            if (blocks) rounds = std::max(rounds, (fold_blocks(p[i]) + blocks - 1) / blocks);
            else ok = ok && p[i].nvec == 0;
        }
        if (rounds == 1) surplus += blocks * m - work;
        ok = ok && blocks * m <= 2 * work + 3 * m && (rounds == 1 || (work <= kFoldLarge && rounds <= kFoldRounds));
    });
    for (int s : seen) ok = ok && s == 1;
    ok = ok && launches <= 1 + 2 * std::log2(1.0 + longest) && (longest > 2 * shortest || launches == 1);
    if (!ok) std::printf("%zu folds of %llu to %llu blocks: %llu launches, %llu of %llu blocks idle\n", f.size(),
                         (unsigned long long)shortest, (unsigned long long)longest, (unsigned long long)launches,
                         (unsigned long long)surplus, (unsigned long long)(surplus + sum));
    return ok;
}

int main() {
    uint64_t bad = 0;
    for (uint64_t big : {0ull, 25'000ull, 250'000ull, 1'638'400ull, 24'127'506ull, 17'179'869'184ull})
        for (size_t few : {1, 2, 12})
            for (size_t n : {1, 2, 10, 60, 120}) {
                std::vector<uint64_t> v(n, 250);
                for (size_t i = 0; i < n && i < few; i++) v[n - 1 - i] = big;
                bad += !check(v);
            }
    std::mt19937_64 rng(1);
    for (int i = 0; i < 20000; i++) {
        std::vector<uint64_t> v(1 + rng() % 120);
        const double spread = std::log(1.0 + rng() % 30'000'000);
        for (auto& x : v) x = (uint64_t)std::exp(spread * (rng() % 1001) / 1000.0);
        bad += !check(v);
    }
    return bad != 0;
}
"""


def test_every_fold_is_launched_once_and_whole(tmp_path):
    src, exe = tmp_path / "rows.cpp", tmp_path / "rows"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-I", os.path.join(ROOT, "mccl_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)
    p = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True, timeout=100)
    assert p.returncode == 0, p.stdout[:2000]
