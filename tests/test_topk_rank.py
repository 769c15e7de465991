"""The last step of a selection in a list (csrc/topk_rank.h), compiled and checked on the CPU: the cut that it finds is reached
by as many entries as are wanted, and lists that hold an entry more often than once give no other cut."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "topk_rank.h"
#include <cstdio>
#include <cstdlib>
#include <random>
#include <set>
#include <vector>
using namespace mcclhip;
#define REQUIRE(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); std::exit(1); } } while (0)

int main() {
    std::mt19937_64 rng(1);
    int refused = 0, distinct = 0;
    for (int i = 0; i < 200000; i++) {
        const uint32_t m = 1 + (uint32_t)(rng() % 128), want = 1 + (uint32_t)(rng() % m), parts = 1 + (uint32_t)(rng() % 16);
        std::vector<uint64_t> list(m);
        const uint64_t values = i % 2 ? 1 + rng() % 200 : ~0ull;   // few values: entries twice, also at the cut
        for (auto& e : list) e = rng() % values;
        uint64_t cut = kNoCut;
        for (const uint64_t e : list) {
            uint32_t reach = 0;                                    // counted in parts, as by several wavefronts
            const uint32_t per = (m + parts - 1) / parts;
            for (uint32_t from = 0; from < m; from += per) reach += reaching_entries(list.data(), from, from + per < m ? from + per : m, e);
            if (reach == want) cut = e;
        }
        const bool once = std::set<uint64_t>(list.begin(), list.end()).size() == m;
        if (cut == kNoCut) {
            REQUIRE(!once);
            refused++;
            continue;
        }
        uint32_t picks = 0;
        for (const uint64_t e : list) picks += e >= cut;
        REQUIRE(picks == want);
        distinct += once;
    }
    REQUIRE(refused > 1000 && distinct > 90000);
    std::puts("ok");
}
"""


def test_the_cut_is_reached_by_as_many_as_wanted(tmp_path):
    src, exe = tmp_path / "rank.cpp", tmp_path / "rank"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wno-unknown-pragmas", "-Werror", "-I", os.path.join(ROOT, "mccl_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], capture_output=True, text=True, timeout=120).stdout == "ok\n"
