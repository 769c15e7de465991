"""The ring fold's grid on the CPU: csrc/ring_cut.h, which the launch and the kernel share, compiled
into a program that walks the rows of many calls and checks that the chunks partition the gradient
and that every 16-byte vector of every chunk lies in a tile of its row."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "ring_cut.h"
#include <cstdio>
#include <random>
using namespace mcclhip;

static bool check(uint64_t out, int es, int ws, bool chunked, uint64_t bucket, uint64_t n) {
    if (bucket > n) bucket = n;
    const uint32_t nb = (uint32_t)((n + bucket - 1) / bucket), nchunks = chunked ? 2 * ws : ws;
    const RingCut cut = ring_cut(n, bucket, nb, nchunks, chunked);
    const uint64_t slots = ring_tiles(cut, out, es, nchunks, ring_tile_vecs(ws)) * ring_tile_vecs(ws);
    uint64_t next = 0;  // first element that no chunk has covered
    for (uint32_t b = 0; b < nb; b++)
        for (uint32_t c = 0; c < nchunks; c++) {
            const RingRow r = ring_row(cut, out, es, b, c);
            const uint64_t tail = r.len - r.head - r.nvec * 16 / es;
            const bool starts = r.len == 0 || r.e0 == next;
            const bool vectors = r.nvec == 0 || ((out + (r.e0 + r.head) * es) % 16 == 0 && r.lead + r.nvec <= slots);
            if (!starts || !vectors || r.head * es >= 16 || tail * es >= 16) {
                std::printf("out %llu es %d ws %d chunked %d bucket %llu n %llu: bucket %u chunk %u\n", (unsigned long long)out,
                            es, ws, chunked, (unsigned long long)bucket, (unsigned long long)n, b, c);
                return false;
            }
            next += r.len;
        }
    return next == n;
}

int main() {
    const uint64_t buckets[] = {5, 4096, 16384, 50001, 65536, 262144, 6553600};
    const uint64_t shorts[] = {0, 1, 4, 8, 12, 64, 100, 1000, 5000};
    uint64_t bad = 0;
    for (int es : {2, 4})
        for (int ws = 1; ws <= 12; ws++)
            for (int chunked = 0; chunked < 2; chunked++)
                for (uint64_t out : {0, 16, 512, 8192 + 1024, es, 16 - es})
                    for (uint64_t be : buckets)
                        for (uint64_t m = 1; m <= 3; m++) {
                            for (uint64_t s : shorts)
                                if (s < be) bad += !check(out, es, ws, chunked, be, m * be - s);
                            bad += !check(out, es, ws, chunked, be, (m - 1) * be + be * 3 / 4 + 1);
                        }
    std::mt19937_64 rng(1);
    for (int i = 0; i < 200000; i++) {
        const int es = rng() % 2 ? 2 : 4;
        const uint64_t be = rng() % 2 ? buckets[rng() % 7] : 1 + rng() % 100000;
        bad += !check(rng() % 4 ? 0 : rng() % 8192 / es * es, es, 1 + rng() % 12, rng() % 2, be, 1 + rng() % (be * (1 + rng() % 20)));
    }
    return bad != 0;
}
"""


def test_every_vector_of_every_chunk_has_a_tile(tmp_path):
    src, exe = tmp_path / "cut.cpp", tmp_path / "cut"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-I", os.path.join(ROOT, "mccl_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)
    p = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True, timeout=100)
    assert p.returncode == 0, p.stdout[:2000]
