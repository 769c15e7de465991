// How the W-way ring fold is cut into chunks, rows of blocks and tiles: plain arithmetic, the same for
// the launch (the grid), the kernel (a block's place) and the test that walks grids on the CPU.
#pragma once

#include <stdint.h>

namespace mcclhip {

// Threads per block of the binary folds and of the ring fold (fold.hip has the measurements).
constexpr int kFoldBlock = 64;
// Blocks go to the XCDs in turn, and tiles start where the destination's address is a multiple of
// 1 KiB and rows of tiles at multiples of 8 KiB (kGroupVecs vectors): an XCD always works on the same
// eighth of every 8 KiB, and no wavefront ends inside a cache line.  Chunks that start anywhere
// else: ring fold of 8 ranks, chunks of 819,204 elements 638 us with tiles that start with the chunk,
// 597 with tiles on 1 KiB, 579 with rows on 8 KiB.
constexpr int kXcds = 8;
constexpr int kGroupVecs = kXcds * kFoldBlock;
// Vectors per lane and rank buffer of the ring fold, in one-wavefront blocks as well: one where the
// world size is known at compile time (all ranks' loads are in flight together; two cost 2-3 % from
// two to eight ranks), four where the ranks come one after the other.
constexpr int ring_unroll(int ws) { return ws == 0 ? 4 : 1; }
constexpr uint64_t ring_tile_vecs(int ws) { return (uint64_t)kFoldBlock * ring_unroll(ws >= 2 && ws <= 8 ? ws : 0); }

// The buckets of a call and the chunks of a bucket: computed by the launch, so that a block starts
// with multiplications only.
struct RingCut {
    uint64_t n_total, bucket_elems;
    uint64_t ce_full, ce_last;  // elements per chunk in a full bucket and in the last one
    uint32_t nbuckets, chunked;
};
// 0 < bucket_elems <= n_total
constexpr RingCut ring_cut(uint64_t n_total, uint64_t bucket_elems, uint32_t nbuckets, uint32_t nchunks, bool chunked) {
    return {n_total, bucket_elems, (bucket_elems + nchunks - 1) / nchunks,
            (n_total - (nbuckets - 1) * bucket_elems + nchunks - 1) / nchunks, nbuckets, chunked ? 1u : 0u};
}

// One chunk of one bucket, which a row of blocks folds: `head` elements up to the output's next
// 16-byte boundary, `nvec` vectors, the rest.  The row's tiles start at a tile group of the output's
// addresses: `lead` vectors lie in front of the chunk.
struct RingRow {
    uint64_t e0, len;  // first element of the chunk in every buffer, elements
    uint64_t head, nvec;
    uint32_t lead;
};
constexpr RingRow ring_row(const RingCut& cut, uint64_t out_addr, int es, uint32_t bucket, uint32_t chunk) {
    const uint64_t bstart = (uint64_t)bucket * cut.bucket_elems;
    const bool last = bucket + 1 == cut.nbuckets;
    const uint64_t bn = last ? cut.n_total - bstart : cut.bucket_elems;
    const uint64_t ce = last ? cut.ce_last : cut.ce_full;
    const uint64_t cstart = (uint64_t)chunk * ce;
    const uint64_t rest = cstart < bn ? bn - cstart : 0;
    const uint64_t len = rest < ce ? rest : ce;
    const uint64_t e0 = bstart + cstart;
    const uint64_t o = out_addr + e0 * es;
    uint64_t head = ((16 - (o & 15)) & 15) / es;
    if (head > len) head = len;
    return {e0, len, head, (len - head) * es / 16, (uint32_t)((o + head * es) >> 4) & (uint32_t)(kGroupVecs - 1)};
}

// Tiles per row: enough for the longest `lead` + `nvec` of any chunk.  A chunk that starts on a tile
// group has no lead; the chunks of the last bucket are cut on their own, and where the full buckets'
// start on groups its chunks need not.
constexpr uint64_t ring_tiles(const RingCut& cut, uint64_t out_addr, int es, uint32_t nchunks, uint64_t tile_vecs) {
    const uint64_t group = 16 * kGroupVecs;
    const uint64_t common = out_addr | cut.bucket_elems * es;
    const uint64_t full = cut.ce_full * es / 16 + ((common | cut.ce_full * es) % group == 0 ? 0 : kGroupVecs - 1);
    const uint64_t last = cut.ce_last * es / 16 + ((common | cut.ce_last * es) % group == 0 ? 0 : kGroupVecs - 1);
    const uint64_t tiles = ((full > last ? full : last) + tile_vecs - 1) / tile_vecs;
    if (nchunks * cut.nbuckets <= 1) return tiles < 1 ? 1 : tiles;
    return tiles < 1 ? kXcds : (tiles + kXcds - 1) / kXcds * kXcds;  // every row starts on the same XCD
}

}  // namespace mcclhip
