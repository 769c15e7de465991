// Which kernels a top-k compress call takes: plain arithmetic on the call's sizes and the device,
// the same for the library and for the test that checks it on the CPU.
#pragma once

#include <cmath>
#include <stdint.h>

namespace mcclhip {

enum Path { kPathExact, kPathStream, kPathResident };

constexpr int kFSample = 8192;              // sampled elements per bucket
constexpr uint64_t kFTile = 4096;           // single-pass path: elements per streaming block
constexpr int kTileSlots = 128;             // ... candidate slots per tile
constexpr int kManySlots = 1024;            // ... of calls with large ratios
constexpr uint64_t kWideTiles = 6144;       // ... a launch of at most this many has blocks of 512 threads
constexpr uint32_t kMaxGroups = 1u << 8;    // ... at most this many groups of tiles per bucket
constexpr uint64_t kFastMinBucket = 1u << 18;
constexpr uint64_t kRMaxBlocks = 128;       // resident path: blocks of one bucket
constexpr uint64_t kRVecElems = 4096;       // ... elements per block and vector of a thread
constexpr uint64_t kRMaxBucket = kRMaxBlocks * kRVecElems * 4;  // 2,097,152 elements

// Groups of tiles per bucket, the power of two.  A group is a bin block and a select block, whose wavefronts go
// through its tiles one after the other, at the end of the call with nothing beside them: the fewer tiles the sooner, as
// long as the call's select blocks go in one launch of 1024 (`groups`: with topk_group_shift_few for every bucket).
// us per call at 1 %, 64 groups against 128: one bucket of 2.5 M elements 27.5 / 28.3, of 6,553,600 34.6 / 32.8, five of
// them 90.7 / 89.6, 15, whose select blocks then go in two launches, 212 / 225; 128 against 256: one of 6,553,600
// 32.8 / 33.9, of 13 M through compress and decompress 77.4 / 75.4.
// At the lines, 64 / 128 / 256 groups: one bucket of 3.6 M 29.0 / 29.1 / 30.5, of 4 M 29.5 / 30.3 / 33.1, of 5 M 31.3 / 32.1 / 34.3, of 7.3 M 37.3 /
// 35.5 / 37.4, of 8.4 M 41.7 / 37.4 / 38.6, of 8.5 M 46.0 / 39.9 / 42.0, of 9.5 M 50.6 / 42.7 / 42.9, of 13.1 M 66.9 / 52.4 / 51.8; two buckets of 4 M
// 37.0 / 35.8 / 41.3, eight 91.4 / 92.0 / 115; 24 listed ones of 1001 to 4 M 53.0 / 54.8 / 58.7.
constexpr uint32_t topk_group_shift_few(uint64_t tiles) { return tiles <= 64 * 14 ? 6 : tiles <= 128 * 16 ? 7 : 8; }
// Otherwise more than 64 only past 28 tiles in each: so many a block keeps in registers, the others it reads again on
// every pass.  64 groups against more: one bucket of 10 M elements 58 / 47, of 13.1 M 72 / 54, of 26.2 M 136 / 89.
constexpr uint32_t topk_group_shift(uint64_t tiles, uint64_t groups) {
    return groups <= 1024 ? topk_group_shift_few(tiles) : tiles <= 64 * 28 ? 6 : tiles <= 128 * 28 ? 7 : 8;
}

constexpr uint32_t topk_tiles(uint64_t elems) { return (uint32_t)((elems + kFTile - 1) / kFTile); }
// Tiles of a group and groups of a bucket.  A group has a tile at least for each of a block's four wavefronts.
constexpr uint32_t topk_group_tiles(uint32_t tiles, uint32_t shift) {
    const uint32_t per = (tiles + (1u << shift) - 1) >> shift;
    return per < 4 ? 4 : per;
}
constexpr uint32_t topk_groups(uint32_t tiles, uint32_t shift) {
    return (tiles + topk_group_tiles(tiles, shift) - 1) / topk_group_tiles(tiles, shift);
}
// Groups that the launches of a buffer's buckets have blocks for, for each bucket: a shorter last bucket can have more of
// them than the others (of at most 128, 1600 tiles make 124 of 13, 1536 make 128 of 12).
constexpr uint32_t topk_launched_groups(uint32_t tiles, uint32_t last_tiles, uint32_t shift) {
    return topk_groups(tiles, shift) > topk_groups(last_tiles, shift) ? topk_groups(tiles, shift) : topk_groups(last_tiles, shift);
}

// Expected share of a bucket inside the sampled window (see sample_window).
inline double window_share(double ratio) {
    const double ks = ratio * kFSample;
    return (ks + 6.0 * std::sqrt(ks) + 16.0) / kFSample;
}

// Whether a call's tiles have slots for many candidates (kManySlots): where the ratio fills 65 % of kTileSlots,
// about 1.13 %, tiles begin to run out of them, and one that does is read again as a whole by every later pass.  us
// per call, 128 slots against 1024: one bucket of 2.5 M elements at 1.1 % 28.8 / 30.1, of 6,553,600 at 1.1 % 36.5 / 35.7, at
// 1.2 % 41.9 / 35.0, at 1.6 % 164 / 35.5, 15 of them at 1.1 % 226 / 223, at 1.2 % 244 / 223, at 1.6 % 430 / 226.
// By the ratio and the bucket's length alone, as the workspace is sized by it, and not for buckets so
// short that their workspace would no longer serve ratios below the line.
constexpr uint64_t kManyMinBucket = 1u << 16;
inline bool topk_many(uint64_t bucket_elems, double ratio) {
    return bucket_elems >= kManyMinBucket && window_share(ratio) > 0.65 * kTileSlots / kFTile;
}
// ... their groups of tiles per bucket, the power of two.  Their blocks read slots again on every pass, a tile
// after the other: as many groups as keep the call's select launch in one (`groups`: with 256 for every bucket).
constexpr uint32_t topk_group_shift_many(uint64_t tiles, uint64_t groups) {
    const uint32_t s = groups <= 1024 ? 8 : groups <= 2048 ? 7 : 6;
    return s > topk_group_shift(tiles, groups) ? s : topk_group_shift(tiles, groups);
}

// Whether the blocks of a streaming launch over that many tiles have 512 threads instead of 256.  Their sample
// is evaluated sooner, and 2048 tiles are resident instead of 1536 (a bucket of 6,553,600 elements has 1600: a
// second round of 64 tiles took as long as half the first); where many rounds follow each other, slots that are
// given back 256 threads at a time are filled sooner.  us per call at 1 %, 256 threads against 512: one bucket of 2.5 M
// elements 30.1 / 28.8, of 6,553,600 38.6 / 36.2, of 10 M 48.0 / 47.3, two of 6,553,600 52.4 / 52.5, four 80.2 / 79.7,
// 24 of 1.7 M 119.1 / 120.4, four of 13.1 M 133 / 138, 15 of 6,553,600 216.6 / 221.3.
constexpr bool stream_wide(uint64_t tiles) { return tiles <= kWideTiles; }

// How long the streaming blocks that start together with the sample blocks hold back, in steps of 512 clocks (0.21 us):
// their loads would bury the samples' few, and they wait for the samples all the same.  A launch whose tiles are loaded
// before its samples are evaluated gains by waiting longer; one with more, by loading sooner.  us per call at 1 %, 7 / 9 / 10 / 11 /
// 12 / 14 steps: one bucket of 2.2 M elements (538 tiles) 25.4 / 25.2 / 25.1 / 24.5 / 24.3 / 24.3, of 4 M (977) 27.9 / 28.0 / 26.9 / 26.5 / 26.0 /
// 26.0, of 1100 tiles 29.2 / 28.6 / 28.1 / 27.5 / 27.4 / 27.5, of 1221 29.5 / 28.9 / 28.5 / 28.1 / 27.9 / 28.1, of 1465 30.6 / 29.8 / 29.4 / 29.3 / 29.3 /
// 29.6, of 1536 30.3 / 29.5 / 29.5 / 29.8 / 29.9 / 30.2, of 1550 30.4 / 31.0 / 30.9 / 31.3 / 31.8 / 32.3, of 1600 31.1 / 30.8 / 31.1 / 32.2 / 32.6 / 33.1, of 8 M (1954)
// 33.8 / 34.2 / 35.4 / 36.2 / 36.8 / 37.8, of 10 M 42.0 / 41.7 / 41.7 / 42.6 / 42.1 / 43.6; two of 2.2 M (1075) 27.0 / 26.4 / 25.9 / 25.5 / 26.4 / 26.0, as a list 27.0 /
// 26.5 / 26.2 / 26.5 / 27.0 / 28.6, of 3 M (1465) 29.8 / 30.1 / 30.1 / 31.3 / 31.5 / 31.4; 24 listed ones of 1001 to 1 M (952) 26.0 / 25.6 / 25.4 / 25.0 / 25.0 / 24.9, to
// 1.5 M (1357) 27.8 / 27.9 / 28.4 / 28.5 / 28.2 / 28.1, 16 of 300,000 (1184) 26.8 / 27.1 / 28.6 / 27.6 / 28.5 / 28.8; one of 4 M at 5 % 33.8 / 33.3 / 32.7 / 32.3 / 31.9 / 31.7.
// (Two runs of one side differ by 0.2 to 0.6.)
constexpr uint32_t stream_hold(uint64_t tiles, uint32_t nbuckets) {
    if (nbuckets == 1) return tiles <= 1024 ? 14 : tiles <= 1536 ? 11 : 7;
    return tiles <= 1152 ? 10 : 7;
}

// The buckets of a call: consecutive ranges of bucket_elems elements, the last one shorter, or, with
// counts, nbuckets buffers of those lengths, bucket_elems the longest.
struct TopkCall {
    uint64_t n_total, bucket_elems;
    uint32_t nbuckets;
    const uint64_t* counts;
    uint32_t k_full;  // picks of a bucket of bucket_elems
    bool many = false;  // topk_many of the call
};

// The most blocks of one resident launch that may wait for others.  Blocks of a bucket wait for each
// other, so every launch that can be under way has to fit the GPU whole, whatever the others are: a
// process's streams share `queues` hardware queues, each with one launch under way.  `slots` blocks
// fit the GPU at once.  Blocks are dealt to the accelerator dies in turn, hence the multiple of eight.
constexpr uint64_t resident_limit(uint64_t slots, uint32_t queues) { return slots / (queues ? queues : 1) / 8 * 8; }

// ... on a stream.  One that is confined to some of the GPU's CUs finds fewer slots, and the runtime gives
// streams of each priority `queues` hardware queues of their own, so that twice or three times as many
// launches could be under way: on neither do blocks wait for others.
struct StreamShare {
    int cus, priority;  // 0: the default
};
constexpr uint64_t stream_limit(const StreamShare& s, int cus, uint64_t per_cu, uint32_t queues) {
    return s.cus < cus || s.priority != 0 ? 0 : resident_limit((uint64_t)cus * per_cu, queues);
}

// Blocks that wait for others with `vecs` vectors per thread: those of every bucket of more than one block.
inline uint64_t resident_waiting(const TopkCall& c, int vecs) {
    const uint64_t per = kRVecElems * (uint64_t)vecs;
    const auto blocks = [&](uint64_t n) { return n > per ? (n + per - 1) / per : 0; };
    if (!c.counts) return (c.nbuckets - 1) * blocks(c.bucket_elems) + blocks(c.n_total - (c.nbuckets - 1) * c.bucket_elems);
    uint64_t sum = 0;
    for (uint32_t b = 0; b < c.nbuckets; b++) sum += blocks(c.counts[b]);
    return sum;
}

// Groups per bucket, the power of two, where `fits` blocks of a select launch may wait (stream_limit): a bucket whose
// selection falls back to the exact one has its groups' blocks wait for each other.  64 of them are resident together on
// 16 CUs; more only where they are whatever else runs.  A wait that runs out instead costs the bucket its payload.
constexpr uint32_t topk_group_shift_fits(uint32_t shift, uint64_t fits) {
    const uint32_t most = fits >= 256 ? 8 : fits >= 128 ? 7 : 6;
    return shift < most ? shift : most;
}
constexpr uint32_t topk_shift(uint64_t tiles, uint64_t groups, bool many, uint64_t fits) {
    return topk_group_shift_fits(many ? topk_group_shift_many(tiles, groups) : topk_group_shift(tiles, groups), fits);
}
constexpr uint64_t kFewestFits = 64;  // blocks of the fewest groups that a long bucket has

// Vectors per thread of a resident launch, 0 when more than `limit` of its blocks would wait.  The barriers
// cost more with more blocks, the passes over a block's elements with more vectors, and a bucket of one block has none of
// the former; measured (one bucket, 1 %): 4097 elements 10.6 / 8.1 us with 1 / 2 vectors, 8192 10.9 / 8.6, but 12,000
// 11.4 / 11.9 with 1 / 4, 16,384 12.2 / 12.1; 262,144 elements 17.8 / 18.0 us with 1 / 2 vectors, 400,000 19.8 / 19.5, 524,288 20.0 / 19.3 / 20.7
// with 1 / 2 / 4, 700,000 21.1 / 22.2 with 2 / 4, 1 M 21.7 / 22.0.  Several buckets take as many as
// bring the launch under the limit.
inline int resident_vecs(const TopkCall& c, uint64_t limit) {
    if (c.bucket_elems > kRMaxBucket) return 0;
    int v = c.bucket_elems > kRVecElems && c.bucket_elems <= 2 * kRVecElems ? 2 : c.bucket_elems <= 64 * kRVecElems ? 1 : c.bucket_elems <= (c.nbuckets == 1 ? 128 : 64) * 2 * kRVecElems ? 2 : 4;
    for (; v <= 4; v *= 2)
        if (resident_waiting(c, v) <= limit) return v;
    return 0;
}

// A list goes in as many launches as it takes to keep each under `limit`.  order[0 .. left): its remaining
// buckets, longest first; brings those of the next launch to the front, in order, and returns their number.
inline uint32_t next_launch(const uint32_t* counts, uint32_t* order, uint32_t left, uint64_t per, uint64_t limit) {
    uint32_t taken = 0;
    uint64_t waiting = 0;
    for (uint32_t i = 0; i < left; i++) {
        const uint32_t b = order[i];
        const uint64_t blocks = counts[b] > per ? (counts[b] + per - 1) / per : 0;
        if (waiting + blocks > limit) continue;
        waiting += blocks;
        for (uint32_t j = i; j > taken; j--) order[j] = order[j - 1];
        order[taken++] = b;
    }
    return taken;
}

// Tiles of a group where the streaming path takes a list in one launch (topk_whole.hip), an even number, the same for
// every bucket; 0 where it takes two.  A group is a select block that waits for others, so a call has at most `limit` of
// them (stream_limit), at most 1 << shift in a bucket, and candidates in it that its block can keep: beyond, a block reads
// them from memory on each of four passes (24 buckets of 1001 to 1 M at 5 %, 33 and 10 tiles a group: 32.7 us in two
// launches, 40 / 30 in one).  us per call, two launches / one, both as they stand (two runs of one side differ by 0.2 at 2 % and
// 5 %, 1 at 1 %): 24 buckets of 1001 to 1.5 M elements (1357 tiles) 30.2 / 28.2, at 0.1 % 28.9 / 25.7, at 2 % 34.6 / 28.7, to 2.2 M 37.3 /
// 34.0, 12 of 1000 to 2 M 26.6 / 25.5, 60 of 1000 to 1 M 42.1 / 37.6, 16 of 300,000 29.5 / 26.9, of 1 M 58.0 / 54.8, two of 2.5 M 28.1 / 27.8, three
// of 2.2 M 31.0 / 29.5, one of 2.5 M 25.1 / 24.5, ten of 1000 to 3 M at 5 % 35.4 / 31.9, 12 of 1000 to 4 M 44.6 / 39.7.  Few large buckets gain
// nothing: two of 4 M 34.9 / 37.4, five of 2.2 M 43.9 / 45.0; nor do those of one buffer, whose two launches have
// no table to read: one bucket of 2.2 M 24.5 / 24.6, of 6,553,600 30.8 / 32.0, eight of 2.5 M 61.8 / 65.3.
// A bucket's groups add to the same counters and meet: with many candidates in few tiles a bucket of many groups waits longer
// than the second launch takes to start.  So above kWholeDenser long buckets go in two launches: three of 100 to 6.5 M 32.7 /
// 33.2, 24 of 1001 to 3 M (2502 tiles, the longest 733) 42.7 / 43.7, 12 of 1000 to 6.5 M 46.2 / 47.2, eight of 1.3 M (318) 42.3 / 42.5, of 2 M (489)
// 54.0 / 55.0; 12 of 1 M (2940, 245) 47.9 / 46.8.  Below, 24 of 1001 to 3 M at 0.1 % 40.3 / 38.2, eight of 2 M 51.0 / 49.0.
// Groups of a call: 24 buckets of 1001 to 1.5 M with 64 / 96 / 160 / 224 of them 29.8 / 28.9 / 28.8 / 27.5.
constexpr uint32_t kWholeMost = 64;      // tiles of a group: a lane each
constexpr uint32_t kWholeOwn = 2600;     // candidates of its group that a select block keeps in LDS
constexpr uint32_t kWholeGroups = 256;
constexpr uint64_t kWholeTiles = 4096;
constexpr double kWholeDenser = 68.0;    // candidates of a tile: a ratio of 0.85 %
inline uint32_t whole_tiles(const TopkCall& c, uint32_t shift, uint64_t limit) {
    if (!c.counts || limit < c.nbuckets) return 0;
    uint64_t sum = 0;
    for (uint32_t b = 0; b < c.nbuckets; b++) sum += topk_tiles(c.counts[b]);
    if (sum > kWholeTiles || (sum > 1664 && c.nbuckets < 8)) return 0;
    const uint64_t longest = topk_tiles(c.bucket_elems);
    const double candidates = window_share((double)c.k_full / (double)c.bucket_elems) * kFTile;  // of a tile
    if (!c.many && candidates > kWholeDenser && longest > (sum > 2304 ? 320 : 1280)) return 0;
    uint32_t per = (uint32_t)((sum + kWholeGroups - 1) / kWholeGroups);
    for (per = per < 8 ? 8 : per + (per & 1); per <= kWholeMost && per * candidates <= 0.92 * kWholeOwn; per += 2) {
        if ((longest + per - 1) / per > 1u << shift) continue;
        uint64_t groups = 0;
        for (uint32_t b = 0; b < c.nbuckets; b++) groups += (topk_tiles(c.counts[b]) + per - 1) / per;
        if (groups <= limit) return per;
    }
    return 0;
}

struct Route {
    Path path;
    int vecs;  // resident path: vectors per thread
};

// `forced`: the tuning key "topk_path" (1 exact, 2 single-pass, 3 resident where it is admitted).
// Measured per call, us:
//   resident where one launch may take the call: 65,536 elements 12.6 against 20.4 streaming and 27.7 exact; 1 M 19.9
//     against 22.5 streaming; 8 x 262,144 21.7 against 23.3 streaming; 16 x 65,536 15.7 against 21.9 streaming and 31.7 exact; 1500 x
//     16,384, where a bucket is one block and nobody waits, 62 against 188 exact.
//   Beyond, several launches are slower than the one or two of the streaming path (24 buckets of 1001 to 1.5 M, three
//     launches: 66 against 28) ...
//   ... unless the streaming path's tiles run out of candidate slots (share of a bucket inside the sampled window
//     times 4096; of 1024 slots 60 % are counted on: ratios up to 0.12).  With slots for many candidates,
//     at 5 %, several resident launches or the exact path against the streaming path: that list 69 / 31, 30 buckets of
//     20,000 to 2 M 163 / 59, one bucket of 2.2 M 63 / 27, of 6.5 M 137 / 38, 4 x 2 M 116 / 40, 20 x 300,000 74 / 36,
//     20 x 1.5 M 283 / 101; one of 6.5 M at 12 % 144 / 47.  Tiles that run out are read again as a whole: with 128 slots
//     that list at 5 % 71 against 199, 30 buckets of 20,000 to 2 M in seven launches 169 against 240.
//   Buckets of one buffer take the exact path then: with 128 slots, at 5 %, one of 6.5 M 144 against 448, 16 x 262,144 57
//     against 99, 4 x 2 M 117 against 167, 20 x 1.5 M 288 against 320; of many large ones the streaming path shares that
//     latency: 12 x 2 M 249 exact, 230 streaming, 50 x 1.7 M 782 and 725, 14 x 6.5 M 905 and 826, 15 x 6.5 M at 20 % with
//     1024 slots 889 and 730.
// `fits`: blocks of a select launch that may wait.  Where not even 64 do, large ratios go by what 128 slots hold: one
// bucket takes the exact path, in which nothing waits.
inline Route choose_path(const TopkCall& c, int forced, uint64_t limit, uint64_t fits = kMaxGroups) {
    const uint64_t tiles = (c.bucket_elems + kFTile - 1) / kFTile;
    const bool streams = (uint64_t)c.nbuckets * (tiles + kMaxGroups + 1) + kMaxGroups < 0x7FFFFFFFull;
    if (forced == 1 && !c.counts) return {kPathExact, 0};
    if (forced == 2 && streams) return {kPathStream, 0};
    // expected share of a bucket inside the sampled window (see sample_window)
    const double ks = (double)c.k_full / (double)c.bucket_elems * kFSample;
    const bool dense = (ks + 6.0 * std::sqrt(ks) + 16.0) / kFSample > (c.many && fits >= kFewestFits ? 0.6 * kManySlots : (double)kTileSlots) / kFTile;
    int vecs = resident_vecs(c, limit);
    // a list can go in several launches, as long as its longest bucket fits one
    if (!vecs && c.counts && (dense || forced == 3) && c.bucket_elems <= (limit < kRMaxBlocks ? limit : kRMaxBlocks) * kRVecElems * 4) vecs = 4;
    if (vecs) return {kPathResident, vecs};
    if (c.counts) return {streams ? kPathStream : kPathExact, 0};
    const bool shared = c.bucket_elems > kRMaxBucket ? c.nbuckets >= 8 : c.bucket_elems >= 400 * kFTile && c.nbuckets >= 12;
    return {streams && c.bucket_elems >= kFastMinBucket && (!dense || shared) ? kPathStream : kPathExact, 0};
}

}  // namespace mcclhip
