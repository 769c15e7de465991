// Top-k compress of a list of buckets: one launch, one pass over memory.
//
// Semantics and ordering as in topk.hip (csrc/compression/TopKCompression.cpp:38-120).
//
// The two launches of topk.hip spend what such a call takes on a chain: the last tiles' candidates are read back, counted
// and listed by bin blocks, the launch ends, the next one starts, reads them again, and selects.  Here one block does both
// for its group of tiles, with the group's candidates in LDS in between.
//
// k_topk_whole - blocks of 512 threads, in dispatch order:
//   sample blocks     one per bucket: the candidate window and the predicted threshold (sample_window), published when
//                     everything that the others add into has been cleared.
//   streaming blocks  two 4096-element tiles each, in address order, as in k_topk_stream (stream_tiles).
//   select blocks     one per group.  When its group's tiles are finished a block takes their candidates into LDS, counts
//                     them per window bin, adds the counts to the bucket's, which gives it places in the bins' lists, and
//                     lists them.  When all of the bucket's select blocks have, each of them finds the bin of the k-th
//                     largest key, selects the threshold and the tie rule in that bin's list, and writes its group's
//                     picks in index order.
//
// Everything that crosses blocks is written and read past the caches (agent scope).
//
// Progress.  Sample and streaming blocks wait for earlier blocks of the grid only, as in k_topk_stream.  The select blocks
// of a bucket wait for each other as well, so a launch has at most as many of them as the resident path has blocks that
// wait (whole_tiles), a quarter of the GPU's slots where a process has four hardware queues: however many launches are under
// way, all of theirs find slots on every XCD, and being the last blocks of their grids they keep no other block from one that
// they wait for.  Every wait has a limit (`limit_ticks`); a bucket that gives up is left as in k_topk_stream.  The window
// stays published behind the launch: blocks that wait for it can leave before the sample block has published, and no count of
// them survives that.  A replay would carry the same epoch, so a call that is recorded takes two launches (launch_by_path).
//
// What bounds it is the chain of round trips behind the last streaming block.  One bucket of 2.2 M elements, us from the
// first block's start, in a build with stamps: window published 7.9, sums stored 10.7, tiles finished 12.5, a group's candidates in
// LDS 13.8, counted and the places known 15.9, listed and met 19.8, the bin found 20.8, threshold 23.7, picks counted 24.3, stored
// 25.4.  24 buckets of 1001 to 1.5 M elements at 1 %, two launches / this one: 30.2 / 28.2 us.  Also built, and slower: streaming
// blocks that count and list their candidates themselves, behind one atomic a bin and block (6.5 M elements 52.7 us), and select
// blocks that add up all groups' rows of counts instead of meeting (31.6 at 2.2 M).
#include "topk_stream.hip.h"

namespace mcclhip {

namespace {

constexpr int kWThreads = 512;
constexpr int kWWaves = kWThreads / kWave;
constexpr uint32_t kWTiles = kWWaves / kFWaves;  // of a streaming block
constexpr int kWOwn = (int)kWholeOwn;  // (four blocks to a CU: 40 KiB of LDS each)
constexpr int kWList = 4;      // entries of the threshold bin's list that a thread keeps
constexpr int kWRank = 128;    // entries that are ranked by counting
constexpr int kWWalk = 4;      // vectors in flight in a walk over a dense tile

// The kernel's first argument (see BucketsArg).
struct WholeBuckets {
    Buckets b;
    uint32_t select[kMaxListed];  // the bucket's first select block, counted from the launch's first one
};
struct Whole {
    uint32_t tpg;    // tiles of a group, an even number, at most kWholeMost
    uint32_t shift;  // rows and counters are laid out for 1 << shift groups a bucket
    uint32_t select_at;   // the first select block
    uint32_t first_wave;  // blocks that start together with the sample blocks ...
    uint32_t hold;        // ... and how long they hold back
};

template <bool MANY>
struct WholeLds {
    union {
        SampleLds<kWThreads> s;  // sample block
        StreamBlockLds<kWWaves, TileShape<MANY>::kStage> a;
        struct {  // select block
            uint32_t lh[kBins0] __attribute__((aligned(16)));
            uint32_t dbuf[kWWaves][kWWalk * kWave];
            uint64_t own[kWOwn];     // the group's candidates, in index order
            uint64_t list[kWRank];   // entries of the threshold bin that share a prefix
            uint64_t cut;
            uint32_t cnt[kCoarse], base[kCoarse];
            uint32_t win[4];
            uint32_t wsum[kWWaves], res[1][2];
            uint32_t wtot[kWWaves], wmine[kWWaves];
            uint32_t scratch[kWWaves + 2];
            uint32_t flag, count;
        } e;
    };
};

static_assert(sizeof(WholeLds<false>) <= 40 * 1024 && sizeof(WholeLds<true>) <= 40 * 1024, "four blocks to a CU");

__device__ __forceinline__ FusedGeo whole_geo(const Geometry& g, BucketsArg bk, uint32_t b, const Whole& h) {
    FusedGeo f;
    f.bn = bucket_count(g, bk, b);
    f.k = bucket_k(g, bk, b);
    f.ntiles = (uint32_t)((f.bn + kFTile - 1) / kFTile);
    f.tpg = h.tpg;
    f.ng = (f.ntiles + f.tpg - 1) / f.tpg;
    return f;
}
// A line of each group: its finished tiles; the arrivals that it counts of the bucket's select blocks; and the word that
// its select block waits at until all have arrived.
__device__ __forceinline__ uint32_t* group_line(const Workspace& w, const Whole& h, uint32_t b, uint32_t grp) {
    return w.grp_cnt + (((uint64_t)b << h.shift) + grp) * kCntStride;
}
enum { G_TILES = 0, G_ARRIVED = 1, G_GO = 2 };
// The group's candidates in the bins above bin j, for each j.
__device__ __forceinline__ uint32_t* group_above(const Workspace& w, const Whole& h, uint32_t b, uint32_t grp) {
    return w.gsuf + (((uint64_t)b << h.shift) + grp) * kCoarse;
}

template <bool MANY>
__device__ __forceinline__ void whole_sample(BucketsArg bk, const Geometry& g, const Workspace& w, const Whole& h, uint32_t b,
                                             uint32_t published, WholeLds<MANY>& L) {
    const FusedGeo fg = whole_geo(g, bk, b, h);
    uint32_t* st = w.state + (uint64_t)b * kStateWords;
    const SampleWindow win = sample_window<kWThreads>(bucket_grad(g, bk, b), bucket_residual(g, bk, b), fg.bn, fg.k, L.s, [&] {
        const u4a z = {0u, 0u, 0u, 0u};
        if (threadIdx.x < fg.ng) store16_agent(group_line(w, h, b, threadIdx.x), z);
        if (threadIdx.x < kCoarse / 4) store16_agent(w.bin_fill + (uint64_t)b * kCoarse + 4 * threadIdx.x, z);
        if (threadIdx.x == 0) {
            st_agent(st + S_OK, 0u);
            st_agent(st + S_TIMEOUT, 0u);
            st_agent(st + S_DONE, 0u);
            store16_agent(st + S_BARF, z);
        }
        // the histograms of the exact selection, should the select blocks need it
        for (uint32_t i = threadIdx.x; i < kHistWords / 4; i += kWThreads) store16_agent(w.hist + (uint64_t)b * kHistWords + 4 * i, z);
    });
    if (threadIdx.x == 0) store16_agent(st + S_LO_KEY, u4a{win.lo, win.hi, win.that, published});
}

// All threads of a select block; every store and atomic of the block has arrived when it is counted.  The blocks arrive at
// eight lines, the last one of each at the bucket's word, and the last of all releases every block at a line of its own:
// a word that many poll serves polls and arrivals in turn, some 25 ns each.
__device__ __forceinline__ bool whole_barrier(const Workspace& w, const Whole& h, uint32_t b, uint32_t grp, uint32_t ng, uint32_t epoch,
                                              uint32_t* flag, uint64_t limit_ticks) {
    constexpr uint32_t kLines = 8;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t lines = ng < kLines ? ng : kLines, l = grp % lines;
        const uint32_t parties = (ng - l + lines - 1) / lines;  // groups with grp % lines == l
        uint32_t last = __hip_atomic_fetch_add(group_line(w, h, b, l) + G_ARRIVED, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == parties;
        if (last) {
            uint32_t* const st = w.state + (uint64_t)b * kStateWords;
            last = __hip_atomic_fetch_add(st + S_DONE, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == lines;
        }
        *flag = last;
    }
    __syncthreads();
    if (*flag) {
        if (threadIdx.x < ng) st_agent(group_line(w, h, b, threadIdx.x) + G_GO, epoch);
        return true;
    }
    __syncthreads();
    if (threadIdx.x == 0) *flag = wait_word<1>(group_line(w, h, b, grp) + G_GO, epoch, limit_ticks);
    __syncthreads();
    return *flag != 0;
}

template <bool MANY>
__device__ __forceinline__ void whole_select(BucketsArg bk, const Geometry& g, const Workspace& w, const Whole& h, uint32_t b, uint32_t grp,
                                             const FusedGeo& fg, uint32_t epoch, uint64_t limit_ticks, WholeLds<MANY>& L) {
    auto& S = L.e;
    constexpr int kSlots = TileShape<MANY>::kSlots;
    uint32_t* st = w.state + (uint64_t)b * kStateWords;
    uint32_t* out = bucket_wire(g, bk, b);
    float* const rp = bucket_residual(g, bk, b);
    const uint32_t lane_id = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const uint64_t below = (1ull << lane_id) - 1ull;
    const uint32_t k = fg.k, ng = fg.ng;
    const uint64_t bn = fg.bn;
    uint32_t* const line = group_line(w, h, b, grp);
    // this group's tiles, and this wavefront's share of them
    const uint32_t tg0 = grp * fg.tpg, tg1 = tg0 + fg.tpg < fg.ntiles ? tg0 + fg.tpg : fg.ntiles;
    const uint32_t share = (tg1 - tg0 + kWWaves - 1) / kWWaves;
    const uint32_t wt0 = tg0 + wave * share < tg1 ? tg0 + wave * share : tg1, wt1 = wt0 + share < tg1 ? wt0 + share : tg1;
    const uint64_t* const slots = w.slots + (uint64_t)b * g.ftiles * kSlots;
    const uint32_t* const tile_cnt = w.tile_cnt + (uint64_t)b * g.ftiles;
    if (threadIdx.x < kCoarse) S.cnt[threadIdx.x] = 0;
    if (threadIdx.x == 0) {
        S.cut = kNoCut;
        u4a wn = wait_window(st, epoch, limit_ticks);  // (the counters are only meaningful once the sample block has cleared them)
        if (wn[3] && !wait_word<4>(line + G_TILES, tg1 - tg0, limit_ticks)) wn[3] = 0u;
        S.win[0] = wn[0]; S.win[1] = wn[1]; S.win[2] = wn[2]; S.win[3] = wn[3];
    }
    __syncthreads();
    if (!S.win[3]) {
        fused_give_up(w, st, out);
        return;
    }
    const uint32_t lo = S.win[0], hi = S.win[1], that_key = S.win[2], wmul = window_mul(lo, hi);
    // ---- the group's candidates, in index order, to LDS ----------------------------------------------------------
    uint32_t own;  // how many there are
    bool in_lds;   // else they are read from the slots, and from dense tiles, whenever they are looked at
    {
        static_assert(kWholeMost <= kWave, "a lane for each tile");
        const uint32_t c0 = lane_id < tg1 - tg0 ? ld_agent(tile_cnt + tg0 + lane_id) : 0u;
        // the first tiles' slots are asked for with the counts (slots past a count are never looked at)
        constexpr int kTilesAtOnce = MANY ? 1 : 4, kAtOnce = MANY ? 6 : 2;
        uint64_t e[kTilesAtOnce][kAtOnce];
        const auto ask = [&](uint32_t t, uint64_t (&to)[kAtOnce]) {
#pragma unroll
            for (int x = 0; x < kAtOnce; x++) to[x] = ld_agent64(slots + (uint64_t)t * kSlots + x * kWave + lane_id);
        };
#pragma unroll
        for (int i = 0; i < kTilesAtOnce; i++) ask(wt0 + i < wt1 ? wt0 + i : tg0, e[i]);
        const uint32_t p0 = wave_inclusive_scan(c0);
        own = (uint32_t)__builtin_amdgcn_readlane((int)p0, kWave - 1);
        in_lds = !__ballot(c0 == kDense) && own <= (uint32_t)kWOwn;
        if (in_lds) {
            const auto keep = [&](uint32_t t, const uint64_t (&from)[kAtOnce]) {
                const int i = (int)(t - tg0);
                const uint32_t cnt = (uint32_t)__builtin_amdgcn_readlane((int)c0, i);
                uint64_t* const to = S.own + ((uint32_t)__builtin_amdgcn_readlane((int)p0, i) - cnt);
#pragma unroll
                for (int x = 0; x < kAtOnce; x++)
                    if ((uint32_t)(x * kWave) + lane_id < cnt) to[x * kWave + lane_id] = from[x];
                if constexpr (MANY) {
#pragma unroll 1
                    for (uint32_t x = kAtOnce * kWave + lane_id; x < cnt; x += kWave) to[x] = ld_agent64(slots + (uint64_t)t * kSlots + x);
                }
            };
#pragma unroll
            for (int i = 0; i < kTilesAtOnce; i++)
                if (wt0 + i < wt1) keep(wt0 + i, e[i]);
#pragma unroll 1
            for (uint32_t t = wt0 + kTilesAtOnce; t < wt1; t++) {
                ask(t, e[0]);
                keep(t, e[0]);
            }
            __syncthreads();
        }
    }
    bool failed = false;
    uint32_t pos = 0;                       // where this wavefront's next pick goes
    uint32_t T = 0, istar = 0;              // picks: key > T, or key == T and index <= istar
    // ---- the candidates are looked at four times: 0 counted per bin, 1 listed by bin, 2 picks counted, 3 picks written
#pragma unroll 1
    for (int pass = 0; pass < 4 && !failed; pass++) {
        // (or the addresses that every pass forms from them would be kept, in registers that are not there)
        uint32_t lane = lane_id, tid = threadIdx.x, first_tile = wt0;
        asm volatile("" : "+v"(lane), "+v"(tid), "+s"(first_tile));
        uint32_t* const cells = pass == 0 ? S.cnt : S.base;
        auto see = [&](bool valid, uint64_t e, bool zeroed) {
            const uint32_t key = key64(e), idx = (uint32_t)e, bitsv = (uint32_t)(e >> 32);
            if (pass < 2) {
                const uint32_t bin = coarse_bin(key, lo, hi, wmul);
                // the top bin, keys >= hi, holds picks for certain as long as the window holds, and has no list
                const uint64_t top = __ballot(valid && bin == (uint32_t)(kCoarse - 1));
                if (top && lane == 0 && pass == 0) atomicAdd(&S.cnt[kCoarse - 1], (uint32_t)__popcll(top));
                if (valid && bin != (uint32_t)(kCoarse - 1)) {
                    const uint32_t at = atomicAdd(&cells[bin], 1u);
                    if (pass == 1 && at < g.lcapb) st_agent64(w.blist + ((uint64_t)b * (kCoarse - 1) + bin) * g.lcapb + at, e);
                }
                return;
            }
            const bool pick = valid && (key > T || (key == T && idx <= istar));
            const uint64_t mk = __ballot(pick);
            if (pass == 3) {
                const uint32_t p = pos + (uint32_t)__popcll(mk & below);
                if (pick && p < k) {  // (p < k whatever the scratch memory held)
                    const u2a pr = {idx, bitsv};
                    *(u2a4*)(out + 1 + 2 * (uint64_t)p) = pr;
                }
                // the streaming block stored 0.0f for key >= predicted threshold: repaired where the prediction was wrong
                if (valid && pick != (zeroed && key >= that_key)) st_agent((uint32_t*)rp + idx, pick ? 0u : bitsv);
            }
            pos += (uint32_t)__popcll(mk);
        };
        if (in_lds) {
            const uint32_t part = ((own + kWWaves - 1) / kWWaves + kWave - 1) / kWave * kWave;  // of a wavefront
            const uint32_t from = part * wave, to = from + part < own ? from + part : own;
#pragma unroll 1
            for (uint32_t i = from; i < to; i += kWave) see(i + lane < to, S.own[i + lane < to ? i + lane : from], true);
        } else {
#pragma unroll 1
            for (uint32_t t = first_tile; t < wt1; t++) {
                const uint32_t cnt = (uint32_t)__builtin_amdgcn_readfirstlane((int)ld_agent(tile_cnt + t));
                if (cnt == kDense) {
                    dense_tile_walk<true, kWWalk>(rp, bn, t, S.dbuf[wave], [&](uint32_t i, uint32_t v, bool in) {
                        see(in && (v & 0x7FFFFFFFu) >= lo, (uint64_t)i | ((uint64_t)v << 32), false);
                    });
                } else {
                    constexpr int kAhead = MANY ? 4 : 2;
                    const uint64_t* l = slots + (uint64_t)t * kSlots;
#pragma unroll 1
                    for (uint32_t i = 0; i < cnt; i += kAhead * kWave) {
                        uint64_t e[kAhead];
#pragma unroll
                        for (int x = 0; x < kAhead; x++) e[x] = ld_agent64(l + (i + x * kWave + lane < cnt ? i + x * kWave + lane : 0u));
#pragma unroll
                        for (int x = 0; x < kAhead; x++)
                            if (i + x * kWave < cnt) see(i + x * kWave + lane < cnt, e[x], true);
                    }
                }
            }
        }
        if (pass == 0) {
            __syncthreads();
            if (tid < kCoarse) {
                // the bucket's count of the bin; what it held before is where this group's entries go in the bin's list
                const uint32_t c = S.cnt[tid];
                S.base[tid] = c ? __hip_atomic_fetch_add(w.bin_fill + (uint64_t)b * kCoarse + tid, c, __ATOMIC_RELAXED,
                                                                 __HIP_MEMORY_SCOPE_AGENT)
                                        : 0u;
            } else if (wave == kCoarse / kWave) {
                // this group's candidates above each bin: lane l takes bins 126 - 2 l and 127 - 2 l
                const u2a c = *(const u2a*)&S.cnt[kCoarse - 2 - 2 * lane];
                const uint32_t inc = wave_inclusive_scan(c[0] + c[1]);
                st_agent64((uint64_t*)(group_above(w, h, b, grp) + kCoarse - 2 - 2 * lane), (uint64_t)(inc - c[0] - c[1]) << 32 | (inc - c[0]));
            }
            __syncthreads();
        } else if (pass == 1) {
            if (!whole_barrier(w, h, b, grp, ng, epoch, &S.flag, limit_ticks)) {
                fused_give_up(w, st, out);
                return;
            }
            // ---- the threshold's bin --------------------------------------------------------------------------------
            // scanned from the top bin downwards: lane l looks at bins 127 - 2 l (tot[1]) and 126 - 2 l (tot[0])
            const uint64_t two = ld_agent64((const uint64_t*)(w.bin_fill + (uint64_t)b * kCoarse + kCoarse - 2 - 2 * lane));
            const u2a tot = {(uint32_t)two, (uint32_t)(two >> 32)};
            const uint32_t inc = wave_inclusive_scan(tot[0] + tot[1]);
            const uint64_t reach = __ballot(inc >= k);
            const int lstar = reach ? __ffsll((long long)reach) - 1 : 0;
            auto at = [&](uint32_t v) { return (uint32_t)__builtin_amdgcn_readlane((int)v, lstar); };
            const uint32_t above_pair = at(inc) - at(tot[0]) - at(tot[1]);  // candidates in the bins above the pair
            const bool in_hi = above_pair + at(tot[1]) >= k;                // the upper bin of the pair reaches k
            const uint32_t jstar = (uint32_t)(kCoarse - 1 - 2 * lstar) - (in_hi ? 0u : 1u);
            const uint32_t n2 = in_hi ? at(tot[1]) : at(tot[0]);                 // its entries
            const uint32_t need = k - above_pair - (in_hi ? 0u : at(tot[1]));    // the picks among them
            // fewer than k candidates; the threshold lies at or above the window's upper end; or more keys share its bin
            // than the list holds (heavy ties, clustered values)
            failed = !reach || jstar == (uint32_t)(kCoarse - 1) || n2 > g.lcapb;
            if (failed) break;
            // certain picks (bins above the threshold's) of the groups before this one
            static_assert(kMaxGroups <= kWThreads, "one thread per group of the bucket");
            uint32_t before = tid < grp ? ld_agent(group_above(w, h, b, tid) + jstar) : 0u;
            // ---- the need-th largest entry of its list by (key, then lower index): radix rounds of 11 bits over both ----
            const uint64_t* const list = w.blist + ((uint64_t)b * (kCoarse - 1) + jstar) * g.lcapb;
            const uint32_t bin_lo = window_bin_lo(lo, wmul, jstar);
            const uint32_t span = window_bin_lo(lo, wmul, jstar + 1) - bin_lo;  // jstar <= kCoarse - 2
            auto order = [&](uint64_t e) { return ((uint64_t)(key64(e) - bin_lo) << 32) | (uint32_t)~(uint32_t)e; };
            uint64_t held[kWList];
#pragma unroll
            for (int j = 0; j < kWList; j++) {
                const uint32_t i = (uint32_t)j * kWThreads + tid;
                held[j] = i < n2 ? ld_agent64(list + i) : 0ull;
            }
#pragma unroll
            for (int j = 0; j < kWList; j++) held[j] = order(held[j]);
            int bits = 32 + (span > 1 ? 32 - __clz((int)(span - 1)) : 0);  // of what is still open
            uint64_t prefix = 0, cut = 0;
            uint32_t want = need, m = n2;
            const uint64_t first_elem = (uint64_t)tg0 * kFTile;
            // 0: a histogram of the next digit; 1: the entries that share the prefix are ranked (entries differ in their
            // index, so that few are left after the last digit at the latest); 2: the picks that lie before this group
            int step = m <= (uint32_t)kWRank ? 1 : 0;
#pragma unroll 1
            for (;;) {
                const int sh = bits > 11 ? bits - 11 : 0;
                if (step == 0) {
                    ((u4a*)S.lh)[tid] = u4a{0u, 0u, 0u, 0u};
                    static_assert(kBins0 == 4 * kWThreads, "cleared by one store each");
                } else if (tid == 0) {
                    S.count = 0;
                }
                __syncthreads();
                auto look = [&](bool valid, uint64_t o) {
                    if (step == 2) {
                        before += valid && o >= cut && (uint64_t)(uint32_t)~(uint32_t)o < first_elem ? 1u : 0u;
                    } else if (valid && (o >> bits) == (prefix >> bits)) {
                        if (step == 0) {
                            atomicAdd(&S.lh[(uint32_t)((o ^ prefix) >> sh)], 1u);
                        } else {
                            const uint32_t i = atomicAdd(&S.count, 1u);
                            if (i < (uint32_t)kWRank) S.list[i] = o;
                        }
                    }
                };
#pragma unroll
                for (int j = 0; j < kWList; j++)
                    if ((uint32_t)j * kWThreads < n2) look((uint32_t)j * kWThreads + tid < n2, held[j]);
#pragma unroll 1
                for (uint32_t i = kWList * kWThreads + tid; i < n2; i += kWThreads) look(true, order(ld_agent64(list + i)));
                if (step == 2) break;
                __syncthreads();
                if (step == 0) {
                    const uint32_t wants[1] = {want};
                    uint32_t anew = threadIdx.x;  // (what is formed from it in the loop would be kept in registers)
                    asm volatile("" : "+v"(anew));
                    sample_pick<kBins0, 1, kWThreads>(S.lh, wants, S.wsum, S.res, anew);
                    const uint32_t bin = S.res[0][0];
                    if (bin >= (uint32_t)kBins0 || bits == 0) {  // the list holds fewer entries than the counts promised, or one of them twice
                        failed = true;
                        break;
                    }
                    want = S.res[0][1];
                    m = S.lh[bin];
                    prefix |= (uint64_t)bin << sh;
                    bits = sh;
                    step = m <= (uint32_t)kWRank ? 1 : 0;
                    __syncthreads();  // the next round clears and writes what was read here
                } else {
                    if (S.count != m) {
                        failed = true;
                        break;
                    }
                    if (tid < m) {
                        const uint64_t me = S.list[tid];
                        if (reaching_entries(S.list, 0, m, me) == want) S.cut = me;
                    }
                    __syncthreads();
                    cut = S.cut;
                    step = 2;
                }
            }
            failed |= cut == kNoCut;  // (an entry twice)
            if (failed) break;
            T = bin_lo + (uint32_t)(cut >> 32);
            istar = ~(uint32_t)cut;
            const uint32_t mine = wave_inclusive_scan(before);
            if (lane == kWave - 1) S.wmine[wave] = mine;
        } else if (pass == 2) {
            if (lane == 0) S.wtot[wave] = pos;
            __syncthreads();
            pos = 0;
#pragma unroll
            for (int i = 0; i < kWWaves; i++) {
                pos += S.wmine[i];
                if (i < wave) pos += S.wtot[i];
            }
        }
    }
    if (failed) {
        // (all of a bucket's blocks come here, for the same reason)
        __syncthreads();
        uint32_t lane = lane_id;
        asm volatile("" : "+v"(lane));
        // what the streaming blocks stored as 0.0f in this group's tiles
        const auto restore = [&] {
#pragma unroll 1
            for (uint32_t t = wt0; t < wt1; t++) {
                const uint32_t cnt = (uint32_t)__builtin_amdgcn_readfirstlane((int)ld_agent(tile_cnt + t));
                if (cnt == kDense) continue;
#pragma unroll 1
                for (uint32_t i = lane; i < cnt; i += kWave) {
                    const uint64_t e = ld_agent64(slots + (uint64_t)t * kSlots + i);
                    if (key64(e) >= that_key) st_agent((uint32_t*)rp + (uint32_t)e, (uint32_t)(e >> 32));
                }
            }
            // the range is read through the caches from here on, by this block alone
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        };
        if (!select_exact_group<kWThreads>(bk, g, w, b, grp, fg, (uint64_t)b << h.shift, restore, S, limit_ticks)) {
            fused_give_up(w, st, out);
            return;
        }
    }
    if (grp == 0 && threadIdx.x == 0) {
        if (!failed) {
            st[S_T] = T;
            st[S_ISTAR] = istar;
            st[S_OK] = 1u;
        }
        if (!ld_agent(st + S_TIMEOUT)) out[0] = k;
    }
}

template <bool MANY>
__global__ __launch_bounds__(kWThreads, 8) void k_topk_whole(WholeBuckets, Geometry g, Workspace w, Whole h, uint32_t epoch, uint32_t published,
                                                             uint64_t limit_ticks) {
    g.listed = 1;  // (known to the compiler)
    const BucketsArg bk = buckets_arg();
    __shared__ WholeLds<MANY> L;
    if (blockIdx.x < g.nbuckets) {
        whole_sample<MANY>(bk, g, w, h, blockIdx.x, published, L);
        return;
    }
    const bool select = blockIdx.x >= h.select_at;
    uint32_t t;
    const auto* const selects = ((const __attribute__((address_space(4))) WholeBuckets*)bk)->select;
    const uint32_t b = listed_bucket(select ? selects : bk->lfirst, blockIdx.x - (select ? h.select_at : g.nbuckets), &t);
    const FusedGeo fg = whole_geo(g, bk, b, h);
    if (select) {
        whole_select<MANY>(bk, g, w, h, b, t, fg, epoch, limit_ticks, L);
        return;
    }
    // the blocks that start together with the sample blocks hold back (stream_hold)
    if (blockIdx.x < h.first_wave)
        for (uint32_t i = 0; i < h.hold; i++) __builtin_amdgcn_s_sleep(8);
    stream_tiles<kWThreads, MANY>(bk, g, w, b, t * kWTiles, fg, h.shift, epoch, limit_ticks, L.a);
}

// Blocks of a launch that fit a CU.
uint64_t whole_per_cu() {
    static const uint64_t per_cu = [] {
        int least = 1 << 20;
        for (const void* k : {(const void*)k_topk_whole<false>, (const void*)k_topk_whole<true>}) {
            int n = 0;
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k, kWThreads, 0) != hipSuccess) n = 0;
            least = n < least ? n : least;
        }
        return (uint64_t)least;
    }();
    return per_cu;
}

}  // namespace

uint64_t whole_limit_on(const StreamShare& share) {
    return waiting_limit(share, whole_per_cu());
}

void launch_whole(const Buckets& call, const Geometry& g, const Workspace& w, uint32_t group_tiles, uint32_t groups_shift, uint32_t epoch,
                  uint32_t published, uint64_t limit_ticks, hipStream_t st) {
    WholeBuckets bk = {call, {}};
    Whole h = {};
    h.tpg = group_tiles;
    h.shift = groups_shift;
    // longest bucket first, each with the blocks that it has
    uint32_t order[kMaxListed], streams = 0, selects = 0;
    longest_first(call, g.nbuckets, order);
    for (uint32_t b = 0; b < g.nbuckets; b++) {
        place_bucket(&bk.b, b, call, order[b], streams);
        bk.select[b] = selects;
        const uint32_t tiles = topk_tiles(bk.b.lcount[b]);
        streams += (tiles + kWTiles - 1) / kWTiles;
        selects += (tiles + group_tiles - 1) / group_tiles;
    }
    for (uint32_t b = g.nbuckets; b < kMaxListed; b++) bk.b.lfirst[b] = bk.select[b] = 0xFFFFFFFFu;
    h.select_at = g.nbuckets + streams;
    h.first_wave = g.nbuckets + (uint32_t)(device_info().num_cus * whole_per_cu());
    h.hold = stream_hold(kWTiles * (uint64_t)streams, g.nbuckets);
    (g.many ? k_topk_whole<true> : k_topk_whole<false>)<<<h.select_at + selects, kWThreads, 0, st>>>(bk, g, w, h, epoch, published, limit_ticks);
}

}  // namespace mcclhip
