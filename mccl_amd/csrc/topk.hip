// Top-k gradient sparsifier with error feedback for gfx950.
//
// Semantics (csrc/compression/TopKCompression.cpp:38-120): per bucket,
// adjusted = grad + residual; the k elements of largest |adjusted| go on the
// wire in ascending index order as [u32 k][k x {u32 index, f32 value}];
// residual = adjusted everywhere except 0.0f at the picks.  Ties at the
// threshold magnitude go to the lower index.
//
// Ordering by fabs() is ordering of the 31-bit pattern `key = bits & 0x7FFFFFFF`
// (NaN patterns sort above infinity), so selection is an exact radix select on
// that key.  All buckets of a gradient run in the same launches.
//
// RESIDENT PATH (topk_resident.hip; one launch): buckets of up to 2 M elements, 2 M a call.
// SINGLE-PASS PATH (one pass over the gradient, 12 B/element of HBM traffic, two launches):
// larger buckets and many buckets at a time; see the section "single-pass path" below.  Lists of middle-sized buckets
// take it in one launch (topk_whole.hip).
// EXACT PATH (any input; six launches): ratios above 12 %, many small buckets,
// and topk_path = 1 (topk_route.h has the rule and its measurements).
//   [pass A]   residual <- grad + residual, histogram of key[30:20]
//   refine x2  histograms of key[19:10], key[9:0] among prefix matches
//   count      per 4096-element tile: #(key > T), #(key == T)
//   emit       an element at index i lands at gt_before(i) + min(eq_before(i),
//              need); ties are accepted while eq_before(i) < need
//   Each kernel first derives the previous round's pick from the finished
//   histogram (every block redundantly; the result is identical), so no
//   separate pick launches are needed.
#include "topk_stream.hip.h"

#include <atomic>
#include <type_traits>
#include <vector>

namespace mcclhip {

namespace {

__global__ __launch_bounds__(kBlock) void k_zero_words(uint32_t* p, uint64_t n) {
    // n is a multiple of 4 and p is 16-byte aligned (see carve())
    u4a* v = (u4a*)p;
    const u4a z = {0u, 0u, 0u, 0u};
    for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < n / 4; i += (uint64_t)gridDim.x * kBlock)
        v[i] = z;
}

// Adds the block's LDS histogram into the bucket's global one (non-empty bins only).
template <int THREADS>
__device__ __forceinline__ void flush_hist(const uint32_t* lds, uint32_t* global, int bins) {
    for (int i = threadIdx.x; i < bins; i += THREADS) {
        uint32_t c = lds[i];
        if (c) atomicAdd(&global[i], c);
    }
}

// ================================ exact path ======================================

// residual <- grad + residual, histogram of key[30:20].
__global__ __launch_bounds__(kBlock) void k_topk_pass_a(const float* __restrict__ grad, float* residual,
                                                        Geometry g, Workspace w) {
    __shared__ uint32_t lh[kBins0];
    for (int i = threadIdx.x; i < kBins0; i += kBlock) lh[i] = 0;
    __syncthreads();
    const uint32_t b = blockIdx.y;
    const uint64_t bn = bucket_count(g, b);
    const float* gp = grad + (uint64_t)b * g.bucket_elems;
    float* rp = residual + (uint64_t)b * g.bucket_elems;
    const uint64_t nvec = bn / 4;
    constexpr int U = 2;
    const uint64_t tile = (uint64_t)kBlock * U;
    for (uint64_t base = (uint64_t)blockIdx.x * tile; base < nvec; base += (uint64_t)gridDim.x * tile) {
        u4a gv[U], rv[U];
        uint64_t idx[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            idx[u] = base + (uint64_t)u * kBlock + threadIdx.x;
            if (idx[u] < nvec) {
                gv[u] = *(const u4u4*)(gp + idx[u] * 4);
                rv[u] = *(const u4u4*)(rp + idx[u] * 4);
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (idx[u] < nvec) {
                u4a a;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    float adj = u2f(gv[u][q]) + u2f(rv[u][q]);
                    a[q] = f2u(adj);
                    atomicAdd(&lh[key_of(adj) >> 20], 1u);
                }
                *(u4u4*)(rp + idx[u] * 4) = a;
            }
        }
    }
    const uint64_t gtid = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (gtid < 4 && nvec * 4 + gtid < bn) {
        const uint64_t i = nvec * 4 + gtid;
        float adj = gp[i] + rp[i];
        rp[i] = adj;
        atomicAdd(&lh[key_of(adj) >> 20], 1u);
    }
    __syncthreads();
    flush_hist<kBlock>(lh, w.hist + (uint64_t)b * kHistWords, kBins0);
    if (blockIdx.x == 0 && threadIdx.x == 0) w.state[(uint64_t)b * kStateWords + S_EXACT_HIST] = 1;
}

// Derives (prefix, remaining) after `rounds_done` rounds for bucket b from the
// finished histograms; block (0, b) also records them in the state.
__device__ __forceinline__ void exact_prefix(const Geometry& g, const Workspace& w, uint32_t b, int rounds_done,
                                             bool record, uint32_t* prefix, uint32_t* remaining,
                                             uint32_t* scratch) {
    const uint32_t* h = w.hist + (uint64_t)b * kHistWords;
    uint32_t* st = w.state + (uint64_t)b * kStateWords;
    uint32_t p = 0, r = bucket_k(g, b);
    if (rounds_done >= 1) {
        uint32_t left;
        const uint32_t bin = pick_bin<kBins0, kBlock>(h, r, 0, &left, scratch);
        p = bin << 20;
        r = left;
        if (record && rounds_done == 1 && threadIdx.x == 0) { st[S_P0] = p; st[S_R0] = r; }
    }
    if (rounds_done >= 2) {
        uint32_t left;
        const uint32_t bin = pick_bin<kBinsR, kBlock>(h + kBins0, r, 0, &left, scratch);
        p |= bin << 10;
        r = left;
        if (record && rounds_done == 2 && threadIdx.x == 0) { st[S_P1] = p; st[S_R1] = r; }
    }
    if (rounds_done >= 3) {
        uint32_t left;
        const uint32_t bin = pick_bin<kBinsR, kBlock>(h + kBins0 + kBinsR, r, 0, &left, scratch);
        p |= bin;
        r = left;
        if (record && threadIdx.x == 0) { st[S_T] = p; st[S_NEED] = r; }
    }
    *prefix = p;
    *remaining = r;
}

// round 0: full histogram of key[30:20] (only for buckets the fast path gave up on);
// round 1 / 2: histogram of the next 10 key bits among elements matching the prefix.
__global__ __launch_bounds__(kBlock) void k_topk_refine(const float* residual, Geometry g, Workspace w,
                                                        int round, int only_failed) {
    __shared__ uint32_t lh[kBins0];
    __shared__ uint32_t scratch[kBlock / kWave + 2];
    const uint32_t b = blockIdx.y;
    const uint32_t* st = w.state + (uint64_t)b * kStateWords;
    if (only_failed && st[S_OK]) return;
    if (round == 0 && st[S_EXACT_HIST]) return;
    const int bins = round == 0 ? kBins0 : kBinsR;
    for (int i = threadIdx.x; i < bins; i += kBlock) lh[i] = 0;
    uint32_t prefix = 0, remaining = 0;
    if (round > 0) exact_prefix(g, w, b, round, blockIdx.x == 0, &prefix, &remaining, scratch);
    __syncthreads();
    const uint64_t bn = bucket_count(g, b);
    const float* rp = residual + (uint64_t)b * g.bucket_elems;
    const int shift = round == 0 ? 20 : (round == 1 ? 10 : 0);
    const int hi_shift = round == 0 ? 31 : shift + 10;
    const uint32_t want = round == 0 ? 0u : prefix >> hi_shift;
    const uint32_t mask = (uint32_t)bins - 1u;
    const uint64_t nvec = bn / 4;
    constexpr int U = 4;
    const uint64_t tile = (uint64_t)kBlock * U;
    for (uint64_t base = (uint64_t)blockIdx.x * tile; base < nvec; base += (uint64_t)gridDim.x * tile) {
        u4a v[U];
        uint64_t idx[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            idx[u] = base + (uint64_t)u * kBlock + threadIdx.x;
            if (idx[u] < nvec) v[u] = *(const u4u4*)(rp + idx[u] * 4);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (idx[u] < nvec) {
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const uint32_t key = v[u][q] & 0x7FFFFFFFu;
                    if ((key >> hi_shift) == want) atomicAdd(&lh[(key >> shift) & mask], 1u);
                }
            }
        }
    }
    const uint64_t gtid = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (gtid < 4 && nvec * 4 + gtid < bn) {
        const uint32_t key = key_of(rp[nvec * 4 + gtid]);
        if ((key >> hi_shift) == want) atomicAdd(&lh[(key >> shift) & mask], 1u);
    }
    __syncthreads();
    const int off = round == 0 ? 0 : (round == 1 ? kBins0 : kBins0 + kBinsR);
    flush_hist<kBlock>(lh, w.hist + (uint64_t)b * kHistWords + off, bins);
}

// Four consecutive elements of a tile; elements past the bucket end are invalid.
struct Quad {
    uint32_t bits[4];
    bool valid[4];
    uint64_t e;  // bucket-relative index of bits[0]
};

__device__ __forceinline__ Quad load_quad(const float* rp, uint64_t bn, uint32_t t, int it) {
    Quad q;
    q.e = (uint64_t)t * kTile + (uint64_t)it * (kBlock * 4) + (uint64_t)threadIdx.x * 4;
    if (q.e + 4 <= bn) {
        u4a v = *(const u4u4*)(rp + q.e);
#pragma unroll
        for (int j = 0; j < 4; j++) { q.bits[j] = v[j]; q.valid[j] = true; }
    } else {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            q.valid[j] = q.e + j < bn;
            q.bits[j] = q.valid[j] ? f2u(rp[q.e + j]) : 0u;
        }
    }
    return q;
}

__global__ __launch_bounds__(kBlock) void k_topk_count(const float* residual, Geometry g, Workspace w,
                                                       int only_failed) {
    __shared__ uint32_t scratch[kBlock / kWave + 2];
    const uint32_t b = blockIdx.y;
    if (only_failed && w.state[(uint64_t)b * kStateWords + S_OK]) return;
    const uint64_t bn = bucket_count(g, b);
    const float* rp = residual + (uint64_t)b * g.bucket_elems;
    uint32_t T, need;
    exact_prefix(g, w, b, 3, blockIdx.x == 0, &T, &need, scratch);
    for (uint32_t t = blockIdx.x; t < g.tiles; t += gridDim.x) {
        uint32_t packed = 0;  // gt in the low half, eq in the high half (each <= 4096)
        if ((uint64_t)t * kTile < bn) {
#pragma unroll
            for (int it = 0; it < kTile / (kBlock * 4); it++) {
                Quad q = load_quad(rp, bn, t, it);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const uint32_t key = q.bits[j] & 0x7FFFFFFFu;
                    if (q.valid[j]) packed += (key > T ? 1u : 0u) + (key == T ? 0x10000u : 0u);
                }
            }
        }
        uint32_t total;
        block_exclusive_scan(packed, scratch, &total);
        if (threadIdx.x == 0) {
            w.tile_gt[(uint64_t)b * g.tiles + t] = total & 0xFFFFu;
            w.tile_eq[(uint64_t)b * g.tiles + t] = total >> 16;
        }
    }
}

__global__ __launch_bounds__(kBlock) void k_topk_emit(float* residual, Geometry g, Workspace w,
                                                      uint8_t* wire, uint64_t wire_stride, int only_failed) {
    __shared__ uint32_t smem[kBlock / kWave + 2];
    const uint32_t b = blockIdx.y;
    const uint32_t* st = w.state + (uint64_t)b * kStateWords;
    if (only_failed && st[S_OK]) return;
    const uint64_t bn = bucket_count(g, b);
    uint32_t* out = (uint32_t*)(wire + (uint64_t)b * wire_stride);
    if (blockIdx.x == 0 && threadIdx.x == 0) out[0] = bucket_k(g, b);
    float* rp = residual + (uint64_t)b * g.bucket_elems;
    const uint32_t T = st[S_T];
    const uint32_t need = st[S_NEED];
    const uint32_t* tgt = w.tile_gt + (uint64_t)b * g.tiles;
    const uint32_t* teq = w.tile_eq + (uint64_t)b * g.tiles;
    for (uint32_t t = blockIdx.x; t < g.tiles; t += gridDim.x) {
        if ((uint64_t)t * kTile >= bn) break;
        // picks before this tile: sum of the counts of all earlier tiles
        uint32_t sg = 0, se = 0;
        for (uint32_t i = threadIdx.x; i < t; i += kBlock) { sg += tgt[i]; se += teq[i]; }
        uint32_t gt_run, eq_run;
        block_exclusive_scan(sg, smem, &gt_run);
        block_exclusive_scan(se, smem, &eq_run);
#pragma unroll 1
        for (int it = 0; it < kTile / (kBlock * 4); it++) {
            Quad q = load_quad(rp, bn, t, it);
            uint32_t packed = 0;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t key = q.bits[j] & 0x7FFFFFFFu;
                if (q.valid[j]) packed += (key > T ? 1u : 0u) + (key == T ? 0x10000u : 0u);
            }
            uint32_t total;
            const uint32_t ex = block_exclusive_scan(packed, smem, &total);
            uint32_t gt_b = gt_run + (ex & 0xFFFFu);
            uint32_t eq_b = eq_run + (ex >> 16);
            if (packed) {
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const uint32_t key = q.bits[j] & 0x7FFFFFFFu;
                    const bool is_gt = q.valid[j] && key > T;
                    const bool is_eq = q.valid[j] && key == T;
                    if (is_gt || (is_eq && eq_b < need)) {
                        const uint32_t pos = gt_b + (eq_b < need ? eq_b : need);
                        out[1 + 2 * (uint64_t)pos] = (uint32_t)(q.e + j);
                        out[2 + 2 * (uint64_t)pos] = q.bits[j];
                        rp[q.e + j] = 0.0f;
                    }
                    gt_b += is_gt ? 1u : 0u;
                    eq_b += is_eq ? 1u : 0u;
                }
            }
            gt_run += total & 0xFFFFu;
            eq_run += total >> 16;
        }
    }
}

// ================================ single-pass path ==================================
// Two launches.
//
// k_topk_stream - blocks of the 1D grid, in dispatch order:
//   sample blocks   one per bucket, the first blocks of the grid.  8192 evenly spread
//                   elements of grad + residual -> the candidate window [lo, hi) and the
//                   predicted threshold; the block clears the bucket's counters and then
//                   publishes the call's epoch number in S_READY.
//   then, segment by segment (segment s = the tiles of bucket s, then the bin blocks of
//   bucket s - 1; the bin blocks of the last bucket close the grid):
//   (The buckets of a list go longest first, each with the blocks it has.  24 buckets of 1001 to 1.5 M elements,
//   5.5 M together, 1 %: as many blocks for each as for the longest, streaming blocks and select launches chosen by
//   that number, 50.5 us; so, 37.6.)
//   streaming blocks one per 4096-element tile, in address order.  A wavefront loads its
//                   1024 elements, waits until the bucket's S_READY shows the epoch, stores
//                   residual <- grad + residual (0.0f at or above the predicted threshold)
//                   and stages its candidates (key >= lo) in LDS in index order; the block
//                   writes them to the tile's slots and counts itself into its group of
//                   tiles (topk_groups of them per bucket).
//   bin blocks      one per group.  Block g waits until group g's tiles are finished (when it
//                   is dispatched - one bucket later - they are, except in the last bucket),
//                   counts the group's candidates per coarse window bin (128 bins), publishes
//                   the counts and copies the candidates, binned, to the bucket's per-bin
//                   lists.  It waits for nothing else.
// k_topk_select - one block per group; nothing crosses blocks any more: every block
//                   redundantly finds the bin that holds the k-th largest key (from the
//                   groups' counts), the exact threshold and the tie rule (from that bin's
//                   list) and the number of picks in the groups before its own, then writes
//                   its group's picks, in index order, at that offset of the payload and
//                   repairs the residual where the predicted threshold and the true one
//                   disagree.  A failed selection (threshold outside the window, a bin list
//                   overflow) hands the bucket to the exact selection, run by the bucket's
//                   blocks together through counter barriers; a launch covers at most 1024
//                   blocks, so that all of them are resident at the same time.
//
// Progress in k_topk_stream.  The hardware deals the blocks of a grid to the XCDs round-robin
// and every XCD dispatches its share in grid order.  A streaming block waits only for its
// bucket's sample block, which precedes every streaming block in the grid.  A bin block waits
// only for streaming blocks that precede it in the grid.  Nothing waits for a later block.
// (Variants in which blocks of the streaming launch also performed the selection were built
// and measured: with the streaming block that finishes a group last going on as the group's
// emitter, the slowest XCD collects every emitter, slows down further and jams; with
// dedicated selection blocks in the grid nothing jams, but every dependent memory round trip
// of the selection takes 5 to 8 microseconds while the stream is in flight, the blocks live
// 50 to 100 microseconds each, and the stream loses a quarter of its block slots to them.
// With every bucket's selection blocks at the very end of the grid the launch boundary
// disappears, but the kernel then carries the selection's registers: at 125 registers four
// blocks fit a CU instead of six and the stream - whose blocks idle while their stores are
// acknowledged - takes 15.3 microseconds per bucket instead of 11.8; trimmed to 89 registers
// it streams at 12.6, while the bin blocks' lists and counts have to be written through
// (scattered 8-byte stores, a memory transaction each: 10 microseconds per call; an L2
// write-back per bin block instead costs 380) and every selection block reads its bucket's
// list past its L2.  Whole call 228 microseconds against 221 for the two launches.  Two tiles
// per streaming block, the second tile's loads under way while the first tile's stores are
// acknowledged, stream slower as well: 220 against 205 microseconds.)
// All waits are bounded all the same (`limit_ticks`): a block that gives up sets S_TIMEOUT,
// overwrites the bucket's payload header with kPoisonK and leaves; k_topk_select leaves such
// a bucket alone.
//
// Everything that crosses blocks inside a launch is written and read with agent-scope
// accesses (the XCDs' L2 caches are not coherent for plain ones), and a writer waits for
// its stores' acknowledgements before it signals.

template <int THREADS, bool MANY>
struct StreamLds {
    static constexpr int kWaves = StreamShape<THREADS>::kWaves;
    union {
        SampleLds<THREADS> s;  // sample block
        StreamBlockLds<kWaves, TileShape<MANY>::kStage> a;
        struct {  // bin block
            uint32_t dbuf[kWaves][16 * kWave];  // dense_tile_walk's staging area, one per wavefront
            uint32_t cnt[kCoarse];
            uint32_t base[kCoarse];
            uint32_t win[4];
        } e;
    };
};
struct SelectLds {
    uint32_t lh[kBins0] __attribute__((aligned(16)));  // radix rounds, tie-break, exact fallback
    uint32_t dbuf[kFWaves][16 * kWave];  // dense_tile_walk's staging area, one per wavefront
    uint32_t wsum[kBlock / kWave];
    uint32_t res[1][2];
    uint32_t rcnt[kFWaves][kHeld];
    uint32_t wtot[kFWaves];
    uint32_t scratch[kBlock / kWave + 2];
    uint32_t flag;
};

// The bucket's candidate window; clears what the launches accumulate into, then publishes the
// window and the epoch with one store.
template <int THREADS, class Lds>
__device__ __forceinline__ void fused_sample(BucketsArg bk, const Geometry& g, const Workspace& w, uint32_t b,
                                             uint32_t epoch, Lds& L) {
    const FusedGeo fg = fused_geo(g, bk, b);
    uint32_t* st = w.state + (uint64_t)b * kStateWords;
    const SampleWindow win = sample_window<THREADS>(bucket_grad(g, bk, b), bucket_residual(g, bk, b), fg.bn, fg.k, L.s, [&] {
        // (the acknowledgements are back long before the window is published)
        if (threadIdx.x >> g.gshift == 0) st_agent(w.grp_cnt + (((uint64_t)b << g.gshift) + threadIdx.x) * kCntStride, 0u);
        if (threadIdx.x < kCoarse) st_agent(w.bin_fill + (uint64_t)b * kCoarse + threadIdx.x, 0u);
        if (threadIdx.x == 0) {
            st_agent(st + S_OK, 0u);
            st_agent(st + S_TIMEOUT, 0u);
            st_agent(st + S_BARF, 0u); st_agent(st + S_BARF + 1, 0u); st_agent(st + S_BARF + 2, 0u); st_agent(st + S_BARF + 3, 0u);
        }
    });
    if (threadIdx.x == 0) {
        // every store above must have arrived before the window is published
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        store16_agent(st + S_LO_KEY, u4a{win.lo, win.hi, win.that, epoch});
    }
    // off the critical path: the histograms of the exact selection, should the select launch need it
    for (int i = threadIdx.x; i < kHistWords; i += THREADS) w.hist[(uint64_t)b * kHistWords + i] = 0u;
}

// ---- bin block -----------------------------------------------------------------------------
template <int THREADS, bool MANY>
__device__ __forceinline__ void fused_bin(BucketsArg bk, const Geometry& g, const Workspace& w, uint32_t b,
                                          uint32_t grp, const FusedGeo& fg, uint32_t epoch, uint64_t limit_ticks,
                                          StreamLds<THREADS, MANY>& L) {
    uint32_t* st = w.state + (uint64_t)b * kStateWords;
    // the group's tiles are finished: all its streaming blocks have arrived
    {
        const uint32_t tg0 = grp * fg.tpg;
        const uint32_t in_group = (tg0 + fg.tpg < fg.ntiles ? tg0 + fg.tpg : fg.ntiles) - tg0;
        // the counter is only meaningful once the sample block has cleared it
        if (threadIdx.x == 0) {
            u4a wn = wait_window(st, epoch, limit_ticks);
            if (wn[3] && !wait_word(w.grp_cnt + (((uint64_t)b << g.gshift) + grp) * kCntStride, in_group, limit_ticks)) wn[3] = 0u;
            L.e.win[0] = wn[0]; L.e.win[1] = wn[1]; L.e.win[2] = wn[2]; L.e.win[3] = wn[3];
        }
        __syncthreads();
        if (!L.e.win[3]) {
            fused_give_up(w, st, bucket_wire(g, bk, b));
            return;
        }
    }
    const uint32_t lo = L.e.win[0], hi = L.e.win[1], wmul = window_mul(L.e.win[0], L.e.win[1]);
    const uint64_t bn = fg.bn;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const float* rp = bucket_residual(g, bk, b);
    typedef StreamShape<THREADS> Shape;
    std::conditional_t<MANY, ManyTiles<kAgent, Shape::kWaves>, GroupTiles<kAgent, Shape::kWaves, Shape::kHeld>> G;
    G.load(g, w, b, grp, fg);
    // candidates per coarse bin
    if (threadIdx.x < kCoarse) L.e.cnt[threadIdx.x] = 0;
    static_assert(kCoarse <= THREADS, "one thread per coarse bin");
    __syncthreads();
    G.sweep([&](uint32_t, uint32_t, uint32_t cnt, uint64_t a0, uint64_t a1) {
                if ((uint32_t)lane < cnt) atomicAdd(&L.e.cnt[coarse_bin(key64(a0), lo, hi, wmul)], 1u);
                if ((uint32_t)(kWave + lane) < cnt) atomicAdd(&L.e.cnt[coarse_bin(key64(a1), lo, hi, wmul)], 1u);
            },
            [&](uint32_t, uint32_t t) {
                dense_tile_walk<true>(rp, bn, t, L.e.dbuf[wave], [&](uint32_t, uint32_t v, bool in) {
                    const uint32_t key = v & 0x7FFFFFFFu;
                    const bool cand = in && key >= lo;
                    wave_hist_add(L.e.cnt, cand, cand ? coarse_bin(key, lo, hi, wmul) : 0u);
                });
            });
    __syncthreads();
    if (threadIdx.x < kCoarse) {
        // the bucket's count per bin; what it held before is where this group's entries go in the
        // bin's list (the top bin, keys >= hi, holds picks for certain as long as the window holds
        // and has no list)
        const uint32_t c = L.e.cnt[threadIdx.x];
        L.e.base[threadIdx.x] = c ? __hip_atomic_fetch_add(w.bin_fill + (uint64_t)b * kCoarse + threadIdx.x, c,
                                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                                  : 0u;
    }
    if (wave == 0) {
        // this group's candidates above each bin: lane l takes bins 127 - 2 l and 126 - 2 l
        const uint32_t c_hi = L.e.cnt[kCoarse - 1 - 2 * lane], c_lo = L.e.cnt[kCoarse - 2 - 2 * lane];
        const uint32_t inc = wave_inclusive_scan(c_hi + c_lo);
        uint32_t* col = w.gsuf + (((uint64_t)b * kCoarse) << g.gshift) + grp;
        col[(uint64_t)(kCoarse - 1 - 2 * lane) << g.gshift] = inc - c_hi - c_lo;
        col[(uint64_t)(kCoarse - 2 - 2 * lane) << g.gshift] = inc - c_lo;
    }
    __syncthreads();
    // binned copies (read by the next launch: plain stores)
    uint64_t* bl = w.blist + (uint64_t)b * (kCoarse - 1) * g.lcapb;
    auto put = [&](bool valid, uint32_t cb, uint64_t e) {
        if (valid && cb < (uint32_t)(kCoarse - 1)) {
            const uint32_t pos = atomicAdd(&L.e.base[cb], 1u);
            if (pos < g.lcapb) bl[(uint64_t)cb * g.lcapb + pos] = e;
        }
    };
    G.sweep([&](uint32_t, uint32_t, uint32_t cnt, uint64_t a0, uint64_t a1) {
                put((uint32_t)lane < cnt, coarse_bin(key64(a0), lo, hi, wmul), a0);
                put((uint32_t)(kWave + lane) < cnt, coarse_bin(key64(a1), lo, hi, wmul), a1);
            },
            [&](uint32_t, uint32_t t) {
                dense_tile_walk<true>(rp, bn, t, L.e.dbuf[wave], [&](uint32_t i, uint32_t v, bool in) {
                    const uint32_t key = v & 0x7FFFFFFFu;
                    const bool cand = in && key >= lo;
                    put(cand, cand ? coarse_bin(key, lo, hi, wmul) : 0u, (uint64_t)i | ((uint64_t)v << 32));
                });
            });
}

// ---- the streaming launch ------------------------------------------------------------------
// LISTED: the call's buckets are a list (g.listed), known to the compiler: a block finds its work before it can
// load, and one kernel for both layouts kept 13 more scalar registers in vector lanes (the 96.5 M gradient 2.5 us).
template <int THREADS, bool LISTED, bool MANY>
__global__ __launch_bounds__(THREADS, StreamShape<THREADS>::kPerSimd) void k_topk_stream(Buckets, Geometry g, Workspace w, uint32_t epoch,
                                                        uint32_t published, uint32_t first_wave, uint32_t hold,
                                                        uint64_t limit_ticks) {
    g.listed = LISTED;
    const BucketsArg bk = buckets_arg();
    constexpr uint32_t kTiles = StreamShape<THREADS>::kTiles;
    __shared__ StreamLds<THREADS, MANY> L;
    if (blockIdx.x < g.nbuckets) {
        fused_sample<THREADS>(bk, g, w, blockIdx.x, published, L);
        return;
    }
    // segment s of the grid: the tiles of bucket s, then the bin blocks of bucket s - 1 (whose
    // tiles are finished or about to be by then: a bin block that is dispatched early only
    // polls); after the last segment the bin blocks of the last bucket
    const uint32_t j = blockIdx.x - g.nbuckets;
    uint32_t b, t;
    bool emit = false;
    if constexpr (LISTED) {
        b = listed_bucket(bk->lfirst, j, &t);
        const uint32_t sblocks = (topk_tiles(bk->lcount[b]) + kTiles - 1) / kTiles;
        if (t >= sblocks) {
            t -= sblocks;
            emit = true;
            if (b) {
                const uint32_t before = topk_groups(topk_tiles(bk->lcount[b - 1]), g.gshift);
                if (t < before) b -= 1;
                else t -= before;
            }
        }
    } else {
        const uint32_t sblocks = (g.ftiles + kTiles - 1) / kTiles;
        const uint32_t per = sblocks + g.ngroups;
        b = j / per;
        t = j - b * per;
        if (b >= g.nbuckets) {
            t = j - g.nbuckets * per;
            b = g.nbuckets - 1;
            emit = true;
        } else if (t >= sblocks) {
            if (b == 0) return;
            t -= sblocks;
            b -= 1;
            emit = true;
        }
    }
    const FusedGeo fg = fused_geo(g, bk, b);
    if (emit) {
        if (t < fg.ng) fused_bin<THREADS, MANY>(bk, g, w, b, t, fg, epoch, limit_ticks, L);
        return;
    }
    if (t * kTiles >= fg.ntiles) return;
    // The blocks that start together with the sample blocks hold back (stream_hold).
    if (blockIdx.x < first_wave)
        for (uint32_t i = 0; i < hold; i++) __builtin_amdgcn_s_sleep(8);
    stream_tiles<THREADS, MANY>(bk, g, w, b, t * kTiles, fg, g.gshift, epoch, limit_ticks, L.a);
}

// ---- the select launch ----------------------------------------------------------------------
// blockIdx.x = group, blockIdx.y = bucket - first_bucket; of a list, blocks of all its buckets in a row
// (Buckets::lfirst).  Everything the streaming launch
// left behind is read with plain loads; only the exact fallback talks across blocks.
template <bool LISTED, bool MANY>
__global__ __launch_bounds__(kBlock, 4) void k_topk_select(Buckets, Geometry g, Workspace w, uint32_t first_bucket,
                                                           uint64_t limit_ticks) {
    g.listed = LISTED;
    const BucketsArg bk = buckets_arg();
    __shared__ SelectLds L;
    uint32_t b = first_bucket + blockIdx.y, grp = blockIdx.x;
    if (g.listed) b = listed_bucket(bk->lfirst, blockIdx.x, &grp);
    const FusedGeo fg = fused_geo(g, bk, b);
    if (grp * fg.tpg >= fg.ntiles) return;  // (no division on the way to the first loads)
    uint32_t* st = w.state + (uint64_t)b * kStateWords;
    uint32_t* out = bucket_wire(g, bk, b);
    // Every load of the first round trip is issued before the first value is looked at, the small
    // ones first: loads complete in order, and the threshold bin is found (and its list requested)
    // while the group's slots are still arriving.
    const u4a win = *(const u4a*)(st + S_LO_KEY);
    const uint32_t gave_up = st[S_TIMEOUT];
    static_assert(kBinsPerLane == 2, "a lane owns two neighbouring bins");
    // scanned from the top bin downwards: lane l looks at bins 127 - 2 l (tot[1]) and 126 - 2 l (tot[0])
    const u2a tot = *(const u2a*)(w.bin_fill + (uint64_t)b * kCoarse + kCoarse - 2 - 2 * (threadIdx.x & (kWave - 1)));
    std::conditional_t<MANY, ManyTiles<kEarlier, kFWaves>, GroupTiles<kEarlier, kFWaves, kHeld>> G;
    G.load(g, w, b, grp, fg);
    // a replay of a captured launch carries the same epoch: also behind a run that was given up
    if (grp == 0 && threadIdx.x == 0) st[S_READY] = 0u;
    if (gave_up) return;  // the streaming launch gave the bucket up: its payload header says so
    const uint32_t lo = win[0], that_key = win[2];
    const uint32_t k = fg.k;
    const uint64_t bn = fg.bn;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const uint64_t below = (1ull << lane) - 1ull;
    float* rp = bucket_residual(g, bk, b);

    bool failed = false;
    do {
    // ---- 3: threshold bin from the bucket's counts ------------------------------------------
    const uint32_t inc = wave_inclusive_scan(tot[0] + tot[1]);
    const uint64_t reach = __ballot(inc >= k);
    if (!reach) {  // fewer than k candidates
        failed = true;
        break;
    }
    const int lstar = __ffsll((long long)reach) - 1;
    auto at_lstar = [&](uint32_t v) { return (uint32_t)__builtin_amdgcn_readlane((int)v, lstar); };
    const uint32_t pair_hi = at_lstar(tot[1]), pair_lo = at_lstar(tot[0]);
    const uint32_t above_pair = at_lstar(inc) - pair_hi - pair_lo;  // candidates in the bins above the pair
    const bool in_hi = above_pair + pair_hi >= k;                                     // the upper bin of the pair reaches k
    const uint32_t jstar = (uint32_t)(kCoarse - 1 - 2 * lstar) - (in_hi ? 0u : 1u);
    if (jstar == (uint32_t)(kCoarse - 1)) {  // the threshold lies at or above the window's upper end
        failed = true;
        break;
    }
    const uint32_t n2 = in_hi ? pair_hi : pair_lo;                     // candidates in the threshold bin
    const uint32_t above_total = above_pair + (in_hi ? 0u : pair_hi);
    const uint32_t need = k - above_total;                              // picks inside the bin, 1..n2
    // certain picks (bins above the threshold bin) in the groups before this one: requested now,
    // summed when the bin's list has been requested as well
    const uint32_t ab = threadIdx.x < grp ? w.gsuf[(((uint64_t)b * kCoarse + jstar) << g.gshift) + threadIdx.x] : 0u;
    if (n2 > g.lcapb) {  // more keys in the threshold bin than its list holds (heavy ties, clustered values)
        failed = true;
        break;
    }

    // ---- 4: exact threshold from the bin's list ---------------------------------------------
    const uint64_t* l2 = w.blist + ((uint64_t)b * (kCoarse - 1) + jstar) * g.lcapb;
    // The need-th largest entry by (key, then lower index): rounds of 10 bits over both until few entries share the
    // prefix, and these are ranked by each wavefront for itself.  Most lists take one round (3500 entries over up to 1024
    // digits), and ties need no search of their own.  With rounds over the whole key, of 1.3 us each, and searches for ties
    // and for the group's place behind them a bucket of 6.5 M elements took 32.9 us, and 30.9 this way.
    // the first 4096 entries stay in registers (a bin of the expected width holds about 3500)
    constexpr int kL2Regs = 16;
    uint64_t ent[kL2Regs];
#pragma unroll
    for (int j = 0; j < kL2Regs; j++) {
        const uint32_t i = (uint32_t)j * kBlock + threadIdx.x;
        ent[j] = l2[i < n2 ? i : n2 - 1];  // (n2 >= need >= 1)
    }
    // (the bin's bounds take three divisions: made while the entries are on their way, with the first bound of the
    // window hidden until here, as the compiler would make them before; 30.9 us -> 30.6)
    uint32_t wlo = lo;
    asm volatile("" : "+s"(wlo));
    const uint32_t wmul = window_mul(wlo, win[1]);
    const uint32_t bin_lo = window_bin_lo(wlo, wmul, jstar);  // smallest key of the threshold bin
    const uint32_t bin_span = window_bin_lo(wlo, wmul, jstar + 1) - bin_lo;  // jstar <= kCoarse - 2
    const uint32_t last = (uint32_t)(bn - 1);
    const int index_bits = 32 - __clz((int)last);
    auto order = [&](uint64_t e) { return ((uint64_t)(key64(e) - bin_lo) << index_bits) | (last - (uint32_t)e); };
    // past the list's end: shares no prefix, and lies before no group
#pragma unroll
    for (int j = 0; j < kL2Regs; j++) ent[j] = (uint32_t)j * kBlock + threadIdx.x < n2 ? order(ent[j]) : 1ull << 63;
    auto for_list2 = [&](auto&& body) {
#pragma unroll
        for (int j = 0; j < kL2Regs; j++)
            if ((uint32_t)j * kBlock < n2) body(ent[j]);
#pragma unroll 1
        for (uint32_t i = kL2Regs * kBlock + threadIdx.x; i < n2; i += kBlock) body(order(l2[i]));
    };
    uint32_t* lh = L.lh;
    uint64_t* const few = (uint64_t*)(lh + kBinsR);  // the entries to rank
    uint32_t* const nfew = lh + kBinsR + 2 * kWave;
    int bits = index_bits + (bin_span > 1 ? 32 - __clz((int)(bin_span - 1)) : 0);  // of the entries still open
    uint64_t prefix = 0;
    uint32_t want = need, m = n2;
    if (threadIdx.x == 0) *nfew = 0;
#pragma unroll 1
    while (m > (uint32_t)kWave && !failed) {  // block-uniform
        const int sh = bits > 10 ? bits - 10 : 0;
        ((u4a*)lh)[threadIdx.x] = u4a{0u, 0u, 0u, 0u};
        static_assert(kBinsR == 4 * kBlock, "cleared by one store each");
        __syncthreads();
        for_list2([&](uint64_t o) {
            if ((o >> bits) == (prefix >> bits)) atomicAdd(&lh[(uint32_t)((o ^ prefix) >> sh)], 1u);
        });
        __syncthreads();
        const uint32_t wants[1] = {want};
        sample_pick<kBinsR, 1, kBlock>(lh, wants, L.wsum, L.res);
        const uint32_t bin = L.res[0][0];
        want = L.res[0][1];
        // the list holds fewer entries than the counts promised, or one of them twice
        failed = bin >= (uint32_t)kBinsR || bits == 0;
        if (!failed) m = lh[bin];
        prefix |= (uint64_t)bin << sh;
        bits = sh;
        __syncthreads();  // the next round clears and writes what was read here
    }
    if (failed) break;
    if (m == n2) __syncthreads();  // (no round was taken)
    for_list2([&](uint64_t o) {
        if ((o >> bits) == (prefix >> bits)) {
            const uint32_t i = atomicAdd(nfew, 1u);
            if (i < (uint32_t)kWave) few[i] = o;
        }
    });
    __syncthreads();
    if (*nfew != m) {
        failed = true;
        break;
    }
    uint64_t cut;  // the last pick
    {
        const uint64_t mine = few[lane];
        const int at = __ffsll((long long)__ballot((uint32_t)lane < m && reaching_entries(few, 0, m, mine) == want)) - 1;
        if (at < 0) {  // (an entry twice)
            failed = true;
            break;
        }
        cut = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(mine >> 32), at) << 32 |
              (uint32_t)__builtin_amdgcn_readlane((int)mine, at);
    }
    const uint32_t T = bin_lo + (uint32_t)(cut >> index_bits);
    const uint32_t istar = last - (uint32_t)(cut & ((1ull << index_bits) - 1));
    auto is_pick = [&](bool valid, uint32_t key, uint32_t idx) {
        return valid && (key > T || (key == T && idx <= istar));
    };
    // the picks at indices below this group's first element
    const uint32_t from_end = last - G.t0 * (uint32_t)kFTile;  // what `last - index` exceeds there
    uint32_t before = ab;
    for_list2([&](uint64_t o) {
        before += o >= cut && (uint32_t)(o & ((1ull << index_bits) - 1)) > from_end ? 1u : 0u;
    });
    before = wave_inclusive_scan(before);
    if (lane == kWave - 1) L.wsum[wave] = before;
    // ---- 5: payload, in index order -----------------------------------------------------------
    // picks per tile first: the register-held tiles' into rcnt, the others' into the total
    uint32_t w_total = 0;
    G.sweep([&](uint32_t h, uint32_t, uint32_t cnt, uint64_t a0, uint64_t a1) {
              const uint32_t c = (uint32_t)__popcll(__ballot(is_pick((uint32_t)lane < cnt, key64(a0), (uint32_t)a0))) +
                                 (uint32_t)__popcll(__ballot(is_pick((uint32_t)(kWave + lane) < cnt, key64(a1), (uint32_t)a1)));
              if (h != ~0u) L.rcnt[wave][h] = c;
              w_total += c;
          },
          [&](uint32_t h, uint32_t t) {
              uint32_t c = 0;
              dense_tile_walk<false>(rp, bn, t, L.dbuf[wave], [&](uint32_t i, uint32_t v, bool in) {
                  c += (uint32_t)__popcll(__ballot(is_pick(in && (v & 0x7FFFFFFFu) >= lo, v & 0x7FFFFFFFu, i)));
              });
              if (h != ~0u) L.rcnt[wave][h] = c;
              w_total += c;
          });
    if (lane == 0) L.wtot[wave] = w_total;
    __syncthreads();
    uint32_t wave_off = 0;
#pragma unroll
    for (int i = 0; i < kFWaves; i++) {
        wave_off += L.wsum[i];
        if (i < wave) wave_off += L.wtot[i];
    }
    auto emit_half = [&](bool valid, uint64_t e, uint32_t pos) {
        const uint32_t key = key64(e), idx = (uint32_t)e, bitsv = (uint32_t)(e >> 32);
        const bool pick = is_pick(valid, key, idx);
        const uint64_t m = __ballot(pick);
        if (pick) {
            const u2a pr = {idx, bitsv};
            *(u2a4*)(out + 1 + 2 * (uint64_t)(pos + (uint32_t)__popcll(m & below))) = pr;
        }
        // the streaming block stored 0.0f for key >= predicted threshold; repair where the prediction was wrong
        if (valid && pick != (key >= that_key)) rp[idx] = pick ? 0.0f : u2f(bitsv);
        return pos + (uint32_t)__popcll(m);
    };
    auto emit_dense = [&](uint32_t t, uint32_t pos) {
        // a dense tile's residual holds plain sums (nothing was stored as zero)
        dense_tile_walk<false>(rp, bn, t, L.dbuf[wave], [&](uint32_t i, uint32_t v, bool in) {
            const bool pick = is_pick(in && (v & 0x7FFFFFFFu) >= lo, v & 0x7FFFFFFFu, i);
            const uint64_t m = __ballot(pick);
            if (pick) {
                const uint32_t p = pos + (uint32_t)__popcll(m & below);
                out[1 + 2 * (uint64_t)p] = i;
                out[2 + 2 * (uint64_t)p] = v;
                rp[i] = 0.0f;
            }
            pos += (uint32_t)__popcll(m);
        });
        return pos;
    };
    if constexpr (MANY) {
        uint32_t pos = wave_off;
        G.sweep([&](uint32_t, uint32_t, uint32_t cnt, uint64_t a0, uint64_t a1) {
                    pos = emit_half((uint32_t)lane < cnt, a0, pos);
                    pos = emit_half((uint32_t)(kWave + lane) < cnt, a1, pos);
                },
                [&](uint32_t, uint32_t t) { pos = emit_dense(t, pos); });
    } else {
        uint32_t pos = wave_off;
#pragma unroll
        for (int h = 0; h < kHeld; h++) {
            if (G.wt0 + h < G.wt1) {
                if (G.cnt[h] != kDense) {
                    pos = emit_half((uint32_t)lane < G.cnt[h], G.e0[h], pos);
                    pos = emit_half((uint32_t)(kWave + lane) < G.cnt[h], G.e1[h], pos);
                } else {
                    pos += L.rcnt[wave][h];  // written out by the loop below
                }
            }
        }
        if (G.more) {
            pos = wave_off;
#pragma unroll 1
            for (uint32_t t = G.wt0; t < G.wt1; t++) {
                const uint32_t cnt = (uint32_t)__builtin_amdgcn_readfirstlane((int)G.tcnt[t]);
                if (cnt == kDense) {
                    pos = emit_dense(t, pos);
                } else if (t - G.wt0 < (uint32_t)kHeld) {
                    pos += L.rcnt[wave][t - G.wt0];
                } else {
                    const uint64_t a0 = G.slots[(uint64_t)t * kTileSlots + lane];
                    const uint64_t a1 = G.slots[(uint64_t)t * kTileSlots + kWave + lane];
                    pos = emit_half((uint32_t)lane < cnt, a0, pos);
                    pos = emit_half((uint32_t)(kWave + lane) < cnt, a1, pos);
                }
            }
        }
    }
    if (grp == 0 && threadIdx.x == 0) {
        st[S_T] = T;
        st[S_ISTAR] = istar;
        st[S_OK] = 1u;
    }
    } while (false);
    // the exact selection for a bucket the window could not finish (S_OK stays 0)
    if (failed) {
        const auto restore = [&] {
            G.sweep([&](uint32_t, uint32_t, uint32_t cnt, uint64_t a0, uint64_t a1) {
                        if ((uint32_t)lane < cnt && key64(a0) >= that_key) rp[(uint32_t)a0] = u2f((uint32_t)(a0 >> 32));
                        if ((uint32_t)(kWave + lane) < cnt && key64(a1) >= that_key) rp[(uint32_t)a1] = u2f((uint32_t)(a1 >> 32));
                    },
                    [&](uint32_t, uint32_t) {});
        };
        if (!select_exact_group<kBlock>(bk, g, w, b, grp, fg, (uint64_t)b << g.gshift, restore, L, limit_ticks)) {
            fused_give_up(w, st, out);
            return;
        }
    }
    if (grp == 0 && threadIdx.x == 0 && !ld_agent(st + S_TIMEOUT)) out[0] = k;
}

// ================================ host side =======================================

uint64_t align4(uint64_t words) { return (words + 3) & ~uint64_t(3); }

uint64_t zeroed_words(const Geometry& g) {
    return align4((uint64_t)g.nbuckets * kHistWords) + align4((uint64_t)g.nbuckets * kStateWords);
}

// Groups that the workspace has room for: the most that a call with such tiles cuts its buckets into, so that it does
// not shrink where a bucket more makes them fewer.
uint32_t most_groups_shift(const Geometry& g) { return g.many ? 8 : topk_group_shift_few(g.ftiles); }
uint64_t all_groups(const Geometry& g) { return (uint64_t)g.nbuckets << most_groups_shift(g); }

// `groups`: those of the whole call with as many as that; `fits`: see topk_group_shift_fits.
void set_groups(Geometry* g, uint64_t groups, uint64_t fits) {
    g->gshift = topk_shift(g->ftiles, groups, g->many != 0, fits);
    g->ngroups = topk_launched_groups(g->ftiles, topk_tiles(g->n_total - (uint64_t)(g->nbuckets - 1) * g->bucket_elems), g->gshift);
}

uint64_t workspace_words(const Geometry& g) {
    const uint64_t groups = all_groups(g);
    return zeroed_words(g) + 2 * align4((uint64_t)g.nbuckets * g.tiles) + 2 * align4(groups) +
           align4((uint64_t)g.nbuckets * g.ftiles) + align4((uint64_t)g.nbuckets * g.ftiles * g.slots * 2) +
           align4(groups * kCntStride) + align4(groups * kCoarse) +
           align4((uint64_t)g.nbuckets * kCoarse) + align4((uint64_t)g.nbuckets * (kCoarse - 1) * g.lcapb * 2);
}

Workspace carve(void* base, const Geometry& g) {
    Workspace w;
    uint32_t* p = (uint32_t*)base;
    w.hist = p;        p += align4((uint64_t)g.nbuckets * kHistWords);
    w.state = p;       p += align4((uint64_t)g.nbuckets * kStateWords);
    w.tile_gt = p;     p += align4((uint64_t)g.nbuckets * g.tiles);
    w.tile_eq = p;     p += align4((uint64_t)g.nbuckets * g.tiles);
    w.blk_above = p;   p += align4(all_groups(g));
    w.blk_eq = p;      p += align4(all_groups(g));
    w.tile_cnt = p;    p += align4((uint64_t)g.nbuckets * g.ftiles);
    w.slots = (uint64_t*)p;  p += align4((uint64_t)g.nbuckets * g.ftiles * g.slots * 2);
    w.grp_cnt = p;     p += align4(all_groups(g) * kCntStride);
    w.gsuf = p;        p += align4(all_groups(g) * kCoarse);
    w.bin_fill = p;    p += align4((uint64_t)g.nbuckets * kCoarse);
    w.blist = (uint64_t*)p;
    // The resident path's scratch lies where the streaming path has its lists: a call takes one of the two.
    // It is used for buckets of more than one block, more than kRVecElems elements; theirs hold at least 2048
    // entries a bin.  (Words of its own would make the size fall from 2 M elements to 2 M + 1, and refuse a
    // workspace sized for a longer bucket.)
    static_assert((kCoarse - 1) * 2048 * 2 >= kRWords && kRVecElems >= 2048, "fits the lists");
    w.rmem = p;
    w.status = nullptr;
    return w;
}

bool make_geometry(uint64_t n_total, uint64_t bucket_elems, double ratio, Geometry* g) {
    if (n_total == 0 || bucket_elems == 0 || n_total > MCCL_HIP_MAX_ELEMS) return false;
    if (bucket_elems > n_total) bucket_elems = n_total;
    if (bucket_elems > 0xFFFFFFFFull) return false;  // indices are 32-bit
    const uint64_t nb = (n_total + bucket_elems - 1) / bucket_elems;
    if (nb > 65535) return false;
    g->n_total = n_total;
    g->bucket_elems = bucket_elems;
    g->nbuckets = (uint32_t)nb;
    g->tiles = (uint32_t)((bucket_elems + kTile - 1) / kTile);
    g->k_full = mccl_hip_topk_k(bucket_elems, ratio);
    g->k_last = mccl_hip_topk_k(n_total - (nb - 1) * bucket_elems, ratio);
    g->listed = 0;
    g->ftiles = (uint32_t)((bucket_elems + kFTile - 1) / kFTile);
    g->many = topk_many(bucket_elems, ratio) ? 1 : 0;
    g->slots = g->many ? kManySlots : kTileSlots;
    g->gshift = g->ngroups = 0;  // launch_single_pass' part
    // a coarse bin holds about k / 80 candidates when the window is as wide as a sample of 8192
    // leaves it, the bins at the window's lower end three times that; k / 10 + 2048 entries
    // leave room for more uneven ones
    uint64_t capb = (uint64_t)g->k_full / 10 + 2048;
    if (capb > bucket_elems) capb = bucket_elems;
    g->lcapb = (uint32_t)capb;
    return true;
}

// Every call of the single-pass path carries a number of its own; a bucket's window counts
// as published when its S_READY word shows that number (whatever a workspace held before,
// it is not this call's number; zero is what a finished call leaves behind).
std::atomic<uint32_t> g_epoch{0x5EED0001u};

uint32_t next_epoch() {
    uint32_t e = ++g_epoch;
    if (e == 0) e = ++g_epoch;
    return e;
}

// The two launches of the single-pass path.
template <int THREADS, bool LISTED, bool MANY>
void launch_stream(Buckets& bk, const Geometry& g, const Workspace& w, uint64_t tiles, uint64_t limit_ticks, hipStream_t st) {
    // a sample block per bucket, then per bucket its tiles and its bin blocks
    constexpr uint32_t per = StreamShape<THREADS>::kTiles;
    uint64_t blocks = (uint64_t)g.nbuckets * ((g.ftiles + per - 1) / per + g.ngroups + 1) + g.ngroups;
    if constexpr (LISTED) {
        // segment b: the tiles of bucket b, then the bin blocks of bucket b - 1
        uint32_t at = 0, before = 0;
        for (uint32_t b = 0; b < g.nbuckets; b++) {
            const uint32_t tiles = topk_tiles(bk.lcount[b]);
            bk.lfirst[b] = at;
            at += (tiles + per - 1) / per + before;
            before = topk_groups(tiles, g.gshift);
        }
        blocks = g.nbuckets + at + before;
    }
    const uint32_t epoch = next_epoch();
    // blocks that are resident from the start of the launch: they wait for the sample blocks
    static const int per_cu = [] {
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_topk_stream<THREADS, LISTED, MANY>, THREADS, 0) != hipSuccess || n < 1)
            n = StreamShape<THREADS>::kPerSimd * 4 * kWave / THREADS;
        return n;
    }();
    const uint32_t first_wave = g.nbuckets + (uint32_t)device_info().num_cus * (uint32_t)per_cu;
    // (tests of the give-up path: the sample blocks publish a number nobody waits for)
    const uint32_t published = tuning().topk_stall_test ? ~epoch : epoch;
    k_topk_stream<THREADS, LISTED, MANY><<<(uint32_t)blocks, THREADS, 0, st>>>(bk, g, w, epoch, published, first_wave,
                                                                                          stream_hold(tiles, g.nbuckets), limit_ticks);
}

template <bool LISTED, bool MANY>
void launch_single_pass(const Buckets& call, const Geometry& geometry, const Workspace& w, uint64_t fits, hipStream_t st) {
    // 100 MHz ticks a block may wait before it gives up
    const uint64_t lim = (uint64_t)tuning().topk_barrier_ms * 100000ull;
    // A list's blocks are those that its buckets have, longest bucket first: the bin blocks that nothing is
    // streamed beside are those of the shortest.
    Buckets bk = call;
    Geometry g = geometry;
    uint64_t tiles = (uint64_t)g.nbuckets * g.ftiles;
    if constexpr (!LISTED) set_groups(&g, g.nbuckets * (uint64_t)topk_groups(g.ftiles, most_groups_shift(g)), fits);
    if constexpr (LISTED) {
        uint32_t order[kMaxListed];
        longest_first(call, g.nbuckets, order);
        uint64_t groups = 0;
        tiles = 0;
        for (uint32_t b = 0; b < g.nbuckets; b++) {
            place_bucket(&bk, b, call, order[b], 0);
            tiles += topk_tiles(bk.lcount[b]);
            groups += topk_groups(topk_tiles(bk.lcount[b]), most_groups_shift(g));
        }
        for (uint32_t b = g.nbuckets; b < kMaxListed; b++) bk.lfirst[b] = 0xFFFFFFFFu;
        set_groups(&g, groups, fits);
    }
    if (stream_wide(tiles)) launch_stream<512, LISTED, MANY>(bk, g, w, tiles, lim, st);
    else launch_stream<256, LISTED, MANY>(bk, g, w, tiles, lim, st);
    // the select launch, at most kSelBlocks blocks at a time: all of them are resident
    // together, whatever the order in which the hardware dispatches them
    for (uint32_t b0 = 0; b0 < g.nbuckets;) {
        if constexpr (LISTED) {
            uint32_t blocks = 0, b = b0;
            for (uint32_t i = 0; i < b0; i++) bk.lfirst[i] = 0;  // before b0, which starts there and is the last that does
            for (; b < g.nbuckets; b++) {
                const uint32_t groups = topk_groups(topk_tiles(bk.lcount[b]), g.gshift);
                if (blocks + groups > kSelBlocks) break;
                bk.lfirst[b] = blocks;
                blocks += groups;
            }
            for (uint32_t i = b; i < g.nbuckets; i++) bk.lfirst[i] = 0xFFFFFFFFu;
            k_topk_select<true, MANY><<<blocks, kBlock, 0, st>>>(bk, g, w, b0, lim);
            b0 = b;
        } else {
            const uint32_t at_once = kSelBlocks / g.ngroups;
            const uint32_t nb = g.nbuckets - b0 < at_once ? g.nbuckets - b0 : at_once;
            k_topk_select<false, MANY><<<dim3(g.ngroups, nb), kBlock, 0, st>>>(bk, g, w, b0, lim);
            b0 += nb;
        }
    }
}

// Blocks of a select launch that may wait for others: those of a bucket whose selection falls back.
uint64_t select_limit_on(const StreamShare& share) {
    static const uint64_t per_cu = [] {
        int least = 1 << 20;
        for (const void* k : {(const void*)k_topk_select<false, false>, (const void*)k_topk_select<false, true>,
                              (const void*)k_topk_select<true, false>, (const void*)k_topk_select<true, true>}) {
            int n = 0;
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k, kBlock, 0) != hipSuccess) n = 0;
            least = n < least ? n : least;
        }
        return (uint64_t)least;
    }();
    return waiting_limit(share, per_cu);
}

// False when the call has to take the exact path.
bool launch_by_path(const Buckets& bk, const Geometry& g, const Workspace& w, const uint64_t* counts, hipStream_t st) {
    const StreamShare share = stream_share(st);
    const uint64_t limit = g.bucket_elems <= kRMaxBucket ? resident_limit_on(share) : 0, fits = select_limit_on(share);
    const TopkCall call = {g.n_total, g.bucket_elems, g.nbuckets, counts, g.k_full, g.many != 0};
    const Route route = choose_path(call, tuning().topk_path, limit, fits);
    if (route.path == kPathExact) return false;
    const uint64_t limit_ticks = (uint64_t)tuning().topk_barrier_ms * 100000ull;  // of 10 ns
    // (tests of the give-up path: the sample and lead blocks publish a number nobody waits for)
    const auto published = [](uint32_t epoch) { return tuning().topk_stall_test ? ~epoch : epoch; };
    const uint32_t shift = most_groups_shift(g);
    // A recorded list takes two launches, the second of which takes the windows back, also behind a first one that was given up.
    // (One launch with a kernel in front of it that takes them back: 24 buckets of 1001 to 1.5 M elements replayed in 35.7 us, two
    // launches 33.1; 16 of 300,000 34.8 / 32.0, 16 of 1 M 62.6 / 62.7, 12 of 1000 to 4 M at 5 % 48.1 / 47.9.)
    const uint32_t group_tiles = route.path == kPathStream && !is_capturing(st) ? whole_tiles(call, shift, whole_limit_on(share)) : 0;
    if (group_tiles) {
        const uint32_t epoch = next_epoch();
        launch_whole(bk, g, w, group_tiles, shift, epoch, published(epoch), limit_ticks, st);
    } else if (route.path == kPathStream) {
        if (g.listed) (g.many ? launch_single_pass<true, true> : launch_single_pass<true, false>)(bk, g, w, fits, st);
        else (g.many ? launch_single_pass<false, true> : launch_single_pass<false, false>)(bk, g, w, fits, st);
    } else {
        const uint32_t epoch = next_epoch();
        launch_resident(bk, g, w, route.vecs, limit, epoch, published(epoch), limit_ticks, st);
    }
    return true;
}

}  // namespace
}  // namespace mcclhip

using namespace mcclhip;

extern "C" {

uint32_t mccl_hip_topk_k(uint64_t count, double ratio) {
    uint32_t k = static_cast<uint32_t>(static_cast<double>(count) * ratio);
    return k < 1u ? 1u : k;
}

uint64_t mccl_hip_topk_max_compressed_size(uint64_t nbytes, double ratio) {
    const uint64_t count = nbytes / 4;
    const uint32_t k = static_cast<uint32_t>(static_cast<double>(count) * ratio) + 1u;
    return 4u + (uint64_t)k * 8u;
}

uint64_t mccl_hip_topk_workspace_bytes(uint64_t n_total, uint64_t bucket_elems, double ratio) {
    Geometry g;
    if (!(ratio > 0.0 && ratio <= 1.0)) return 0;
    if (!make_geometry(n_total, bucket_elems, ratio, &g)) return 0;
    return workspace_words(g) * 4 + 256;
}

int mccl_hip_topk_compress(const float* grad, float* residual, uint64_t n_total,
                           uint64_t bucket_elems, double ratio, void* wire,
                           uint64_t wire_stride, void* workspace, uint64_t workspace_bytes,
                           int* status, void* stream) {
    if (!grad || !residual || !wire || !workspace) return MCCL_HIP_ERR_ARG;
    if (!(ratio > 0.0 && ratio <= 1.0)) return MCCL_HIP_ERR_ARG;
    Geometry g;
    if (!make_geometry(n_total, bucket_elems, ratio, &g)) return MCCL_HIP_ERR_ARG;
    if ((wire_stride & 3) || ((uintptr_t)wire & 3)) return MCCL_HIP_ERR_ARG;
    const uint32_t kmax = g.k_full > g.k_last ? g.k_full : g.k_last;
    if (wire_stride < 4 + 8 * (uint64_t)kmax) return MCCL_HIP_ERR_CAPACITY;
    if (workspace_bytes < workspace_words(g) * 4 + 16) return MCCL_HIP_ERR_WORKSPACE;
    int rc = mccl_hip_init();
    if (rc) return rc;
    hipStream_t st = (hipStream_t)stream;
    // the carved arrays are 16-byte aligned inside the caller's buffer
    void* aligned = (void*)(((uintptr_t)workspace + 15) & ~(uintptr_t)15);
    Workspace w = carve(aligned, g);
    w.status = status;
    const uint64_t cap = (uint64_t)device_info().num_cus * (uint64_t)(tuning().fold_blocks_per_cu < 256 ? tuning().fold_blocks_per_cu : 256);
    const uint64_t nvec = g.bucket_elems / 4;
    const uint64_t bx = (cap + g.nbuckets - 1) / g.nbuckets;
    const uint64_t need_r = (nvec + kBlock * 4 - 1) / (kBlock * 4);
    const uint32_t bx_r = clamp_u32(bx < need_r ? bx : need_r, 1, 65535);
    const uint32_t bx_t = clamp_u32(bx < g.tiles ? bx : g.tiles, 1, 65535);
    Buckets bk = {};
    bk.grad = grad;
    bk.residual = residual;
    bk.wire = (uint8_t*)wire;
    bk.wire_stride = wire_stride;
    if (!launch_by_path(bk, g, w, nullptr, st)) {
        const uint64_t zw = zeroed_words(g);
        k_zero_words<<<clamp_u32((zw / 4 + kBlock - 1) / kBlock, 1, cap), kBlock, 0, st>>>(w.hist, zw);
        const uint64_t need_a = (nvec + kBlock * 2 - 1) / (kBlock * 2);
        const uint32_t bx_a = clamp_u32(bx < need_a ? bx : need_a, 1, 65535);
        k_topk_pass_a<<<dim3(bx_a, g.nbuckets), kBlock, 0, st>>>(grad, residual, g, w);
        k_topk_refine<<<dim3(bx_r, g.nbuckets), kBlock, 0, st>>>(residual, g, w, 1, 0);
        k_topk_refine<<<dim3(bx_r, g.nbuckets), kBlock, 0, st>>>(residual, g, w, 2, 0);
        k_topk_count<<<dim3(bx_t, g.nbuckets), kBlock, 0, st>>>(residual, g, w, 0);
        k_topk_emit<<<dim3(bx_t, g.nbuckets), kBlock, 0, st>>>(residual, g, w, (uint8_t*)wire, wire_stride, 0);
    }
    return launch_status();
}

uint64_t mccl_hip_topk_list_workspace_bytes(const uint64_t* host_counts, uint32_t nbuckets, double ratio) {
    if (!host_counts || nbuckets == 0 || nbuckets > kMaxListed) return 0;
    uint64_t longest = 0;
    for (uint32_t b = 0; b < nbuckets; b++) {
        if (host_counts[b] == 0) return 0;
        longest = host_counts[b] > longest ? host_counts[b] : longest;
    }
    return mccl_hip_topk_workspace_bytes(longest * nbuckets, longest, ratio);
}

int mccl_hip_topk_compress_list(const float* const* host_grads, float* const* host_residuals,
                                const uint64_t* host_counts, void* const* host_wires,
                                const uint64_t* host_wire_capacities, uint32_t nbuckets, double ratio,
                                void* workspace, uint64_t workspace_bytes, int* status, void* stream) {
    if (!host_grads || !host_residuals || !host_counts || !host_wires || !host_wire_capacities || !workspace)
        return MCCL_HIP_ERR_ARG;
    if (nbuckets == 0 || nbuckets > kMaxListed || !(ratio > 0.0 && ratio <= 1.0)) return MCCL_HIP_ERR_ARG;
    Buckets bk = {};
    uint64_t longest = 0;
    for (uint32_t b = 0; b < nbuckets; b++) {
        if (!host_grads[b] || !host_residuals[b] || !host_wires[b] || ((uintptr_t)host_wires[b] & 3))
            return MCCL_HIP_ERR_ARG;
        if (host_counts[b] == 0 || host_counts[b] > 0xFFFFFFFFull) return MCCL_HIP_ERR_ARG;  // indices are 32-bit
        const uint32_t k = mccl_hip_topk_k(host_counts[b], ratio);
        if (host_wire_capacities[b] < 4 + 8 * (uint64_t)k) return MCCL_HIP_ERR_CAPACITY;
        bk.lgrad[b] = host_grads[b];
        bk.lresidual[b] = host_residuals[b];
        bk.lwire[b] = (uint8_t*)host_wires[b];
        bk.lcount[b] = (uint32_t)host_counts[b];
        bk.lk[b] = k;
        longest = host_counts[b] > longest ? host_counts[b] : longest;
    }
    Geometry g;
    if (!make_geometry(longest * nbuckets, longest, ratio, &g)) return MCCL_HIP_ERR_ARG;
    g.listed = 1;
    if (workspace_bytes < workspace_words(g) * 4 + 16) return MCCL_HIP_ERR_WORKSPACE;
    int rc = mccl_hip_init();
    if (rc) return rc;
    void* aligned = (void*)(((uintptr_t)workspace + 15) & ~(uintptr_t)15);
    Workspace w = carve(aligned, g);
    w.status = status;
    if (!launch_by_path(bk, g, w, host_counts, (hipStream_t)stream)) return MCCL_HIP_ERR_ARG;
    return launch_status();
}


int mccl_hip_topk_path_report(const void* workspace, uint64_t n_total, uint64_t bucket_elems, double ratio,
                              uint32_t* host_single_pass_buckets, uint32_t* host_buckets, void* stream) {
    if (!workspace || !host_single_pass_buckets || !host_buckets) return MCCL_HIP_ERR_ARG;
    Geometry g;
    if (!(ratio > 0.0 && ratio <= 1.0) || !make_geometry(n_total, bucket_elems, ratio, &g)) return MCCL_HIP_ERR_ARG;
    void* aligned = (void*)(((uintptr_t)workspace + 15) & ~(uintptr_t)15);
    Workspace w = carve(aligned, g);
    std::vector<uint32_t> st((size_t)g.nbuckets * kStateWords);
    MCCLHIP_TRY(hipMemcpyAsync(st.data(), w.state, st.size() * 4, hipMemcpyDeviceToHost, (hipStream_t)stream));
    MCCLHIP_TRY(hipStreamSynchronize((hipStream_t)stream));
    uint32_t ok = 0;
    for (uint32_t b = 0; b < g.nbuckets; b++) {
        if (st[(size_t)b * kStateWords + S_TIMEOUT]) return MCCL_HIP_ERR_TIMEOUT;  // the payload is invalid
        ok += st[(size_t)b * kStateWords + S_OK] ? 1u : 0u;
    }
    *host_single_pass_buckets = ok;
    *host_buckets = g.nbuckets;
    return MCCL_HIP_OK;
}

}  // extern "C"

