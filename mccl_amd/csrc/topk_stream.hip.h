// What the kernels of the single-pass top-k path (topk.hip: two launches, topk_whole.hip: one) share: the tiles, their
// candidate slots and window bins, the streaming blocks, and the exact selection that a bucket's select blocks run together when
// the window fails.
#pragma once

#include "topk_common.hip.h"

namespace mcclhip {

// Scans a finished histogram from its top bin downwards and returns the bin in
// which the running count reaches `remaining`, and through *left how many of
// the remaining picks fall inside that bin.  Called by all THREADS threads of a
// block with identical arguments; every thread receives the result.
// `floor_bin`: bins below it count as empty.  Returns BINS when the histogram
// holds fewer than `remaining` elements.
template <int BINS, int THREADS>
__device__ __forceinline__ uint32_t pick_bin(const uint32_t* h, uint32_t remaining, uint32_t floor_bin,
                                             uint32_t* left, uint32_t* scratch /* THREADS/kWave + 2 words */) {
    constexpr int PER = (BINS + THREADS - 1) / THREADS;
    uint32_t c[PER];
    uint32_t sum = 0;
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int r = threadIdx.x * PER + j;  // reversed bin number
        const int bin = BINS - 1 - r;
        c[j] = (r < BINS && (uint32_t)bin >= floor_bin) ? h[bin] : 0u;
        sum += c[j];
    }
    uint32_t total;
    uint32_t above = block_exclusive_scan_n<THREADS>(sum, scratch, &total);
    uint32_t* res = scratch + THREADS / kWave;
    if (threadIdx.x == 0) { res[0] = BINS; res[1] = 0; }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PER; j++) {
        if (above < remaining && remaining <= above + c[j]) {
            res[0] = BINS - 1 - (threadIdx.x * PER + j);
            res[1] = remaining - above;
        }
        above += c[j];
    }
    __syncthreads();
    const uint32_t bin = res[0];
    *left = res[1];
    __syncthreads();
    return bin;
}

constexpr int kFRegion = 1024;                // elements one wavefront streams
constexpr int kFWaves = 4;                    // wavefronts of a tile
static_assert(kFTile == kFRegion * kFWaves, "elements per streaming tile");
// The streaming launch's blocks have 256 threads or 512 (THREADS), a streaming block a tile for every 256.
template <int THREADS>
struct StreamShape {
    static constexpr int kWaves = THREADS / kWave;
    static constexpr uint32_t kTiles = kWaves / kFWaves;       // of a streaming block
    static constexpr int kHeld = kTiles == 1 ? 7 : 4;          // tiles per wavefront whose slots a bin block keeps in registers
    static constexpr int kPerSimd = kTiles == 1 ? 6 : 8;       // wavefronts that the registers are to leave room for
};
// What a tile keeps of its candidates.  MANY: calls whose ratio makes more of them than kTileSlots take (topk_many); a
// quarter of a wavefront's elements is staged, of which a ratio of 12 % takes 58 % (window_share: 148 of 256).  15 buckets of 6,553,600 elements, us: at 2 % 669 on
// the path with 128 slots (most tiles dense), 230 so; at 5 % 852 / 252; one bucket at 5 % 140 on the exact path, 38.5 so.  What
// bounds it is the same stream as at 1 % (186 us of it) and, at 5 %, the candidates' 16 bytes written, read twice and listed.
template <bool MANY>
struct TileShape {
    static constexpr int kStage = MANY ? 256 : 64;                        // candidates a wavefront stages
    static constexpr int kSlots = MANY ? kManySlots : kTileSlots;         // of a tile
};
static_assert(kManySlots >= kFWaves * 256, "what a tile's wavefronts stage fits its slots");
constexpr int kFVecs = kFRegion / (kWave * 4);  // 16-byte vectors per lane and array: all issued at once
constexpr int kCoarse = 128;                  // coarse window bins; the last one holds keys >= hi
constexpr int kBinsPerLane = kCoarse / kWave; // 2
constexpr int kCntStride = 64;                // words between two groups' arrival counters: 256 bytes, so that the
                                              // arrivals of a bucket's tiles spread over memory channels
constexpr int kHeld = 7;                      // tiles per wavefront whose slots a select block keeps in registers
constexpr uint32_t kSelBlocks = 1024;         // blocks of a k_topk_select launch: all resident
constexpr uint32_t kGaveUp = 0xFFFFFFFEu;     // a wavefront's count: its wait for the sample timed out
static_assert(kFVecs == 4, "the streaming role is written for four vectors per lane");

// a / b rounded down, for whole numbers a below 2^41.  The quotient is a multiple of 1 / b, and the doubles about it lie
// closer than 2^-11 / b: the division's rounding never reaches the next whole number.  (100 instructions fewer than a
// division of 64-bit numbers, on the way between two loads that need each other.)
__device__ __forceinline__ double whole_quotient(double a, uint32_t b) { return a / (double)b; }

// The kCoarse - 1 bins below the top one divide [lo, hi) evenly: bin = ((key - lo) * mul) >> 32.
__device__ __forceinline__ uint32_t window_mul(uint32_t lo, uint32_t hi) {
    const uint32_t range = hi - lo;  // key - lo < range for every key below hi
    if (range <= (uint32_t)(kCoarse - 1)) return 0xFFFFFFFFu;  // a bin per key
    return (uint32_t)whole_quotient((double)(kCoarse - 1) * 4294967296.0, range);
}
// The smallest key of bin j (1 <= j <= kCoarse - 1; bin 0 starts at lo): lo + ceil(j * 2^32 / mul).
__device__ __forceinline__ uint32_t window_bin_lo(uint32_t lo, uint32_t mul, uint32_t j) {
    if (j == 0) return lo;
    return lo + (uint32_t)whole_quotient((double)j * 4294967296.0 + (double)(mul - 1), mul);
}

struct FusedGeo {       // per-bucket tiling, derived the same way by every block
    uint64_t bn;        // elements
    uint32_t k;
    uint32_t ntiles;    // streaming tiles
    uint32_t tpg;       // tiles per group
    uint32_t ng;        // groups
};
__device__ __forceinline__ FusedGeo fused_geo(const Geometry& g, BucketsArg bk, uint32_t b) {
    FusedGeo f;
    f.bn = bucket_count(g, bk, b);
    f.k = bucket_k(g, bk, b);
    f.ntiles = (uint32_t)((f.bn + kFTile - 1) / kFTile);
    f.tpg = topk_group_tiles(f.ntiles, g.gshift);
    f.ng = (f.ntiles + f.tpg - 1) / f.tpg;
    return f;
}

// Coarse window bin of a candidate key (key >= lo).
__device__ __forceinline__ uint32_t coarse_bin(uint32_t key, uint32_t lo, uint32_t hi, uint32_t mul) {
    return key >= hi ? (uint32_t)(kCoarse - 1) : __umulhi(key - lo, mul);
}

// Waits until *p == want.  Called by a whole wavefront or a single thread; false when the wait timed out.
// Every poll is a memory transaction on one address (agent-scope loads are not cached):
// few pollers and a pause between polls, or the channel that holds the word becomes the
// bottleneck of every stream that crosses it.
template <int SLEEP = 16>
__device__ __forceinline__ bool wait_word(const uint32_t* p, uint32_t want, uint64_t limit_ticks) {
    uint64_t t0 = 0;
    uint32_t polls = 0;
    while ((uint32_t)__builtin_amdgcn_readfirstlane((int)ld_agent(p)) != want) {
        __builtin_amdgcn_s_sleep(SLEEP);
        if ((++polls & 63u) == 0) {
            const uint64_t now = (uint64_t)wall_clock64();
            if (t0 == 0) t0 = now;
            else if (now - t0 > limit_ticks) return false;
        }
    }
    asm volatile("" ::: "memory");
    return true;
}

// ---- a wavefront's candidates ----------------------------------------------------------
// Appends the lanes' candidates (mask4: which of a lane's four elements) to the `staged` ones of the wavefront, in
// index order: lane-major, element-minor.  Nearly every call finds a few lanes with one candidate each: one ballot,
// one 8-byte LDS store.  False, and nothing is stored, when they are more than STAGE then.
template <int STAGE>
__device__ __forceinline__ bool stage_append(uint64_t* slots, uint32_t& staged, uint32_t mask4, const u4a& a, uint32_t first_idx) {
    auto lanes_below = [](uint64_t m) {
        return (uint32_t)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
    };
    auto pick = [](const u4a& v4, uint32_t q) {
        uint32_t v = v4[0];
        v = q == 1 ? v4[1] : v;
        v = q == 2 ? v4[2] : v;
        return q == 3 ? v4[3] : v;
    };
    const uint64_t m1 = __ballot(mask4 != 0);
    if (!m1) return true;  // wave-uniform
    const uint32_t c = __popc(mask4);
    uint32_t before = lanes_below(m1), total = __popcll(m1);
    const uint64_t m2 = __ballot(c >= 2);
    if (m2) {  // wave-uniform
        before += lanes_below(m2);
        total += __popcll(m2);
        const uint64_t m3 = __ballot(c >= 3);
        if (m3) {
            const uint64_t m4 = __ballot(c >= 4);
            before += lanes_below(m3) + lanes_below(m4);
            total += __popcll(m3) + __popcll(m4);
        }
    }
    total = (uint32_t)__builtin_amdgcn_readfirstlane((int)total);
    if (staged + total > (uint32_t)STAGE) return false;
    if (mask4) {
        uint32_t pos = staged + before;
        const uint32_t q = (uint32_t)__ffs((int)mask4) - 1u;
        slots[pos] = (uint64_t)(first_idx + q) | ((uint64_t)pick(a, q) << 32);
        uint32_t rest = mask4 & (mask4 - 1u);
        while (rest) {
            const uint32_t q2 = (uint32_t)__ffs((int)rest) - 1u;
            slots[++pos] = (uint64_t)(first_idx + q2) | ((uint64_t)pick(a, q2) << 32);
            rest &= rest - 1u;
        }
    }
    staged = (uint32_t)__builtin_amdgcn_readfirstlane((int)(staged + total));
    return true;
}

// ---- streaming block ---------------------------------------------------------------------
template <int WAVES, int STAGE>
struct StreamBlockLds {
    uint64_t stage[WAVES][STAGE];  // a wavefront's candidates, (bits << 32) | index, in index order
    uint32_t wcnt[WAVES];
    uint32_t win[4];               // the bucket's window as wavefront 0 read it: lo, hi, predicted threshold, ready
};
// The block's tiles, from tile t on: a tile for every four wavefronts.  The groups' counters are laid out for 1 << shift a
// bucket.
template <int THREADS, bool MANY, class Lds>
__device__ __forceinline__ void stream_tiles(BucketsArg bk, const Geometry& g, const Workspace& w, uint32_t b, uint32_t t, const FusedGeo& fg,
                                             uint32_t shift, uint32_t epoch, uint64_t limit_ticks, Lds& L) {
    constexpr int kStage = TileShape<MANY>::kStage, kSlots = TileShape<MANY>::kSlots;
    const uint64_t bn = fg.bn;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const int first_wave_of_tile = wave / kFWaves * kFWaves;
    t += (uint32_t)(wave / kFWaves);  // the wavefront's tile
    const uint64_t w0 = (uint64_t)t * kFTile + (uint64_t)(wave - first_wave_of_tile) * kFRegion;  // first element of this wave's region
    const bool live = w0 < bn;                                             // wave-uniform
    float* const rbase = bucket_residual(g, bk, b);
    const float* gp = bucket_grad(g, bk, b) + w0;
    float* rp = rbase + w0;
    const uint32_t len = live ? (uint32_t)((bn - w0) < (uint64_t)kFRegion ? (bn - w0) : (uint64_t)kFRegion) : 0u;
    const uint32_t nfull = len / 4;  // full vectors in this region
    uint32_t* st = w.state + (uint64_t)b * kStateWords;
    u4a gv[kFVecs], rv[kFVecs];
    {
        // One path without branches between the loads (with them the 96.5 M gradient at 5 % took 247.0 us, so 246.2, one bucket of
        // 13 M at 1 % 51.5, so 51.0): lanes past the end ask for the region's last vector, and wavefronts without a whole one for
        // the bucket's state words; neither looks at them.
        const float* const gl = nfull ? gp : (const float*)st;
        const float* const rl = nfull ? rp : (const float*)st;
        const uint32_t last = nfull ? nfull - 1 : 0u;
#pragma unroll
        for (int u = 0; u < kFVecs; u++) {
            const uint32_t vi = (uint32_t)u * kWave + lane, at = (vi < last ? vi : last) * 4;
            gv[u] = __builtin_nontemporal_load((const u4u4*)(gl + at));
            rv[u] = __builtin_nontemporal_load((const u4u4*)(rl + at));
        }
    }
    uint32_t* out = bucket_wire(g, bk, b);
    // the window of this bucket: wait for its sample block (one wavefront polls for the block)
    if (wave == 0) {
        const u4a wn = wait_window(st, epoch, limit_ticks);
        if (lane == 0) { L.win[0] = wn[0]; L.win[1] = wn[1]; L.win[2] = wn[2]; L.win[3] = wn[3]; }
    }
    __syncthreads();
    const bool ready = L.win[3] != 0;
    const uint32_t lo_key = L.win[0], that_key = L.win[2];
    // both the same in every lane, and kept in scalar registers by saying so at every update
    uint32_t staged = 0;  // candidates of the region so far
    uint32_t dense = 0;   // 1: more candidates than slots
    uint64_t* const slots = L.stage[wave];
    // Puts back the region's staged candidates that were stored as zeros.
    auto restore_staged = [&]() {
#pragma unroll
        for (int i = 0; i < kStage; i += kWave) {
            if ((uint32_t)(i + lane) < staged) {
                const uint64_t e = slots[i + lane];
                if (((uint32_t)(e >> 32) & 0x7FFFFFFFu) >= that_key) st_agent((uint32_t*)rbase + (uint32_t)e, (uint32_t)(e >> 32));
            }
        }
    };
    auto append = [&](uint32_t mask4, const u4a& a, uint32_t first_idx) {
        if (dense) return;
        if (!stage_append<kStage>(slots, staged, mask4, a, first_idx)) {
            // the region goes dense: its earlier candidates were stored as zeros where
            // they reached the predicted threshold; put those values back
            dense = 1u;
            restore_staged();
        }
    };
    if (ready) {
#pragma unroll
        for (int u = 0; u < kFVecs; u++) {
            const uint32_t vi = (uint32_t)u * kWave + lane;
            u4a a = {0u, 0u, 0u, 0u}, z = {0u, 0u, 0u, 0u};
            uint32_t mask4 = 0;
            if (vi < nfull) {
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const float adj = u2f(gv[u][q]) + u2f(rv[u][q]);
                    a[q] = f2u(adj);
                    z[q] = key_of(adj) >= that_key ? 0u : a[q];
                    mask4 |= (key_of(adj) >= lo_key ? 1u : 0u) << q;
                }
            }
            append(mask4, a, (uint32_t)w0 + vi * 4);  // may turn the region dense
            if (vi < nfull) store_through(rp, vi * 4, dense ? a : z);
        }
        // the bucket's last partial vector (bucket length not a multiple of 4) lies in its last region
        if (len & 3) {
            u4a a = {0u, 0u, 0u, 0u};
            uint32_t mask4 = 0;
            if (lane == 0) {
                for (uint32_t q = 0; q < (len & 3); q++) {
                    const float adj = gp[nfull * 4 + q] + rp[nfull * 4 + q];
                    a[q] = f2u(adj);
                    mask4 |= (key_of(adj) >= lo_key ? 1u : 0u) << q;
                }
            }
            append(mask4, a, (uint32_t)w0 + nfull * 4);
            if (lane == 0) {
                for (uint32_t q = 0; q < (len & 3); q++)
                    st_agent((uint32_t*)rp + nfull * 4 + q, (!dense && (a[q] & 0x7FFFFFFFu) >= that_key) ? 0u : a[q]);
            }
        }
    }
    // ---- the tile's candidates, in index order, to its slots ------------------------------
    if (lane == 0) L.wcnt[wave] = !ready ? kGaveUp : (dense ? kDense : staged);
    __syncthreads();
    uint32_t before = 0, total = 0;
    bool tile_dense = false, gave_up = false;
#pragma unroll
    for (int i = 0; i < kFWaves; i++) {
        const uint32_t c = L.wcnt[first_wave_of_tile + i];
        gave_up |= c == kGaveUp;
        tile_dense |= c == kDense;
        if (first_wave_of_tile + i < wave) before += c;
        total += c;
    }
    if (gave_up) {  // a wavefront never saw the sample arrive: the bucket's result is invalid
        fused_give_up(w, st, out);
        return;     // without counting the tile: the bucket's bin blocks give up as well
    }
    tile_dense |= total > (uint32_t)kSlots;
    if (tile_dense) {
        if (!dense) restore_staged();  // a tile is dense as a whole: its residual holds plain sums
    } else {
#pragma unroll
        for (int i = 0; i < kStage; i += kWave)
            if ((uint32_t)(i + lane) < staged)
                st_agent64(w.slots + ((uint64_t)b * g.ftiles + t) * kSlots + before + i + lane, slots[i + lane]);
    }
    const bool counts = wave == first_wave_of_tile && lane == 0 && t < fg.ntiles;
    if (counts) st_agent(w.tile_cnt + (uint64_t)b * g.ftiles + t, tile_dense ? kDense : total);
    // ---- the block counts itself into its group once all its stores have arrived ----------
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (counts)
        __hip_atomic_fetch_add(w.grp_cnt + (((uint64_t)b << shift) + t / fg.tpg) * kCntStride, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---- a dense tile's elements ---------------------------------------------------------
// Calls f(index, bits, in_range) for every element of tile t of the bucket, 64 elements per
// step, every lane of the wavefront taking part in every step; the loads of B steps are in
// flight together and parked in LDS, so the code stays a loop.  AGENT: the residual was
// written by other blocks of the same launch.
template <bool AGENT, int B = 16, class F>
__device__ __forceinline__ void dense_tile_walk(const float* rp, uint64_t bn, uint32_t t, uint32_t* buf, F&& f) {
    const int lane = threadIdx.x & (kWave - 1);
    const uint64_t e0 = (uint64_t)t * kFTile;
    const uint64_t e1 = e0 + kFTile < bn ? e0 + kFTile : bn;
#pragma unroll 1
    for (uint64_t base = e0; base < e1; base += (uint64_t)B * kWave) {
        uint32_t v[B];
#pragma unroll
        for (int j = 0; j < B; j++) {
            const uint64_t i = base + (uint64_t)j * kWave + lane;
            if constexpr (AGENT) v[j] = i < e1 ? ld_agent((const uint32_t*)rp + i) : 0u;
            else v[j] = i < e1 ? f2u(rp[i]) : 0u;
        }
#pragma unroll
        for (int j = 0; j < B; j++) buf[j * kWave + lane] = v[j];  // a lane reads back only what it wrote
#pragma unroll 1
        for (int j = 0; j < B && base + (uint64_t)j * kWave < e1; j++) {  // wave-uniform trip count
            const uint64_t i = base + (uint64_t)j * kWave + lane;
            f((uint32_t)i, buf[j * kWave + lane], i < e1);
        }
    }
}

// ---- a group's tiles as a bin block / select block sees them ------------------------------
// The slots of up to HELD tiles per wavefront stay in registers, the rest (groups of more
// than NW * HELD tiles) are re-read from memory on every sweep.
enum Reads {
    kEarlier,  // the slots were written by an earlier launch
    kAgent     // ... by blocks of the same launch: past the caches
};
template <Reads READS, int NW, int HELD>
struct GroupTiles {
    static constexpr int kHeld = HELD;
    const uint32_t* tcnt;
    const uint64_t* slots;
    uint32_t t0;        // the group's first tile
    uint32_t wt0, wt1;  // this wavefront's tiles: a contiguous share of the group's, one of NW
    int lane;
    bool more;          // wave-uniform: dense tiles, or tiles past the register window
    uint32_t cnt[kHeld];            // candidates in the tile's slots, or kDense (wave-uniform)
    uint64_t e0[kHeld], e1[kHeld];  // slot `lane` and slot `64 + lane`

    static __device__ __forceinline__ uint32_t ld32(const uint32_t* p) {
        if constexpr (READS == kAgent) return ld_agent(p);
        else return *p;
    }
    static __device__ __forceinline__ uint64_t ld64(const uint64_t* p) {
        if constexpr (READS == kAgent) return ld_agent64(p);
        else return *p;
    }
    // every load issued at once
    __device__ __forceinline__ void load(const Geometry& g, const Workspace& w, uint32_t b, uint32_t grp,
                                         const FusedGeo& fg) {
        lane = threadIdx.x & (kWave - 1);
        const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
        tcnt = w.tile_cnt + (uint64_t)b * g.ftiles;
        slots = w.slots + (uint64_t)b * g.ftiles * kTileSlots;
        t0 = grp * fg.tpg;
        const uint32_t t1 = t0 + fg.tpg < fg.ntiles ? t0 + fg.tpg : fg.ntiles;
        const uint32_t pw = (t1 - t0 + NW - 1) / NW;
        wt0 = t0 + wave * pw < t1 ? t0 + wave * pw : t1;
        wt1 = wt0 + pw < t1 ? wt0 + pw : t1;
#pragma unroll
        for (int h = 0; h < kHeld; h++) {
            const uint32_t t = wt0 + h < wt1 ? wt0 + h : t0;  // stays inside the bucket's arrays
            cnt[h] = (uint32_t)__builtin_amdgcn_readfirstlane((int)ld32(tcnt + t));
            e0[h] = ld64(slots + (uint64_t)t * kTileSlots + lane);  // slots past the count: ignored by the sweeps
            e1[h] = ld64(slots + (uint64_t)t * kTileSlots + kWave + lane);
        }
        bool any_dense = false;
#pragma unroll
        for (int h = 0; h < kHeld; h++) any_dense |= wt0 + h < wt1 && cnt[h] == kDense;
        more = any_dense || wt1 > wt0 + kHeld;
    }
    // nd(h, t, cnt, e0, e1) for every ordinary tile (h < kHeld: register-held, else ~0u), dn(h, t)
    // for every dense one.  Order: register-held ordinary tiles first, then the dense ones and
    // those past the register window, in index order.
    template <class ND, class DN>
    __device__ __forceinline__ void sweep(ND&& nd, DN&& dn) const {
#pragma unroll
        for (int h = 0; h < kHeld; h++)
            if (wt0 + h < wt1 && cnt[h] != kDense) nd((uint32_t)h, wt0 + h, cnt[h], e0[h], e1[h]);
        if (more) {
#pragma unroll 1
            for (uint32_t t = wt0; t < wt1; t++) {
                const uint32_t h = t - wt0 < (uint32_t)kHeld ? t - wt0 : ~0u;
                const uint32_t c = (uint32_t)__builtin_amdgcn_readfirstlane((int)ld32(tcnt + t));
                if (c == kDense) {
                    dn(h, t);
                } else if (h == ~0u) {
                    const uint64_t a0 = ld64(slots + (uint64_t)t * kTileSlots + lane);
                    const uint64_t a1 = ld64(slots + (uint64_t)t * kTileSlots + kWave + lane);
                    nd(h, t, c, a0, a1);
                }
            }
        }
    }
};
// The same for tiles with slots for many candidates: nothing is kept, every sweep reads the slots again, in
// index order, a tile's (up to 384 candidates, what a ratio of 7 % makes) while the tile before it is looked at.
// One round trip of 0.7 us a sweep is exposed; registers for 384 entries of each tile would halve
// the blocks that fit a CU.
template <Reads READS, int NW>
struct ManyTiles {
    static constexpr int kPairs = 3;  // of 128 entries, read ahead
    static constexpr int kSlots = TileShape<true>::kSlots;
    const uint32_t* tcnt;
    const uint64_t* slots;
    uint32_t t0, wt0, wt1;  // as GroupTiles'
    int lane;

    static __device__ __forceinline__ uint64_t ld64(const uint64_t* p) {
        if constexpr (READS == kAgent) return ld_agent64(p);
        else return *p;
    }
    __device__ __forceinline__ void load(const Geometry& g, const Workspace& w, uint32_t b, uint32_t grp, const FusedGeo& fg) {
        lane = threadIdx.x & (kWave - 1);
        const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
        tcnt = w.tile_cnt + (uint64_t)b * g.ftiles;
        slots = w.slots + (uint64_t)b * g.ftiles * kSlots;
        t0 = grp * fg.tpg;
        const uint32_t t1 = t0 + fg.tpg < fg.ntiles ? t0 + fg.tpg : fg.ntiles;
        const uint32_t pw = (t1 - t0 + NW - 1) / NW;
        wt0 = t0 + wave * pw < t1 ? t0 + wave * pw : t1;
        wt1 = wt0 + pw < t1 ? wt0 + pw : t1;
    }
    // nd(~0u, t, cnt, e0, e1) for every 128 candidates of an ordinary tile (cnt: how many of them there are),
    // dn(~0u, t) for a dense one, all in index order.
    template <class ND, class DN>
    __device__ __forceinline__ void sweep(ND&& nd, DN&& dn) const {
#pragma unroll 1
        for (uint32_t c0 = wt0; c0 < wt1; c0 += kWave) {
            const uint32_t n = wt1 - c0 < (uint32_t)kWave ? wt1 - c0 : (uint32_t)kWave;
            uint32_t cnts = 0;
            if ((uint32_t)lane < n) {
                if constexpr (READS == kAgent) cnts = ld_agent(tcnt + c0 + lane);
                else cnts = tcnt[c0 + lane];
            }
            uint64_t e[2 * kPairs], next[2 * kPairs];
            // (lanes past the count read entry 0: no branches between the loads, no lines touched for nothing)
            auto fetch = [&](uint32_t i, uint64_t (&to)[2 * kPairs]) {
                const uint32_t cnt = (uint32_t)__builtin_amdgcn_readlane((int)cnts, (int)i);
                const uint64_t* p = slots + (uint64_t)(c0 + i) * kSlots;
#pragma unroll
                for (int r = 0; r < 2 * kPairs; r++) {
                    const uint32_t at = (uint32_t)(r * kWave + lane);
                    to[r] = ld64(p + (at < cnt ? at : 0u));
                }
            };
            fetch(0, e);
#pragma unroll 1
            for (uint32_t i = 0; i < n; i++) {
                fetch(i + 1 < n ? i + 1 : i, next);
                const uint32_t t = c0 + i, cnt = (uint32_t)__builtin_amdgcn_readlane((int)cnts, (int)i);
                if (cnt == kDense) {
                    dn(~0u, t);
                } else {
#pragma unroll
                    for (int v = 0; v < kPairs; v++)
                        if (cnt > (uint32_t)(v * 2 * kWave)) nd(~0u, t, cnt - v * 2 * kWave, e[2 * v], e[2 * v + 1]);
#pragma unroll 1
                    for (uint32_t from = kPairs * 2 * kWave; from < cnt; from += 2 * kWave) {
                        const uint64_t* p = slots + (uint64_t)t * kSlots + from;
                        const uint32_t left = cnt - from;
                        const uint64_t a0 = ld64(p + ((uint32_t)lane < left ? lane : 0));
                        const uint64_t a1 = ld64(p + ((uint32_t)(kWave + lane) < left ? kWave + lane : 0));
                        nd(~0u, t, left, a0, a1);
                    }
                }
#pragma unroll
                for (int r = 0; r < 2 * kPairs; r++) e[r] = next[r];
            }
        }
    }
};
__device__ __forceinline__ uint32_t key64(uint64_t e) { return (uint32_t)(e >> 32) & 0x7FFFFFFFu; }

// The exact selection of one bucket by its select blocks together (same algorithm as the exact
// path: three radix rounds over the key, then an ordered emit), each on its own group's
// element range; four barriers.  Returns false when a barrier wait timed out.
// `at`: the bucket's first word of blk_above and blk_eq; restore() puts the group's values back.
template <int THREADS, class Restore, class Lds>
__device__ __forceinline__ bool select_exact_group(BucketsArg bk, const Geometry& g, const Workspace& w, uint32_t b,
                                                   uint32_t grp, const FusedGeo& fg, uint64_t at,
                                                   Restore&& restore, Lds& L, uint64_t limit_ticks) {
    uint32_t* st = w.state + (uint64_t)b * kStateWords;
    const uint64_t bn = fg.bn;
    float* rp = bucket_residual(g, bk, b);
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    const uint64_t below = (1ull << lane) - 1ull;
    const uint64_t e0 = (uint64_t)grp * fg.tpg * kFTile;
    const uint64_t e1r = e0 + (uint64_t)fg.tpg * kFTile;
    const uint64_t e1 = e1r < bn ? e1r : bn;
    // 1: put back what the streaming blocks stored as 0.0f in this group's tiles
    restore();
    __syncthreads();  // a block only ever reads the range it restored itself: plain accesses
    // 2: radix select; every wavefront walks a contiguous quarter of the group's range
    constexpr int NW = THREADS / kWave;
    const uint64_t quarter = ((e1 - e0 + NW - 1) / NW + kWave - 1) / kWave * kWave;
    const uint64_t ws0 = e0 + (uint64_t)wave * quarter < e1 ? e0 + (uint64_t)wave * quarter : e1;
    const uint64_t ws1 = ws0 + quarter < e1 ? ws0 + quarter : e1;
    auto walk = [&](auto&& f) {
        constexpr int B = 8;
#pragma unroll 1
        for (uint64_t base = ws0; base < ws1; base += (uint64_t)B * kWave) {
            uint32_t v[B];
#pragma unroll
            for (int j = 0; j < B; j++) {
                const uint64_t i = base + (uint64_t)j * kWave + lane;
                v[j] = i < ws1 ? f2u(rp[i]) : 0u;
            }
#pragma unroll
            for (int j = 0; j < B; j++) {
                const uint64_t i = base + (uint64_t)j * kWave + lane;
                if (base + (uint64_t)j * kWave < ws1) f(i, v[j], i < ws1);  // wave-uniform
            }
        }
    };
    uint32_t* lh = L.lh;
    uint32_t* gh = w.hist + (uint64_t)b * kHistWords;  // cleared by the bucket's sample block
    uint32_t prefix = 0, remaining = fg.k;
#pragma unroll 1
    for (int round = 0; round < 3; round++) {
        const int bins = round == 0 ? kBins0 : kBinsR;
        const int shift = round == 0 ? 20 : (round == 1 ? 10 : 0);
        const int hi_shift = round == 0 ? 31 : shift + 10;
        uint32_t* ghr = gh + (round == 0 ? 0 : (round == 1 ? kBins0 : kBins0 + kBinsR));
        for (int i = threadIdx.x; i < kBins0; i += THREADS) lh[i] = 0;
        __syncthreads();
        walk([&](uint64_t, uint32_t v, bool valid) {
            const uint32_t key = v & 0x7FFFFFFFu;
            wave_hist_add(lh, valid && (key >> hi_shift) == (prefix >> hi_shift), (key >> shift) & (uint32_t)(bins - 1));
        });
        __syncthreads();
        for (int i = threadIdx.x; i < bins; i += THREADS) {
            const uint32_t c = lh[i];
            if (c) __hip_atomic_fetch_add(&ghr[i], c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (!bucket_barrier(st + S_BARF + round, fg.ng, &L.flag, limit_ticks)) return false;
        for (int i = threadIdx.x; i < bins; i += THREADS) lh[i] = ld_agent(&ghr[i]);
        __syncthreads();
        uint32_t left, bin;
        if (round == 0) bin = pick_bin<kBins0, THREADS>(lh, remaining, 0, &left, L.scratch);
        else bin = pick_bin<kBinsR, THREADS>(lh, remaining, 0, &left, L.scratch);
        prefix |= bin << shift;
        remaining = left;
    }
    const uint32_t T = prefix, need = remaining;
    // 3: keys above and at the threshold per wavefront range, per group, and in the groups before
    uint32_t gt_w = 0, eq_w = 0;  // wave-uniform
    walk([&](uint64_t, uint32_t v, bool valid) {
        const uint32_t key = v & 0x7FFFFFFFu;
        gt_w += (uint32_t)__popcll(__ballot(valid && key > T));
        eq_w += (uint32_t)__popcll(__ballot(valid && key == T));
    });
    uint32_t* wsum = lh;  // LDS words free again: [0..NW) above, [NW..2NW) equal
    __syncthreads();
    if (lane == 0) { wsum[wave] = gt_w; wsum[NW + wave] = eq_w; }
    __syncthreads();
    uint32_t gt_run = 0, eq_run = 0, gt_blk = 0, eq_blk = 0;
#pragma unroll
    for (int i = 0; i < NW; i++) {
        if (i < wave) { gt_run += wsum[i]; eq_run += wsum[NW + i]; }
        gt_blk += wsum[i];
        eq_blk += wsum[NW + i];
    }
    if (threadIdx.x == 0) {
        st_agent(&w.blk_above[at + grp], gt_blk);
        st_agent(&w.blk_eq[at + grp], eq_blk);
    }
    if (!bucket_barrier(st + S_BARF + 3, fg.ng, &L.flag, limit_ticks)) return false;
    {
        static_assert(kMaxGroups <= THREADS, "one thread per group of the bucket");
        const uint32_t vg = threadIdx.x < grp ? ld_agent(&w.blk_above[at + threadIdx.x]) : 0u;
        const uint32_t ve = threadIdx.x < grp ? ld_agent(&w.blk_eq[at + threadIdx.x]) : 0u;
        uint32_t gt_before, eq_before;
        block_exclusive_scan_n<THREADS>(vg, L.scratch, &gt_before);
        block_exclusive_scan_n<THREADS>(ve, L.scratch, &eq_before);
        gt_run += gt_before;
        eq_run += eq_before;
    }
    // 4: this wavefront's picks, in index order
    uint32_t* out = bucket_wire(g, bk, b);
    walk([&](uint64_t i, uint32_t v, bool valid) {
        const uint32_t key = v & 0x7FFFFFFFu;
        const bool is_gt = valid && key > T, is_eq = valid && key == T;
        const uint64_t mg = __ballot(is_gt), me = __ballot(is_eq);
        const uint32_t gt_b = gt_run + (uint32_t)__popcll(mg & below);
        const uint32_t eq_b = eq_run + (uint32_t)__popcll(me & below);
        if (is_gt || (is_eq && eq_b < need)) {
            const uint32_t pos = gt_b + (eq_b < need ? eq_b : need);
            out[1 + 2 * (uint64_t)pos] = (uint32_t)i;
            out[2 + 2 * (uint64_t)pos] = v;
            rp[i] = 0.0f;
        }
        gt_run += (uint32_t)__popcll(mg);
        eq_run += (uint32_t)__popcll(me);
    });
    if (grp == 0 && threadIdx.x == 0) {
        st[S_T] = T;
        st[S_NEED] = need;
    }
    return true;
}


}  // namespace mcclhip
