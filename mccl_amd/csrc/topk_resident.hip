// Top-k compress of buckets that fit the register file: one launch, one pass over memory.
//
// Semantics and ordering as in topk.hip (csrc/compression/TopKCompression.cpp:38-120).
//
// A bucket is cut into blocks of 4096 * V consecutive elements; a block loads grad and residual
// once and keeps its sums in registers until the bucket's threshold is known, then writes residual
// and payload once.  The threshold is found by radix selection over the key's bits: a round
// histograms the keys inside the current key range into 2048 bins in LDS, the blocks add theirs into
// the bucket's histogram in memory, meet at a counter barrier and all pick the same bin.  When the
// picked bin holds at most kRList elements they are gathered into one list, in which every block finds the
// threshold by itself; otherwise the next round splits the bin, down to a single key whose ties are taken in
// index order.  The first round covers a window around the threshold taken from a sample (large
// buckets; the rounds restart on the full key range if it misleads) or every key (small ones); a
// one-block bucket needs no memory but its own.  Any ratio and any distribution takes this path:
// nothing depends on how the keys are spread.
//
// What bounds it is latency, not bandwidth: round trips of 0.6 us to memory that the XCDs share, and sixteen wavefronts
// on four SIMDs, in which 150 instructions take a microsecond.  One bucket of 65,537 elements, us from the first block's
// start: sums loaded 1.1, first round's histogram in LDS 2.3, added up and the blocks met 4.0, bin picked 5.0, listed 5.9,
// met 7.7, threshold 9.5, picks counted 10.0, stored 10.4; of 1 M elements, whose window is published at 6.0, 17.9.
// Per call, with lists of 1024 that were ranked as a whole up to 96, a wait for the lead block in front of the first
// histogram, and picks counted through bits in LDS / so: 1000 elements 6.9 / 6.1 us, 4096 7.3 / 6.9, 8192 (then in two blocks)
// 12.0 / 8.7, 16,384 12.2 / 10.7, 65,537 14.1 / 12.7, 262,144 16.8 / 15.8, 1 M 21.1 / 20.8, 2 M 25.0 / 24.5; at a ratio of
// 5 % 65,537 14.5 / 13.2.  Blocks of 512 threads with twice the vectors are no faster (65,537 12.9, 1 M 21.8), of 256 slower.
//
// The blocks of a bucket wait for one another, so they have to be resident together, whatever else the
// GPU runs.  At 64 registers, 49 KiB of LDS and 1024 threads two blocks fit a CU: 512 the GPU, 64 an XCD.  A
// launch has at most resident_limit of them that wait (topk_route.h): a quarter of those slots, as
// many launches as a process's four hardware queues can have under way.  They are consecutive in the
// grid and dealt to the XCDs in turn, at most 16 to each.  So on every XCD, for any launches under way
// and in any order of dispatch, the blocks that wait are at most as many as its slots, and everything
// else that holds a slot - lead blocks, buckets of one block, other kernels - ends without waiting
// for these.  A block that is not yet dispatched therefore finds a slot, all blocks of every bucket
// come to be resident, and their barriers fill.  (The order of buckets within a launch does not give that: of two
// launches of several hundred blocks one can fill XCD 0 and the other XCD 1, each with buckets that miss
// blocks on the other.)  On a stream that is confined to some of the CUs or has a priority no bucket of several
// blocks takes this path (stream_limit).
#include "topk_common.hip.h"

#include <algorithm>
#include <cstdlib>
#include <type_traits>

namespace mcclhip {

namespace {

constexpr int kRThreads = 1024;
constexpr int kRWaves = kRThreads / kWave;
constexpr int kRBits = 11;
constexpr int kRBins = 1 << kRBits;  // bins of one round
constexpr int kRRank = 64;           // a list longer than this is split before it is ranked
static_assert(kRBins == 2 * kRThreads, "a thread owns two bins");
static_assert(kRList == 2 * kRThreads, "a thread has two entries");

struct ResidentLds {
    uint32_t lh[kRBins + 4] __attribute__((aligned(16)));  // a round's histogram, [kRBins] = keys above the range
    union {
        struct {
            uint64_t list[kRList];             // the picked bin's elements
            uint64_t sub[kRRank];              // ... those that are ranked
            uint32_t rank[kRRank];
        };
        SampleLds<kRThreads> s;
    };
    uint32_t scratch[kRWaves];
    uint32_t pick[3];                          // bin, picks left inside it, elements inside it
    uint32_t win[4];
    uint32_t flag, count, base;
    uint64_t cut;
};

// Exclusive scan of one value per thread over the block; smem: kRWaves words.  (The sums of the
// wavefronts are scanned by a wavefront's lanes: sixteen of them read one by one would take sixteen
// registers.)
__device__ __forceinline__ uint32_t block_scan(uint32_t v, uint32_t* smem, uint32_t* total) {
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const uint32_t inc = wave_inclusive_scan(v);
    if (lane == kWave - 1) smem[wave] = inc;
    __syncthreads();
    const uint32_t s = lane < kRWaves ? smem[lane] : 0u;
    const uint32_t sums = wave_inclusive_scan(s);
    __syncthreads();
    *total = (uint32_t)__builtin_amdgcn_readlane((int)sums, kWave - 1);
    return (uint32_t)__builtin_amdgcn_readlane((int)(sums - s), wave) + inc - v;
}
__device__ __forceinline__ uint32_t block_sum(uint32_t v, uint32_t* smem) {
    uint32_t total;
    block_scan(v, smem, &total);
    return total;
}

// Counting bins from the top, in which the running count reaches r: res = {bin, picks left inside it,
// elements inside it}.  `two` = bins 2046 - 2 t and 2047 - 2 t of thread t, `above` = elements above
// all bins.  Returns the elements in all bins; res is untouched when they do not reach r.
__device__ __forceinline__ uint32_t pick_bin2(u2a two, uint32_t above, uint32_t r, uint32_t* scratch, uint32_t* res) {
    uint32_t total;
    uint32_t run = block_scan(two[0] + two[1], scratch, &total) + above;
#pragma unroll
    for (int q = 1; q >= 0; q--) {
        if (run < r && r <= run + two[q]) {
            res[0] = 2 * (kRThreads - 1 - threadIdx.x) + q;
            res[1] = r - run;
            res[2] = two[q];
        }
        run += two[q];
    }
    __syncthreads();
    return total;
}

// All threads of block x of the bucket; every store and atomic of the block has arrived when it is
// counted.  Atomics on one cache line are carried out one after the other, some 25 ns each: the
// arrivals go to eight lines, and eight lanes read them at once (2 M elements, 123 blocks, one line
// against eight: barrier after the histogram 6.3 / 5.0 us, after the list 4.0 / 3.0; a flag word per
// block instead of counters 5.8 and 3.5).  What is left of the first is the histogram's own 64 lines,
// to which every block adds: fewer bins take as long, copies of it give back in reading what they save.
__device__ __forceinline__ void resident_arrive(uint32_t* counters, uint32_t x) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_fetch_add(counters + 64 * (x % kRBarLines), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool resident_barrier(uint32_t* counters, uint32_t parties, uint32_t x, uint32_t* flag, uint64_t limit_ticks) {
    resident_arrive(counters, x);
    if (threadIdx.x < kWave) {
        const uint32_t lane = threadIdx.x;
        const bool reads = lane < kRBarLines && lane < parties;
        const uint32_t want = (parties - lane + kRBarLines - 1) / kRBarLines;  // blocks x with x % kRBarLines == lane
        uint64_t t0 = 0;
        uint32_t ok = 1, polls = 0;
        while (__ballot(reads && ld_agent(counters + 64 * lane) < want)) {
            __builtin_amdgcn_s_sleep(1);
            if ((++polls & 255u) == 0) {
                const uint64_t now = (uint64_t)wall_clock64();
                if (t0 == 0) t0 = now;
                else if (now - t0 > limit_ticks) {
                    ok = 0;
                    break;
                }
            }
        }
        if (lane == 0) *flag = ok;
    }
    __syncthreads();
    return *flag != 0;
}

// grid: a lead block for each of the first `nlead` buckets, then bucket by bucket its blocks.
template <int V>
__global__ __launch_bounds__(kRThreads, 8) void k_topk_resident(Buckets, Geometry g, Workspace w, uint32_t nlead, uint32_t epoch,
                                                                uint32_t published, uint64_t limit_ticks) {
    constexpr uint32_t PER = kRThreads * 4 * V;  // elements of a block
    // Buckets of this many elements start from a sampled window, which costs about 4 us and saves a round.
    // With a sample and without, us: one of 262,144 elements 16.4 / 16.0, of 300,000 17.0 / 15.9, of 400,000 17.5 / 16.6, of 450,000 17.7 /
    // 17.0, of 500,000 17.5 / 17.9, of 700,000 19.1 / 19.8, of 1 M 20.2 / 22.2, of 2 M 24.1 / 27.6, 2 x 1 M 21.6 / 24.5; 8 x 70,000 16.5 / 16.0, 30 x 33,000 18.2 / 18.8,
    // 3 x 300,000 17.9 / 18.0.  (Several buckets of more cross sooner than one does, 8 x 262,143 20.3 / 22.0, 5 x 400,000 20.4 / 22.1, and go without it
    // all the same: the rule asks for the bucket alone.)
    constexpr uint32_t kSampleMin = 1u << 19;
    const BucketsArg bk = buckets_arg();
    __shared__ ResidentLds L;
    const int lane = threadIdx.x & (kWave - 1);
    const bool lead = blockIdx.x < nlead;
    uint32_t b = blockIdx.x, x = 0;  // bucket, block of the bucket
    if (!lead) {
        const uint32_t j = blockIdx.x - nlead;
        if (g.listed) {
            b = listed_bucket(bk->lfirst, j, &x);
        } else {
            const uint32_t per_bucket = (uint32_t)((g.bucket_elems + PER - 1) / PER);
            b = j / per_bucket;
            x = j - b * per_bucket;
        }
    }
    const uint64_t bn = bucket_count(g, bk, b);
    const uint32_t nblk = (uint32_t)((bn + PER - 1) / PER);
    uint32_t* st = w.state + (uint64_t)b * kStateWords;
    uint32_t* const mem = w.rmem + (uint64_t)b * kRWords;
    float* const rbase = bucket_residual(g, bk, b);
    const float* const gbase = bucket_grad(g, bk, b);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const uint32_t k = bucket_k(g, bk, b);
    if (lead) {
        // ---- lead block: clears what the others add into and publishes the first round's key range
        if (nblk == 1) return;
        auto clear = [&](uint32_t from, uint32_t to) {
            for (uint32_t i = from / 4 + threadIdx.x; i < to / 4; i += kRThreads) store16_agent(mem + i * 4, u4a{0u, 0u, 0u, 0u});
        };
        // Before the window is published: what the blocks touch before they have met once.  The rest is
        // cleared after it, and the lead block takes part in their first barrier.
        auto clear_first = [&] {
            clear(0, kRRow0 + kRRow);
            if (threadIdx.x == 0) {
                st_agent(st + S_OK, 0u);
                st_agent(st + S_TIMEOUT, 0u);
            }
        };
        SampleWindow win = {0u, 0x7FFFFFFFu, 0u};
        if (bn >= kSampleMin) win = sample_window<kRThreads>(gbase, rbase, bn, k, L.s, clear_first);
        else clear_first();
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x == 0) store16_agent(st + S_LO_KEY, u4a{win.lo, win.hi, 0u, published});
        clear(kRRow0 + kRRow, kRCnt);
        resident_arrive(mem, nblk);
        return;
    }
    const uint64_t b0 = (uint64_t)x * PER;                       // the block's first element
    const uint32_t e0 = (uint32_t)wave * (256 * V) + 4 * lane;   // this lane's first element, from b0; vector u is 256 u further
    const bool full = b0 + PER <= bn;
    uint32_t* out = bucket_wire(g, bk, b);

    const auto clear_histogram = [&] {
        for (int i = threadIdx.x; i < (kRBins + 4) / 4; i += kRThreads) ((u4a*)L.lh)[i] = u4a{0u, 0u, 0u, 0u};
    };
    clear_histogram();
    if (threadIdx.x == 0) L.count = 0;
    // ---- load: grad + residual, once ----------------------------------------------------------
    u4a a[V];
    {
        // wave-uniform bases: the lanes only differ by a 32-bit offset
        const float* gp = gbase + b0 + (uint32_t)wave * (256 * V);
        const float* rp = rbase + b0 + (uint32_t)wave * (256 * V);
        const uint32_t l4 = 4 * lane;
        const uint32_t left = full ? PER : (uint32_t)(bn - b0);
        auto load = [&](auto whole) {
            constexpr bool WHOLE = decltype(whole)::value;
            u4a rv[V];
#pragma unroll
            for (int u = 0; u < V; u++) {
                a[u] = rv[u] = u4a{0u, 0u, 0u, 0u};
                if (WHOLE || e0 + 256 * u + 4 <= left) {
                    a[u] = __builtin_nontemporal_load((const u4u4*)(gp + 256 * u + l4));
                    rv[u] = __builtin_nontemporal_load((const u4u4*)(rp + 256 * u + l4));
                }
            }
#pragma unroll
            for (int u = 0; u < V; u++) {
#pragma unroll
                for (int q = 0; q < 4; q++) a[u][q] = f2u(u2f(a[u][q]) + u2f(rv[u][q]));
                if constexpr (!WHOLE) {
                    // Elements past the bucket's end count as +0.0 at indices above every real one: a zero
                    // key is the smallest, and ties go to the lower index, so they are never picked.
                    const uint32_t e = e0 + 256 * u;
                    if (e < left && e + 4 > left) {  // the bucket's partial vector
#pragma unroll
                        for (int q = 0; q < 3; q++)
                            if (e + q < left) a[u][q] = f2u(gp[256 * u + l4 + q] + rp[256 * u + l4 + q]);
                    }
                }
            }
        };
        if (full) load(std::true_type{});
        else load(std::false_type{});
    }
    // Vector u of the lane.  Every pass over the elements starts each vector with a value the compiler
    // knows nothing about: it would otherwise carry derived values (keys, comparisons) of all the
    // vectors from one pass to the next, in registers that are not there.
    auto vec = [&](int u) -> u4a {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" : "+v"(a[u]));
        return a[u];
    };
    auto give_up = [&] { fused_give_up(w, st, out); };

    // ---- rounds -----------------------------------------------------------------------------------
    uint32_t base = 0, span = 0x80000000u;  // keys base .. base + span - 1
    bool window = false;
    // Thread 0 waits for the lead block, the others for it at the next barrier: where there is a window to be had before
    // the first histogram, else only before it is added to the bucket's, which the lead block has cleared by then.
    const bool sampled = nblk > 1 && bn >= kSampleMin;
    const auto wait_for_lead = [&] {
        if (threadIdx.x == 0) {
            const u4a wn = wait_window<2>(st, epoch, limit_ticks);
            L.win[0] = wn[0]; L.win[1] = wn[1]; L.win[3] = wn[3];
        }
    };
    if (sampled) {
        wait_for_lead();
        __syncthreads();
        if (!L.win[3]) {
            give_up();
            return;
        }
        base = L.win[0];
        span = L.win[1] - L.win[0] + 1;
        window = span != 0x80000000u;
    }
    uint32_t r = k;         // picks still to place among the keys of the range and above it
    bool first = true;      // the keys above the range are not accounted for in r yet
    uint32_t sh, bin, m, row = 0;
    for (;;) {
        sh = 32 - __clz(span - 1);
        if (span == 1) sh = 0;
        sh = sh > (uint32_t)kRBits ? sh - kRBits : 0;
        __syncthreads();
        if (base == 0) {
            // every key: zeros, which would all add to one LDS word, are counted by the wavefront
            uint32_t zeros = 0;
#pragma unroll
            for (int u = 0; u < V; u++) {
                const u4a v = vec(u);
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const uint32_t key = v[q] & 0x7FFFFFFFu;
                    zeros += (uint32_t)__popcll(__ballot(key == 0));
                    if (key != 0) atomicAdd(&L.lh[key < span ? key >> sh : (uint32_t)kRBins], 1u);
                }
            }
            if (lane == 0 && zeros) atomicAdd(&L.lh[0], zeros);
        } else {
#pragma unroll
            for (int u = 0; u < V; u++) {
                const u4a v = vec(u);
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const uint32_t d = (v[q] & 0x7FFFFFFFu) - base;
                    if ((int)d >= 0) atomicAdd(&L.lh[d < span ? d >> sh : (uint32_t)kRBins], 1u);
                }
            }
        }
        if (nblk > 1 && !sampled && row == 0) wait_for_lead();
        __syncthreads();
        u2a all = ((const u2a*)L.lh)[kRThreads - 1 - threadIdx.x];
        uint32_t above = first ? L.lh[kRBins] : 0u;
        if (nblk > 1) {
            if (row == 0 && !L.win[3]) {
                give_up();
                return;
            }
            uint32_t* const gh = mem + kRRow0 + row * kRRow;
            const uint64_t c = ((const uint64_t*)L.lh)[threadIdx.x];
            if (c) __hip_atomic_fetch_add((uint64_t*)gh + threadIdx.x, c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // two bins
            if (threadIdx.x == 0 && above) __hip_atomic_fetch_add(gh + kRBins, above, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (!resident_barrier(mem + kRBarWords * row, row == 0 ? nblk + 1 : nblk, x, &L.flag, limit_ticks)) {
                give_up();
                return;
            }
            row++;
            const uint64_t two = ld_agent64((const uint64_t*)gh + (kRThreads - 1 - threadIdx.x));
            above = first ? ld_agent(gh + kRBins) : 0u;
            all = u2a{(uint32_t)two, (uint32_t)(two >> 32)};
        }
        const uint32_t total = pick_bin2(all, above, r, L.scratch, L.pick);
        if (window && first && (r <= above || r > above + total)) {  // the sample misled: every key, from the start
            base = 0;
            span = 0x80000000u;
            window = false;
            clear_histogram();
            continue;
        }
        bin = L.pick[0];
        r = L.pick[1];
        m = L.pick[2];
        first = false;
        base += bin << sh;
        const uint32_t left = span - (bin << sh);
        span = left < (1u << sh) ? left : 1u << sh;
        if (m <= (uint32_t)kRList || span == 1) break;
        clear_histogram();  // (what it held is in registers, and the pick lies behind two barriers)
    }

    // ---- the picked bin -----------------------------------------------------------------------------
    static_assert(PER / 32 <= kRThreads, "a thread for each 32 elements");
    const bool tied = m > (uint32_t)kRList;  // one key, more often than the list holds: ties by index
    const uint32_t eq = L.lh[bin];           // this block's elements in the bin
    uint32_t T, istar, before;  // picks: key > T, or key == T and index <= istar; picks of earlier blocks
    {
        uint64_t* const cnts = (uint64_t*)(mem + kRCnt);
        // where the block's elements go in the list (asked for first: the answer takes as long as what follows)
        uint32_t list_at = 0;
        if (nblk > 1 && threadIdx.x == 0 && !tied && eq)
            list_at = __hip_atomic_fetch_add(mem + kRFill, eq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (!tied && eq) {  // block-uniform
#pragma unroll
            for (int u = 0; u < V; u++) {
                const u4a v = vec(u);
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const uint32_t key = v[q] & 0x7FFFFFFFu;
                    if (key - base < span) {
                        const uint32_t i = atomicAdd(&L.count, 1u);
                        // larger is picked earlier: key, then lower index
                        if (i < (uint32_t)kRList) L.list[i] = ((uint64_t)key << 32) | (uint32_t)~((uint32_t)b0 + e0 + 256 * u + q);
                    }
                }
            }
        }
        uint64_t c = 0;  // of an earlier block: elements above the bin, inside the bin
        if (nblk > 1) {
            const u2a own = ((const u2a*)L.lh)[threadIdx.x];
            uint32_t s = threadIdx.x == 0 ? L.lh[kRBins] : 0u;
#pragma unroll
            for (int q = 0; q < 2; q++) s += 2 * threadIdx.x + q > bin ? own[q] : 0u;
            if (threadIdx.x == 0) L.base = list_at;
            const uint32_t gt = block_sum(s, L.scratch);
            if (threadIdx.x == 0) st_agent64(cnts + x, ((uint64_t)gt << 32) | eq);
            if (!tied) {
                uint64_t* gl = (uint64_t*)(mem + kRListAt) + L.base;
                for (uint32_t i = threadIdx.x; i < eq && L.base + i < (uint32_t)kRList; i += kRThreads) st_agent64(gl + i, L.list[i]);
            }
            if (!resident_barrier(mem + kRBarWords * row, nblk, x, &L.flag, limit_ticks)) {
                give_up();
                return;
            }
            if (threadIdx.x < x) c = ld_agent64(cnts + threadIdx.x);
        } else {
            __syncthreads();
        }
        if (!tied) {
            // The r-th largest entry: by radix rounds over key and index (entries differ in their index), until few enough
            // share a prefix to rank them, by counting for each of them those that reach it.
            uint64_t me[2];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const uint32_t i = (uint32_t)j * kRThreads + threadIdx.x;
                me[j] = i >= m ? 0ull : nblk > 1 ? ld_agent64((const uint64_t*)(mem + kRListAt) + i) : L.list[i];
            }
            if (threadIdx.x == 0) {
                L.count = 0;
                L.cut = kNoCut;
            }
            if (threadIdx.x < (uint32_t)kRRank) L.rank[threadIdx.x] = 0;
            const uint64_t low = (uint64_t)base << 32;
            uint32_t rm = m, rr = r;
            int bits = 32 + (span > 1 ? 32 - __clz((int)(span - 1)) : 0);  // of the entries, less the smallest key's, still open
            uint64_t prefix = 0;
            const auto shares = [&](int j) {
                return (uint32_t)j * kRThreads + threadIdx.x < m && (me[j] - low) >> bits == prefix >> bits;
            };
#pragma unroll 1
            while (rm > (uint32_t)kRRank && bits) {  // block-uniform; ends whatever the scratch memory holds
                const int at = bits > kRBits ? bits - kRBits : 0;
                __syncthreads();
                ((u2a*)L.lh)[threadIdx.x] = u2a{0u, 0u};
                __syncthreads();
#pragma unroll
                for (int j = 0; j < 2; j++)
                    if (shares(j)) atomicAdd(&L.lh[(uint32_t)((me[j] - low ^ prefix) >> at)], 1u);
                __syncthreads();
                pick_bin2(((const u2a*)L.lh)[kRThreads - 1 - threadIdx.x], 0u, rr, L.scratch, L.pick);
                prefix |= (uint64_t)L.pick[0] << at;
                rr = L.pick[1];
                rm = L.pick[2];
                bits = at;
            }
            rm = rm < (uint32_t)kRRank ? rm : (uint32_t)kRRank;
            __syncthreads();
#pragma unroll
            for (int j = 0; j < 2; j++)
                if (shares(j)) {
                    const uint32_t i = atomicAdd(&L.count, 1u);
                    if (i < (uint32_t)kRRank) L.sub[i] = me[j];
                }
            __syncthreads();
            {
                // an entry a lane, and for each wavefront a part of the entries to compare it with
                static_assert(kRRank == kWave, "a lane for each entry");
                const uint32_t per = (rm + kRWaves - 1) / kRWaves, from = per * wave, to = from + per < rm ? from + per : rm;
                if (from < to) {
                    const uint64_t mine = L.sub[lane];
                    const uint32_t rank = reaching_entries(L.sub, from, to, mine);
                    if ((uint32_t)lane < rm && rank) atomicAdd(&L.rank[lane], rank);
                }
                __syncthreads();
                if (threadIdx.x < rm && L.rank[threadIdx.x] == rr) L.cut = L.sub[threadIdx.x];
                __syncthreads();
            }
            const uint64_t cut = L.cut;
            T = (uint32_t)(cut >> 32);
            istar = ~(uint32_t)cut;
            before = 0;
            if (nblk > 1) {
                uint32_t mine = (uint32_t)(c >> 32);
#pragma unroll
                for (int j = 0; j < 2; j++)
                    mine += (uint32_t)j * kRThreads + threadIdx.x < m && me[j] >= cut && ~(uint32_t)me[j] < (uint32_t)b0 ? 1u : 0u;
                before = block_sum(mine, L.scratch);
            }
        } else {
            T = base;
            uint32_t gt_before = 0, eq_before = 0;
            if (nblk > 1) {
                gt_before = block_sum((uint32_t)(c >> 32), L.scratch);
                eq_before = block_sum((uint32_t)c, L.scratch);
            }
            const uint32_t quota = r > eq_before ? (r - eq_before < eq ? r - eq_before : eq) : 0u;
            before = gt_before + (eq_before < r ? eq_before : r);
            istar = 0xFFFFFFFFu;
            if (quota == 0) {
                T = base + 1;
            } else if (quota < eq) {
                // the one block in which the ties run out: the quota-th of its equal keys, from a bit per element
                __syncthreads();
                if (threadIdx.x < PER / 32) L.lh[threadIdx.x] = 0;
                __syncthreads();
#pragma unroll
                for (int u = 0; u < V; u++) {
                    const u4a v = vec(u);
                    uint32_t nib = 0;
#pragma unroll
                    for (int q = 0; q < 4; q++) nib |= ((v[q] & 0x7FFFFFFFu) == base ? 1u : 0u) << q;
                    const uint32_t e = e0 + 256 * u;
                    if (nib) atomicOr(&L.lh[e >> 5], nib << (e & 31));
                }
                __syncthreads();
                uint32_t bitsleft = threadIdx.x < PER / 32 ? L.lh[threadIdx.x] : 0u, tot;
                const uint32_t c = __popc(bitsleft);
                const uint32_t run = block_scan(c, L.scratch, &tot);
                if (run < quota && quota <= run + c) {
                    for (uint32_t n = quota - run; n > 1; n--) bitsleft &= bitsleft - 1;
                    L.flag = (uint32_t)b0 + 32 * threadIdx.x + (uint32_t)__ffs((int)bitsleft) - 1u;
                }
                __syncthreads();
                istar = L.flag;
            }
        }
    }

    // ---- picks, counted over the wavefront's vectors (256 consecutive elements each) and the block's wavefronts, then
    // residual and payload
    uint32_t nibs = 0;  // a bit per element, four of each vector
    uint32_t inc[(V + 1) / 2];  // picks of vectors 2 i and 2 i + 1 in the lanes up to this one, 16 bits each
#pragma unroll
    for (int i = 0; i < (V + 1) / 2; i++) inc[i] = 0;
#pragma unroll
    for (int u = 0; u < V; u++) {
        const u4a v = vec(u);
        const uint32_t e = e0 + 256 * u;
        uint32_t nib = 0;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t key = v[q] & 0x7FFFFFFFu;
            nib |= (key >= T + ((uint32_t)b0 + e + q > istar ? 1u : 0u) ? 1u : 0u) << q;
        }
        nibs |= nib << (4 * u);
        inc[u / 2] += (uint32_t)__popc(nib) << (16 * (u & 1));
    }
    uint32_t total = 0;  // of the wavefront
#pragma unroll
    for (int i = 0; i < (V + 1) / 2; i++) {
        inc[i] = wave_inclusive_scan(inc[i]);
        const uint32_t all = (uint32_t)__builtin_amdgcn_readlane((int)inc[i], kWave - 1);
        total += (all & 0xFFFFu) + (all >> 16);
    }
    if (lane == 0) L.scratch[wave] = total;
    __syncthreads();
    uint32_t pos0 = before;  // the position of the wavefront's first pick, then of each vector's
    {
        const uint32_t t = lane < kRWaves ? L.scratch[lane] : 0u;
        pos0 += (uint32_t)__builtin_amdgcn_readlane((int)(wave_inclusive_scan(t) - t), wave);
    }
    float* const rp = rbase + b0 + (uint32_t)wave * (256 * V);
    const uint32_t l4 = 4 * lane;
    const uint32_t left = full ? PER : (uint32_t)(bn - b0);
#pragma unroll
    for (int u = 0; u < V; u++) {
        const u4a v = vec(u);
        const uint32_t e = e0 + 256 * u;
        const uint32_t nib = (nibs >> (4 * u)) & 15u;
        u4a z;
#pragma unroll
        for (int q = 0; q < 4; q++) z[q] = nib >> q & 1u ? 0u : v[q];
        if (e + 4 <= left) __builtin_nontemporal_store(z, (u4u4*)(rp + 256 * u + l4));
        else if (e < left) {
#pragma unroll
            for (int q = 0; q < 3; q++)
                if (e + q < left) rp[256 * u + l4 + q] = u2f(z[q]);
        }
        const uint32_t up_to = inc[u / 2] >> (16 * (u & 1)) & 0xFFFFu;
        if (nib) {
            uint32_t pos = pos0 + up_to - (uint32_t)__popc(nib);
#pragma unroll
            for (int q = 0; q < 4; q++) {
                if ((nib >> q & 1u) && pos < k) {  // (pos < k whatever the scratch memory held)
                    const u2a pr = {(uint32_t)b0 + e + q, v[q]};
                    *(u2a4*)(out + 1 + 2 * (uint64_t)pos) = pr;
                    pos++;
                }
            }
        }
        pos0 += (uint32_t)__builtin_amdgcn_readlane((int)up_to, kWave - 1);
    }
    if (x == 0 && threadIdx.x == 0 && T == (uint32_t)(kNoCut >> 32)) {
        give_up();  // nothing was picked (a branch where the cut is read takes every call 0.15 us)
    } else if (x == 0 && threadIdx.x == 0) {
        st[S_T] = T;
        st[S_ISTAR] = istar;
        st[S_READY] = 0u;  // a replay of a captured launch carries the same epoch
        if (nblk == 1) st[S_TIMEOUT] = 0u;
        st[S_OK] = 1u;
        if (nblk == 1 || !ld_agent(st + S_TIMEOUT)) out[0] = k;
    }
}

// A replay of a captured launch carries the same epoch.  A run that ends well leaves S_READY zero, one
// that a block gave up may leave it published: the blocks of the next replay would take the old window
// and the old counters for theirs, so a capture records this kernel in front of the launch.  (One
// bucket of 65,537 elements, replayed: 15.9 us, without it 14.3; buckets of one block wait for nobody.)
__global__ __launch_bounds__(kBlock) void k_resident_unpublish(uint32_t* state, uint32_t nbuckets) {
    const uint32_t b = blockIdx.x * kBlock + threadIdx.x;
    if (b < nbuckets) st_agent(state + (uint64_t)b * kStateWords + S_READY, 0u);
}

}  // namespace

bool is_capturing(hipStream_t st) {
    if (!st) return false;  // the null stream cannot be captured, and asking about it can fail while another one is
    hipStreamCaptureStatus s = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &s) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return s != hipStreamCaptureStatusNone;
}

namespace {

// `nlead`: buckets of more than one block, which come first.
template <int V>
void launch_blocks(const Buckets& bk, const Geometry& g, const Workspace& w, uint32_t nlead, uint32_t blocks, uint32_t epoch,
                   uint32_t published, uint64_t limit_ticks, hipStream_t st) {
    if (nlead && is_capturing(st)) k_resident_unpublish<<<(nlead + kBlock - 1) / kBlock, kBlock, 0, st>>>(w.state, nlead);
    k_topk_resident<V><<<nlead + blocks, kRThreads, 0, st>>>(bk, g, w, nlead, epoch, published, limit_ticks);
}

template <int V>
void launch(const Buckets& bk, const Geometry& g, const Workspace& w, uint64_t limit, uint32_t epoch, uint32_t published,
            uint64_t limit_ticks, hipStream_t st) {
    constexpr uint64_t per = kRVecElems * V;
    static_assert(kRVecElems == kRThreads * 4, "one vector per thread");
    if (!g.listed) {
        const uint64_t per_bucket = (g.bucket_elems + per - 1) / per;
        const uint64_t last = g.n_total - (uint64_t)(g.nbuckets - 1) * g.bucket_elems;
        const uint32_t blocks = (uint32_t)((g.nbuckets - 1) * per_bucket + (last + per - 1) / per);
        launch_blocks<V>(bk, g, w, per_bucket > 1 ? g.nbuckets : 0, blocks, epoch, published, limit_ticks, st);
        return;
    }
    // A list goes longest bucket first: it takes longest, and its blocks start while the GPU is empty.
    // Leads before all blocks, no block without a bucket: 24 buckets of 1001 to 1.5 M elements 28.5 us, in
    // the caller's order with as many blocks for each bucket as for the longest 31.1 (both as one launch).
    uint32_t order[kMaxListed];
    longest_first(bk, g.nbuckets, order);
    for (uint32_t done = 0; done < g.nbuckets;) {
        const uint32_t taken = next_launch(bk.lcount, order + done, g.nbuckets - done, per, limit);
        Buckets part = bk;
        uint32_t nlead = 0, blocks = 0;
        for (uint32_t i = 0; i < taken; i++) {
            const uint32_t b = order[done + i];
            place_bucket(&part, i, bk, b, blocks);
            blocks += (uint32_t)((bk.lcount[b] + per - 1) / per);
            if (bk.lcount[b] > per) nlead = i + 1;
        }
        for (uint32_t i = taken; i < kMaxListed; i++) part.lfirst[i] = 0xFFFFFFFFu;
        Workspace pw = w;
        pw.state += (uint64_t)done * kStateWords;
        pw.rmem += (uint64_t)done * kRWords;
        launch_blocks<V>(part, g, pw, nlead, blocks, epoch, published, limit_ticks, st);
        done += taken;
    }
}

// CUs of the stream's mask; all of the device's where there is no mask to be had.
int stream_cus(hipStream_t st) {
    uint32_t mask[32] = {};
    if (hipExtStreamGetCUMask(st, 32, mask) != hipSuccess) {
        (void)hipGetLastError();
        return device_info().num_cus;
    }
    int n = 0;
    for (const uint32_t m : mask) n += __builtin_popcount(m);
    return n;
}

}  // namespace

void longest_first(const Buckets& bk, uint32_t nbuckets, uint32_t* order) {
    for (uint32_t b = 0; b < nbuckets; b++) order[b] = b;
    std::sort(order, order + nbuckets, [&](uint32_t p, uint32_t q) { return bk.lcount[p] != bk.lcount[q] ? bk.lcount[p] > bk.lcount[q] : p < q; });
}

StreamShare stream_share(hipStream_t st) {
    // (asking takes 0.2 us; the null stream's mask is the process's)
    static const int process_cus = stream_cus(nullptr);
    StreamShare share = {process_cus, 0};
    if (st) {
        share.cus = std::min(process_cus, stream_cus(st));
        if (hipStreamGetPriority(st, &share.priority) != hipSuccess) {
            (void)hipGetLastError();
            share.priority = 0;
        }
    }
    return share;
}

uint64_t waiting_limit(const StreamShare& share, uint64_t per_cu) {
    // hardware queues that the process's streams share; HIP's own default is four
    static const uint32_t queues = [] {
        const char* s = std::getenv("GPU_MAX_HW_QUEUES");
        const long q = s ? std::strtol(s, nullptr, 10) : 0;
        return (uint32_t)(q > 0 && q < 1024 ? q : 4);
    }();
    return stream_limit(share, device_info().num_cus, per_cu, queues);
}

uint64_t resident_limit_on(const StreamShare& share) {
    static const uint64_t per_cu = [] {
        int least = 1 << 20;
        for (const void* k : {(const void*)k_topk_resident<1>, (const void*)k_topk_resident<2>, (const void*)k_topk_resident<4>}) {
            int n = 0;
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k, kRThreads, 0) != hipSuccess) n = 0;
            least = n < least ? n : least;
        }
        return (uint64_t)least;
    }();
    return waiting_limit(share, per_cu);
}

void launch_resident(const Buckets& bk, const Geometry& g, const Workspace& w, int vecs, uint64_t limit, uint32_t epoch,
                     uint32_t published, uint64_t limit_ticks, hipStream_t st) {
    switch (vecs) {
        case 1: launch<1>(bk, g, w, limit, epoch, published, limit_ticks, st); break;
        case 2: launch<2>(bk, g, w, limit, epoch, published, limit_ticks, st); break;
        default: launch<4>(bk, g, w, limit, epoch, published, limit_ticks, st); break;
    }
}

}  // namespace mcclhip
