// What the two top-k kernel families (topk.hip: streaming, topk_resident.hip: resident) share:
// the call's geometry, workspace and bucket table, and how blocks of one launch talk to each other.
#pragma once

#include "common.hip.h"
#include "runtime.h"
#include "topk_rank.h"
#include "topk_route.h"

namespace mcclhip {

constexpr int kTile = 4096;    // exact path: elements per compaction tile
constexpr int kBins0 = 2048;   // key[30:20]
constexpr int kBinsR = 1024;   // key[19:10], key[9:0]
constexpr int kHistWords = kBins0 + 2 * kBinsR;
constexpr int kStateWords = 32;
constexpr uint32_t kDense = 0xFFFFFFFFu;  // tile count: more candidates than slots, read the residual range itself
constexpr uint32_t kPoisonK = 0xFFFFFFFFu;    // payload header of a bucket whose selection was abandoned
// resident path (topk_resident.hip): per-bucket scratch, in words
constexpr int kRList = 2048;                  // elements of the picked bin that are selected from as a list
constexpr uint32_t kRRow = 2048 + 64;         // one round's histogram: its bins, the count above them, padding
constexpr uint32_t kRRows = 4;                // a windowed round, three on the full key range (11 + 11 + 9 bits)
constexpr uint32_t kRBars = 6;                // barriers: at most four rounds and the list / ties
constexpr uint32_t kRBarLines = 8;            // counters of a barrier, 256 bytes apart
constexpr uint32_t kRBarWords = 64 * kRBarLines;
constexpr uint32_t kRFill = kRBars * kRBarWords;   // after the barriers: the list's fill counter
constexpr uint32_t kRRow0 = kRFill + 64;
constexpr uint32_t kRCnt = kRRow0 + kRRows * kRRow;           // per block: elements above the bin, inside the bin
constexpr uint32_t kRListAt = kRCnt + 2 * (uint32_t)kRMaxBlocks;
constexpr uint32_t kRWords = kRListAt + 2 * kRList;

// per-bucket state words
enum {
    // single-pass path: the candidate window, published by its sample block with ONE 16-byte store
    S_LO_KEY = 0,         // candidates have key >= this
    S_HI_KEY = 1,         // keys >= this fall into the top coarse bin
    S_THAT = 2,           // predicted threshold key; the streaming blocks store 0.0f for keys >= this
    S_READY = 3,          // the call's epoch number once the other three are valid; 0 after the call, unless a list went in one launch
    S_P0 = 4, S_R0 = 5,   // exact path: key prefix / picks still to place after round 0
    S_P1 = 6, S_R1 = 7,   // after round 1
    S_T = 8, S_NEED = 9,  // exact threshold key, number of keys == T that are taken
    S_ISTAR = 10,         // single-pass path: ties are taken while index <= this
    S_OK = 11,            // single-pass path: 1 when the window selection succeeded for this bucket
    S_EXACT_HIST = 12,    // 1 when hist round 0 holds the full histogram
    S_TIMEOUT = 13,       // single-pass path: a block gave up waiting (result invalid, payload header poisoned)
    S_BARF = 16,          // 16..19: barriers of the exact selection inside the select launch
    S_DONE = 20           // one launch: lines of select blocks that have arrived
};

struct Geometry {
    uint64_t n_total;
    uint64_t bucket_elems;
    uint32_t nbuckets;
    uint32_t tiles;    // exact-path tiles per (full) bucket
    uint32_t k_full;   // k of a bucket with bucket_elems elements
    uint32_t k_last;   // k of the last bucket
    uint32_t listed;   // single-pass path: 1 when the buckets are separate buffers (see Buckets)
    uint32_t ftiles;   // single-pass path: streaming tiles allotted per bucket
    uint32_t gshift;   // single-pass path: at most 1 << gshift groups of tiles per bucket
    uint32_t ngroups;  // single-pass path: groups of the bucket with the most of them (topk_launched_groups)
    uint32_t many;     // single-pass path: 1 when tiles have slots for many candidates (topk_many)
    uint32_t slots;    // single-pass path: candidate slots of a tile
    uint32_t lcapb;    // single-pass path: capacity of one coarse bin's list (entries)
};

struct Workspace {
    // zeroed at the start of every exact-path call; the single-pass path zeroes what it uses itself
    uint32_t* hist;         // [nbuckets][kHistWords]
    uint32_t* state;        // [nbuckets][kStateWords]
    // scratch, written before read
    uint32_t* tile_gt;      // [nbuckets][tiles]
    uint32_t* tile_eq;      // [nbuckets][tiles]
    uint32_t* blk_above;    // [nbuckets][groups] exact selection inside the select launch: keys above the threshold per group
    uint32_t* blk_eq;       // [nbuckets][groups] ... keys equal to the threshold per group
    // single-pass path
    uint32_t* tile_cnt;     // [nbuckets][ftiles] candidates in the tile's slots, or kDense
    uint64_t* slots;        // [nbuckets][ftiles][slots] (bits << 32) | index, index order
    uint32_t* grp_cnt;      // [nbuckets][groups][kCntStride] finished tiles per group (first word of each 256 bytes; one launch: see group_line)
    uint32_t* gsuf;         // [nbuckets][128 bins][groups] a group's candidates in the bins above bin j (one launch: [nbuckets][groups][128 bins])
    uint32_t* bin_fill;     // [nbuckets][128] the bucket's candidates per coarse window bin (= entries of the bin's list)
    uint64_t* blist;        // [nbuckets][127][lcapb] the window's candidates by coarse bin, any order
    uint32_t* rmem;         // [nbuckets][kRWords] resident path
    int* status;            // caller's device word (may be null): receives MCCL_HIP_ERR_TIMEOUT when a block gives up
};

__device__ __forceinline__ uint64_t bucket_count(const Geometry& g, uint32_t b) {
    const uint64_t start = (uint64_t)b * g.bucket_elems;
    const uint64_t left = g.n_total - start;
    return left < g.bucket_elems ? left : g.bucket_elems;
}
__device__ __forceinline__ uint32_t bucket_k(const Geometry& g, uint32_t b) {
    return b + 1 == g.nbuckets ? g.k_last : g.k_full;
}
__device__ __forceinline__ uint32_t key_of(float v) { return f2u(v) & 0x7FFFFFFFu; }

// Where the buckets of a single-pass call live.  Uniform layout: the buckets are
// consecutive ranges of one gradient (mccl_hip_topk_compress).  Listed layout
// (Geometry::listed): every bucket is a buffer of its own with its own length
// (mccl_hip_topk_compress_list); g.bucket_elems is then the longest bucket.
constexpr uint32_t kMaxListed = MCCL_HIP_TOPK_LIST_MAX;
struct Buckets {
    const float* grad;
    float* residual;
    uint8_t* wire;
    uint64_t wire_stride;
    const float* lgrad[kMaxListed];
    float* lresidual[kMaxListed];
    uint8_t* lwire[kMaxListed];
    uint32_t lcount[kMaxListed];
    uint32_t lk[kMaxListed];
    uint32_t lfirst[kMaxListed];  // the bucket's first block in the launch; 0xFFFFFFFF past the list
};
// The kernels index the table by bucket number.  Indexing the by-value parameter would make
// the compiler copy all of it to per-lane scratch memory first (2 KiB per lane, and a launch
// that sets up scratch starts several microseconds later); the kernels read it where it
// already lies instead, in the kernel-argument segment, through scalar loads.  Buckets is
// therefore the FIRST parameter of every kernel that takes one.
typedef const __attribute__((address_space(4))) Buckets* BucketsArg;
__device__ __forceinline__ BucketsArg buckets_arg() { return (BucketsArg)__builtin_amdgcn_kernarg_segment_ptr(); }
__device__ __forceinline__ uint64_t bucket_count(const Geometry& g, BucketsArg bk, uint32_t b) {
    return g.listed ? (uint64_t)bk->lcount[b] : bucket_count(g, b);
}
__device__ __forceinline__ uint32_t bucket_k(const Geometry& g, BucketsArg bk, uint32_t b) {
    return g.listed ? bk->lk[b] : bucket_k(g, b);
}
__device__ __forceinline__ const float* bucket_grad(const Geometry& g, BucketsArg bk, uint32_t b) {
    return g.listed ? bk->lgrad[b] : bk->grad + (uint64_t)b * g.bucket_elems;
}
__device__ __forceinline__ float* bucket_residual(const Geometry& g, BucketsArg bk, uint32_t b) {
    return g.listed ? bk->lresidual[b] : bk->residual + (uint64_t)b * g.bucket_elems;
}
__device__ __forceinline__ uint32_t* bucket_wire(const Geometry& g, BucketsArg bk, uint32_t b) {
    return (uint32_t*)(g.listed ? bk->lwire[b] : bk->wire + (uint64_t)b * bk->wire_stride);
}
// Bucket of block j of a list's launch, and which of the bucket's blocks it is.  On the scalar unit: the
// block's loads wait for it.
__device__ __forceinline__ uint32_t listed_bucket(const __attribute__((address_space(4))) uint32_t* firsts, uint32_t j, uint32_t* x) {
    uint32_t b = 0;
    *x = j;
    for (uint32_t c = 0; c < kMaxListed && firsts[c] <= j; c += 16) {
#pragma unroll
        for (uint32_t i = 0; i < 16; i++) {
            const uint32_t first = firsts[c + i];
            if (first <= j) {
                b = c + i;
                *x = j - first;
            }
        }
    }
    return b;
}


// The list's buckets by length, longest first.
void longest_first(const Buckets& bk, uint32_t nbuckets, uint32_t* order);
// Entry i of the table `to` is entry b of `from`; its blocks start at `first`.
inline void place_bucket(Buckets* to, uint32_t i, const Buckets& from, uint32_t b, uint32_t first) {
    to->lgrad[i] = from.lgrad[b];
    to->lresidual[i] = from.lresidual[b];
    to->lwire[i] = from.lwire[b];
    to->lcount[i] = from.lcount[b];
    to->lk[i] = from.lk[b];
    to->lfirst[i] = first;
}

// The stream's share of the device, and how many blocks of a launch on it, of which `per_cu` fit a CU, may wait for
// others (stream_limit).
StreamShare stream_share(hipStream_t st);
bool is_capturing(hipStream_t st);
uint64_t waiting_limit(const StreamShare& share, uint64_t per_cu);
// ... of a resident launch.
uint64_t resident_limit_on(const StreamShare& share);
// The single-pass path's one launch (topk_whole.hip), for calls that whole_tiles admits.
uint64_t whole_limit_on(const StreamShare& share);
void launch_whole(const Buckets& bk, const Geometry& g, const Workspace& w, uint32_t group_tiles, uint32_t groups_shift, uint32_t epoch,
                  uint32_t published, uint64_t limit_ticks, hipStream_t st);
// A list of buckets goes in as many launches as keep each under `limit`.
void launch_resident(const Buckets& bk, const Geometry& g, const Workspace& w, int vecs, uint64_t limit, uint32_t epoch,
                     uint32_t published, uint64_t limit_ticks, hipStream_t st);

// ---- what blocks of one launch use to talk to each other ----------------------------------
__device__ __forceinline__ uint32_t ld_agent(const uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent(uint32_t* p, uint32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Histogram add called by all lanes of a wavefront (m: this lane has a key).  When all
// keys of the wavefront fall into one bin - zeros, constants: the inputs that reach the
// dense-region and exact paths - one lane adds the count; 64 adds to one LDS address
// would serialise.
__device__ __forceinline__ void wave_hist_add(uint32_t* lh, bool m, uint32_t bin) {
    const uint64_t act = __ballot(m);
    if (!act) return;
    const int first = __ffsll((long long)act) - 1;
    const uint32_t fb = (uint32_t)__shfl((int)bin, first, kWave);
    if (__ballot(m && bin == fb) == act) {
        if ((int)(threadIdx.x & (kWave - 1)) == first) atomicAdd(&lh[fb], (uint32_t)__popcll(act));
    } else if (m) {
        atomicAdd(&lh[bin], 1u);
    }
}

// All threads of the block call it.  Returns false when the wait timed out.
// Everything blocks hand to each other goes through agent-scope stores, atomics
// and loads (they bypass the per-XCD L2 copies), so the barrier needs no cache
// write-back or invalidate: each wavefront only waits until its own stores and
// atomics have been acknowledged before the block's arrival is counted.  (Whole-
// cache fences here, repeated by a thousand polling blocks, made the kernel ten
// times slower.)
__device__ __forceinline__ bool bucket_barrier(uint32_t* counter, uint32_t parties, uint32_t* flag /* LDS */,
                                               uint64_t limit_ticks) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        uint64_t t0 = 0;
        uint32_t ok = 1, polls = 0;
        while (ld_agent(counter) < parties) {
            __builtin_amdgcn_s_sleep(8);
            if ((++polls & 63u) == 0) {  // look at the clock now and then
                const uint64_t now = (uint64_t)wall_clock64();
                if (t0 == 0) t0 = now;
                else if (now - t0 > limit_ticks) {
                    ok = 0;
                    break;
                }
            }
        }
        *flag = ok;
    }
    __syncthreads();
    return *flag != 0;
}


__device__ __forceinline__ uint64_t ld_agent64(const uint64_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent64(uint64_t* p, uint64_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// 16-byte streaming store written through to memory (agent scope): a later 4-byte
// repair of the same line by a block on another XCD must not be overwritten by a
// delayed write-back of this one.  (The wait states: see store16_agent.)
// `base` is the same in every lane, `at` the lane's element behind it.
__device__ __forceinline__ void store_through(float* base, uint32_t at, u4a v) {
    asm volatile("global_store_dwordx4 %0, %1, %2 sc1 nt\n\ts_nop 2" ::"v"(at * 4), "v"(v), "s"(base) : "memory");
}

// A bucket's window is one store16_agent and one load16_agent: the four words change together.
// (waits for every earlier load of the wavefront as well: they complete in order)
__device__ __forceinline__ u4a load16_agent(const uint32_t* p) {
    u4a v;
    asm volatile("global_load_dwordx4 %0, %1, off sc1\n\ts_waitcnt vmcnt(0)" : "=&v"(v) : "v"(p) : "memory");
    return v;
}
// Waits until the bucket's window is published (S_READY == epoch); called by a whole wavefront
// or a single thread.  win[3] = 0 when the wait timed out.
template <int SLEEP = 16>
__device__ __forceinline__ u4a wait_window(const uint32_t* st, uint32_t epoch, uint64_t limit_ticks) {
    uint64_t t0 = 0;
    uint32_t polls = 0;
    for (;;) {
        u4a v = load16_agent(st + S_LO_KEY);
        if ((uint32_t)__builtin_amdgcn_readfirstlane((int)v[3]) == epoch) {
            v[3] = 1u;
            return v;
        }
        __builtin_amdgcn_s_sleep(SLEEP);
        if ((++polls & 63u) == 0) {
            const uint64_t now = (uint64_t)wall_clock64();
            if (t0 == 0) t0 = now;
            else if (now - t0 > limit_ticks) {
                v[3] = 0u;
                return v;
            }
        }
    }
}

// ---- sample ------------------------------------------------------------------------
// The first round's histogram is kept in copies, by lane, a few banks apart: gradients share few
// exponents, and lanes that add to one LDS word take turns (8192 keys: 1.6 to 2.4 us with one copy).
template <int THREADS>
struct SampleLds {
    static constexpr int kCopies = THREADS >= 1024 ? 4 : THREADS >= 512 ? 2 : 1;
    static constexpr int kPad = THREADS >= 1024 ? 0 : 32;  // behind the bins: where zeros add, lanes apart
    static constexpr int kCopy = kBins0 + kPad + 8;  // words
    uint32_t h0[kCopies * kCopy] __attribute__((aligned(16)));
    uint32_t h1[kBins0] __attribute__((aligned(16)));
    uint32_t wsum[THREADS / kWave];
    uint32_t res[3][2];
};

// For NR ranks at once: the bin in which a top-down scan of the histogram reaches rank[z],
// and how many of the rank's elements fall inside that bin.  Thread t owns the PER bins below
// BINS - PER t (vector LDS reads).  res[z] = {bin, left}; bin = BINS when the histogram holds
// fewer than rank[z] elements or rank[z] == 0.  Called by all threads of the block.  COPIES: the
// histogram is the sum of that many, STRIDE words apart.
template <int BINS, int NR, int THREADS, int COPIES = 1, int STRIDE = 0>
__device__ __forceinline__ void sample_pick(const uint32_t* h, const uint32_t (&rank)[NR], uint32_t* wsum, uint32_t (*res)[2],
                                            uint32_t tid = threadIdx.x) {
    constexpr int PER = BINS / THREADS;
    constexpr int RW = PER % 4 == 0 ? 4 : PER;  // bins per LDS read
    static_assert(PER % RW == 0, "whole vectors");
    typedef uint32_t Row __attribute__((ext_vector_type(RW)));
    const int lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane((int)(tid / kWave));
    uint32_t c[PER], sum = 0;  // c[j]: bin BINS - 1 - PER t - j
    const Row* row = (const Row*)&h[BINS - PER * (tid + 1)];
#pragma unroll
    for (int v = 0; v < PER / RW; v++) {
        Row x = row[PER / RW - 1 - v];
#pragma unroll
        for (int d = 1; d < COPIES; d++) x += row[PER / RW - 1 - v + d * (STRIDE / RW)];
#pragma unroll
        for (int q = 0; q < RW; q++) {
            c[v * RW + q] = x[RW - 1 - q];
            sum += x[RW - 1 - q];
        }
    }
    const uint32_t inc = wave_inclusive_scan(sum);
    if (lane == kWave - 1) wsum[wave] = inc;
    if (tid < NR) { res[tid][0] = BINS; res[tid][1] = 0; }
    __syncthreads();
    const uint32_t s = lane < THREADS / kWave ? wsum[lane] : 0u;
    uint32_t above = inc - sum + (uint32_t)__builtin_amdgcn_readlane((int)(wave_inclusive_scan(s) - s), wave);
#pragma unroll
    for (int j = 0; j < PER; j++) {
#pragma unroll
        for (int z = 0; z < NR; z++) {
            if (above < rank[z] && rank[z] <= above + c[j]) {
                res[z][0] = (uint32_t)(BINS - 1 - PER * (int)tid - j);
                res[z][1] = rank[z] - above;
            }
        }
        above += c[j];
    }
    __syncthreads();
}

// Candidate window of a bucket from 8192 evenly spread elements of grad + residual, whose keys stay
// in registers: select of three ranks - upper and lower end of the window, 6 sigma of the sampling
// noise away from the expected rank of the k-th largest key, and the predicted threshold - by 11 key
// bits and then, in one histogram for all three, by 2048 bins over the digits that they lie in.  Zeros are not counted:
// sparse gradients' would all add to one LDS word (at 99 % zeros the window was published two microseconds later, and a call
// of 6,553,600 elements at 0.1 % took 31.7 us, so 29.1), and a rank among them would stretch the digits down to zero's.
// Called by all THREADS threads of a block; the result is valid in thread 0.
// `under_way()` runs while the sample's loads are under way.
struct SampleWindow {
    uint32_t lo, hi, that;
};
template <int THREADS, class UnderWay>
__device__ __forceinline__ SampleWindow sample_window(const float* gp, const float* rp, uint64_t bn, uint32_t k,
                                                      SampleLds<THREADS>& L, UnderWay&& under_way) {
    const uint64_t nvec = bn / 4;
    constexpr int SV = kFSample / 4;     // sampled vectors
    constexpr int PV = SV / THREADS;     // vectors per thread; their 4 * PV keys stay in registers
    // sampled in runs of 8 vectors (one 128-byte line per array), runs evenly spread
    const uint32_t nsv = nvec < (uint64_t)SV ? (uint32_t)(nvec & ~7ull) : (uint32_t)SV;
    const uint64_t stride = nsv ? (nvec / (nsv / 8)) : 8;  // vectors between run starts (>= 8)
    u4a gv[PV], rv[PV];
#pragma unroll
    for (int j = 0; j < PV; j++) {
        const uint32_t i = (uint32_t)j * THREADS + threadIdx.x;
        const uint32_t ii = i < nsv ? i : 0;
        const uint64_t v = (uint64_t)(ii >> 3) * stride + (ii & 7);
        gv[j] = nsv ? *(const u4u4*)(gp + v * 4) : u4a{0u, 0u, 0u, 0u};
        rv[j] = nsv ? *(const u4u4*)(rp + v * 4) : u4a{0u, 0u, 0u, 0u};
    }
    under_way();
    constexpr int COPIES = SampleLds<THREADS>::kCopies, COPY = SampleLds<THREADS>::kCopy;
    {
        const u4a z = {0u, 0u, 0u, 0u};
        static_assert(offsetof(SampleLds<THREADS>, h1) == sizeof(L.h0), "cleared as one");
        for (int i = threadIdx.x; i < (COPIES * COPY + kBins0) / 4; i += THREADS) ((u4a*)L.h0)[i] = z;
    }
    uint32_t* const h0 = L.h0 + (threadIdx.x % COPIES) * COPY;
    uint32_t key[PV][4];
#pragma unroll
    for (int j = 0; j < PV; j++) {
        // an element past the sample gets the key 0, which no histogram counts
        const bool have = (uint32_t)j * THREADS + threadIdx.x < nsv;
#pragma unroll
        for (int q = 0; q < 4; q++) key[j][q] = have ? key_of(u2f(gv[j][q]) + u2f(rv[j][q])) : 0u;
    }
    const uint32_t S = nsv * 4;
    const float ks = (float)k * (float)S / (float)bn;
    const float margin = 6.0f * sqrtf(ks) + 16.0f;
    // ranks: 0 upper end of the window, 1 lower end, 2 the predicted threshold itself
    constexpr int NR = 3;
    uint32_t rank[NR];
    // A k-th largest key expected among the sample's first few (small ratios) leaves no margin
    // above it: the sample's largest key is the upper end then, and a threshold above it (probability
    // e^-ks) fails the window.  Without an upper end the bins would span every float above lo.
    rank[0] = ks - margin >= 1.0f ? (uint32_t)(ks - margin) : (ks >= 3.0f ? 1u : 0u);  // 0: no upper end
    rank[1] = (uint32_t)(ks + margin) + 1u;                       // > S: no lower end
    rank[2] = ks >= 1.0f ? (uint32_t)ks : 1u;
    const bool active[NR] = {rank[0] >= 1u && rank[0] <= S, rank[1] <= S, rank[2] <= S};
    __syncthreads();
    // round 0: key[30:20]
#pragma unroll
    for (int j = 0; j < PV; j++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            // (32 or 16 branches in a row cost a call of 96.5 M elements 1 us, eight cost nothing and save the padding's adds 0.15)
            constexpr uint32_t kPad = SampleLds<THREADS>::kPad;
            if constexpr (kPad > 0) atomicAdd(&h0[key[j][q] ? key[j][q] >> 20 : kBins0 + threadIdx.x % kPad], 1u);
            else if (key[j][q]) atomicAdd(&h0[key[j][q] >> 20], 1u);
        }
    __syncthreads();
    {
        const uint32_t want[NR] = {active[0] ? rank[0] : 0u, active[1] ? rank[1] : 0u, active[2] ? rank[2] : 0u};
        sample_pick<kBins0, NR, THREADS, COPIES, COPY>(L.h0, want, L.wsum, L.res);
    }
    // round 1: the digits that the ranks lie in and those between, few of the keys, in one histogram.  (Compared with each
    // rank's digit and counted in a histogram of its own, the keys take 40 instructions each instead of six: 1.6 us of a
    // block of 512 threads, 1.9 with the three scans.)
    uint32_t first = kBins0, last = 0, above = 0;  // of those digits; the keys above them
    bool found[NR];                                // else among the zeros
#pragma unroll
    for (int z = 0; z < NR; z++) {
        const uint32_t d = L.res[z][0];
        found[z] = active[z] && d < (uint32_t)kBins0;
        if (found[z] && d < first) first = d;
        if (found[z] && d >= last) {
            last = d;
            above = rank[z] - L.res[z][1];
        }
    }
    if (first > last) first = last;
    const uint32_t base = first << 20, span = (last - first + 1) << 20;
    const int open = 32 - __clz((int)(span - 1)), sh = open > 11 ? open - 11 : 0;
#pragma unroll
    for (int j = 0; j < PV; j++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t d = key[j][q] - base;
            if (d < span) atomicAdd(&L.h1[d >> sh], 1u);
        }
    // (what under_way stored has long arrived; every wavefront makes sure of its part before thread 0 publishes)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    {
        const uint32_t want[NR] = {found[0] ? rank[0] - above : 0u, found[1] ? rank[1] - above : 0u, found[2] ? rank[2] - above : 0u};
        sample_pick<kBins0, NR, THREADS>(L.h1, want, L.wsum, L.res);
    }
    SampleWindow win = {0u, 0x7FFFFFFFu, 0x7FFFFFFFu};
    if (threadIdx.x == 0) {
        const auto cell = [&](int z) { return base + (L.res[z][0] << sh); };
        const uint32_t width = 1u << sh;
        win.lo = found[1] ? cell(1) : 0u;
        win.hi = found[0] ? cell(0) + (width - 1) : active[0] ? 0x3FFu : 0x7FFFFFFFu;  // upper end of the window: rounded up
        if (win.hi < win.lo) win.hi = win.lo;
        // predicted threshold: middle of its cell; never below lo: every pre-zeroed
        // element must be a listed candidate
        win.that = found[2] ? cell(2) + width / 2 : active[2] ? 0x200u : 0x7FFFFFFFu;
        if (win.that < win.lo) win.that = win.lo;
    }
    return win;
}

__device__ __forceinline__ void fused_give_up(const Workspace& w, uint32_t* st, uint32_t* out) {
    if (threadIdx.x == 0) {
        st_agent(st + S_TIMEOUT, 1u);
        if (w.status) st_agent((uint32_t*)w.status, (uint32_t)MCCL_HIP_ERR_TIMEOUT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        st_agent(out, kPoisonK);
    }
}

}  // namespace mcclhip
