// Decompress and rank-ordered sparse accumulate of top-k payloads for gfx950.
//
// Payload layout (csrc/compression/TopKCompression.cpp:93-113):
//   [u32 k][k x {u32 index, f32 value}], little endian, indices ascending.
//
// decompress: dense = 0, dense[index] = value (TopKCompression.cpp:122-152).
//
// sparse accumulate: the reference decompresses every peer's payload into a
// dense buffer and folds the dense buffers in ascending rank order
// (csrc/backend/ProcessGroupMCCL.cpp:1692-1709,:2272-2296).  Here the output is
// cut into tiles that live in LDS, start at +0.0, receive rank 0's, rank 1's, ...
// pairs that fall inside them, and are written once, scaled.  Two kernel
// families do that:
//   runs of tiles (up to 8 ranks, payloads of the usual density, a workspace):
//     one wavefront per run of 2048-element tiles, every rank's pairs held in
//     registers, rank order kept by the LDS's in-order execution of one
//     wavefront's adds; a small table says near which pair (to the nearest 80) of each
//     payload a run begins.
//   tile kernels (everything else): one block per 8192-element tile with a
//     barrier between ranks, ranges from a bounds table or by binary search.
// HBM traffic is close to the algorithmic minimum: every payload read once (plus
// one index in 80 for the table), every output element written once.
#include "common.hip.h"
#include "runtime.h"

namespace mcclhip {

namespace {

constexpr int kAccThreads = 512;  // threads per block of the accumulate kernel with bounds
constexpr int kAccTile = 8192;  // output elements per block, accumulated in LDS (32 KiB)

__global__ __launch_bounds__(kBlock) void k_fill_zero(float* p, uint64_t n) {
    // 16-byte stores over the aligned body, scalars at both ends
    uint64_t head = ((16 - ((uintptr_t)p & 15)) & 15) / 4;
    if (head > n) head = n;
    const uint64_t nvec = (n - head) / 4;
    u4a* v = (u4a*)(p + head);
    const u4a z = {0u, 0u, 0u, 0u};
    for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < nvec; i += (uint64_t)gridDim.x * kBlock)
        v[i] = z;
    const uint64_t g = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (g < head) p[g] = 0.0f;
    const uint64_t tail = head + nvec * 4;
    if (g < 4 && tail + g < n) p[tail + g] = 0.0f;
}

__global__ __launch_bounds__(kBlock) void k_scatter(const uint32_t* wire, uint32_t expected_k, float* dense,
                                                    uint64_t count, int* status) {
    const uint32_t k = wire[0];
    if (k != expected_k) {
        if (status && blockIdx.x == 0 && threadIdx.x == 0) *status = MCCL_HIP_ERR_SIZE;
        return;
    }
    for (uint64_t p = (uint64_t)blockIdx.x * kBlock + threadIdx.x; p < k; p += (uint64_t)gridDim.x * kBlock) {
        const uint32_t idx = wire[1 + 2 * p];
        const uint32_t val = wire[2 + 2 * p];
        if (idx < count) dense[idx] = u2f(val);
        else if (status) *status = MCCL_HIP_ERR_INDEX;
    }
}

// ---- decompress of an ascending payload in one launch ---------------------------------
// A block owns a tile of the dense buffer: zeroed in LDS, given the pairs that fall inside it,
// written once.  It finds its pairs without a search: every block reads the same kSamples evenly
// spaced indices, counts those below its first element (s) and below its end (u), and takes the
// strides from sample s - 1 up to sample u - its own pairs and a few neighbours'.  Two dependent
// round trips (samples, pairs) and the stores; fill and scatter are two launches and write the
// picked lines twice.  6,553,600 elements, 65,536 pairs: 6.1 us in the kernel against 5.9 + 3.2 and
// the launch between them.
// The tile goes past the XCD's L2 to the memory-side cache: left in the L2 (all of 26 MB fits there) it would be
// written back after the last block, while the call waits.  That bucket through compress and decompress, 1 %: plain
// stores 56.8 us, nt 55.7, so 55.0.
// Whether the payload ascends is checked on the way, by all blocks together: samples ascend, and
// every block checks the adjacent pairs of its strides and the one that links them to the next
// stride; the last strides of a block are the first of the next one (u of a tile is s of the next),
// so every adjacent pair is looked at by somebody.
constexpr int kDecTile = 8192;
constexpr int kDecSamples = kBlock;      // one per thread
constexpr uint32_t kDecMaxStride = 4096;  // beyond (over a million pairs) fill and scatter are as fast

// DONE: the launch tells the host when its stores have arrived, in one word of pinned host memory; the end of the
// launch itself reaches a host that waits for the stream 5.4 us after such a word does (a launch of one block: 11.6
// against 6.1 us).  Compress and decompress at 1 %, us, waiting for the stream / the word, until the call returns and with a fold
// of the result behind it: 2000 elements 22.5 / 18.1 and 25.6 / 22.0, 65,537 29.7 / 25.3 and 33.0 / 28.5, 6,553,600
// 53.5 / 50.9 and 67.6 / 64.4.  A block arrives when its stores - written past the L2 - have been acknowledged; the block
// that arrives last has seen the others arrive, and nobody waits.  Arrivals at one word take turns, some 25 ns
// each, so that larger grids arrive at 32 words and those at one.
constexpr uint32_t kDoneLines = 32;
constexpr uint32_t kDoneOne = 64;  // grids of at most this many blocks arrive at the one word
static_assert(MCCL_HIP_DONE_BYTES >= (1 + kDoneLines) * 256, "a word every 256 bytes");
struct Done {
    uint64_t* counters;  // [1 + kDoneLines], 256 bytes apart, zero between calls: blocks, blocks with errors << 32
    uint64_t* word;      // host: ticket << 32 | result
    uint32_t ticket;
};
__device__ __forceinline__ bool last_to_arrive(uint64_t* counter, uint32_t parties, uint64_t* sum) {
    *sum += __hip_atomic_fetch_add(counter, *sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if ((uint32_t)*sum != parties) return false;
    __hip_atomic_store(counter, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    return true;
}
// One thread of the block calls it, when all stores of the block have been acknowledged.
__device__ __forceinline__ void arrive_done(const Done& d, bool bad, int brought) {
    uint64_t sum = 1ull | (uint64_t)(bad ? 1 : 0) << 32;
    if (gridDim.x > kDoneOne) {
        const uint32_t line = blockIdx.x % kDoneLines;
        if (!last_to_arrive(d.counters + 32 * (1 + line), (gridDim.x - line + kDoneLines - 1) / kDoneLines, &sum)) return;
        sum = 1ull | (uint64_t)(sum >> 32 ? 1 : 0) << 32;
    }
    if (!last_to_arrive(d.counters, gridDim.x > kDoneOne ? kDoneLines : gridDim.x, &sum)) return;
    const uint32_t result = (uint32_t)(sum >> 32 ? MCCL_HIP_ERR_ORDER : brought);
    __hip_atomic_store(d.word, (uint64_t)d.ticket << 32 | result, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <bool DONE>
__global__ __launch_bounds__(kBlock) void k_decompress_sorted(const uint32_t* wire, uint32_t k, uint32_t stride, float* dense,
                                                              uint64_t count, int* status, const int* flag, int* flag_out,
                                                              Done done) {
    __shared__ __attribute__((aligned(16))) float tile[kDecTile];
    __shared__ uint32_t samp[kDecSamples + 1];
    __shared__ uint32_t below[2], any_bad;
    const uint64_t t0 = (uint64_t)blockIdx.x * kDecTile;
    const uint64_t t1 = t0 + kDecTile < count ? t0 + kDecTile : count;
    const uint32_t* const pairs = wire + 1;
    const uint64_t mypos = (uint64_t)threadIdx.x * stride;
    const uint32_t have_k = wire[0];
    const uint32_t mine = mypos < k ? pairs[2 * mypos] : 0xFFFFFFFFu;
    const bool brings = flag && (DONE || blockIdx.x == 0) && threadIdx.x == 0;
    const int brought = brings ? *flag : 0;
#pragma unroll
    for (int i = 0; i < kDecTile / (4 * kBlock); i++) ((u4a*)tile)[i * kBlock + threadIdx.x] = u4a{0u, 0u, 0u, 0u};
    if (threadIdx.x < 2) below[threadIdx.x] = 0;
    if (threadIdx.x == 0) any_bad = 0;
    if (threadIdx.x == 0) samp[kDecSamples] = 0xFFFFFFFFu;
    samp[threadIdx.x] = mine;
    if (have_k != k) {  // the same in every lane of the grid
        if constexpr (DONE) {
            if (threadIdx.x == 0) arrive_done(done, true, brought);
        } else {
            if (blockIdx.x == 0 && threadIdx.x == 0) *status = MCCL_HIP_ERR_SIZE;
            if (brings) *flag_out = brought;
        }
        return;
    }
    if constexpr (!DONE)
        if (brings) *flag_out = brought;  // (its load went with the samples)
    __syncthreads();
    int bad = 0;
    if (mypos + stride < k && mine >= samp[threadIdx.x + 1]) bad = MCCL_HIP_ERR_ORDER;
    // (a position past the payload reads 0xFFFFFFFF and counts as beyond every element)
    const uint64_t ms = __ballot(mypos < k && mine < t0), mu = __ballot(mypos < k && mine < t1);
    if ((threadIdx.x & (kWave - 1)) == 0) {
        if (ms) atomicAdd(&below[0], (uint32_t)__popcll(ms));
        if (mu) atomicAdd(&below[1], (uint32_t)__popcll(mu));
    }
    __syncthreads();
    const uint64_t s = below[0], u = t1 == count ? kDecSamples : below[1];  // the last tile takes what is left
    const uint64_t p0 = (s ? s - 1 : 0) * stride;
    uint64_t p1 = u * stride;
    if (p1 > k) p1 = k;
    for (uint64_t p = p0 + threadIdx.x; p < p1; p += kBlock) {
        const u2a pr = *(const u2a4*)(pairs + 2 * p);
        const uint32_t next = p + 1 < k ? pairs[2 * (p + 1)] : 0xFFFFFFFFu;
        if (p + 1 < k && pr[0] >= next) bad = MCCL_HIP_ERR_ORDER;
        if (pr[0] >= count) bad = bad ? bad : MCCL_HIP_ERR_INDEX;
        const uint64_t off = (uint64_t)pr[0] - t0;
        if (off < t1 - t0) tile[off] = u2f(pr[1]);
    }
    if (bad) {
        if constexpr (DONE) any_bad = 1;
        else *status = bad;
    }
    __syncthreads();
    float* const out = dense + t0;
    const uint32_t len = (uint32_t)(t1 - t0);
    if (len == (uint32_t)kDecTile) {
#pragma unroll
        for (int i = 0; i < kDecTile / (4 * kBlock); i++)
            store16_agent(out + 4 * (i * kBlock + threadIdx.x), ((const u4a*)tile)[i * kBlock + threadIdx.x]);
    } else {
        for (uint32_t i = threadIdx.x; i < len; i += kBlock) store4_agent(out + i, tile[i]);
    }
    if constexpr (DONE) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x == 0) arrive_done(done, any_bad != 0, brought);
    }
}

__global__ void k_copy_word(const int* from, int* to) { *to = *from; }

struct WirePtrs {
    const uint8_t* w[MCCL_HIP_MAX_WORLD];
};

// Scratch of mccl_hip_sparse_accumulate_static: the position table lives in
// this file-scope device array instead of a caller workspace, so the call
// allocates nothing.  Every GPU holds its own copy at its own address; host
// code only ever uses the address hipGetSymbolAddress returned for the device
// (g_static_ptr), never the array's name.
constexpr uint64_t kStaticWords = MCCL_HIP_SPARSE_STATIC_BYTES / 4;
static __device__ __align__(256) uint32_t scratch[kStaticWords];
constexpr int kMaxDevices = 64;
uint32_t* g_static_ptr[kMaxDevices];

// First pair position in [0, k) whose index is >= target (k if none).
__device__ __forceinline__ uint32_t lower_bound_idx(const uint32_t* pairs, uint32_t k, uint32_t target) {
    uint32_t lo = 0, hi = k;
    while (lo < hi) {
        const uint32_t mid = lo + ((hi - lo) >> 1);
        if (pairs[2 * (uint64_t)mid] < target) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

__global__ __launch_bounds__(kBlock) void k_sparse_accumulate(float* acc, uint64_t n_total,
                                                              uint64_t bucket_elems, WirePtrs wires, int ws,
                                                              uint64_t wire_stride, int apply_scale,
                                                              float scale, int* status) {
    __shared__ float tile[kAccTile];
    __shared__ uint32_t lo_s[MCCL_HIP_MAX_WORLD], hi_s[MCCL_HIP_MAX_WORLD];
    const uint32_t b = blockIdx.y, t = blockIdx.x;
    const uint64_t bstart = (uint64_t)b * bucket_elems;
    const uint64_t bn = (n_total - bstart) < bucket_elems ? (n_total - bstart) : bucket_elems;
    const uint64_t tstart = (uint64_t)t * kAccTile;
    if (tstart >= bn) return;
    const uint32_t tlen = (uint32_t)((bn - tstart) < kAccTile ? (bn - tstart) : kAccTile);
    const uint32_t kmax = (uint32_t)((wire_stride - 4) / 8);

    for (int i = threadIdx.x; i < kAccTile; i += kBlock) tile[i] = 0.0f;
    // range of every rank's pairs inside this tile: thread r -> lower end, thread ws + r -> upper end
    if (threadIdx.x < 2 * ws) {
        const int r = threadIdx.x < ws ? threadIdx.x : threadIdx.x - ws;
        const uint32_t* wp = (const uint32_t*)(wires.w[r] + (uint64_t)b * wire_stride);
        uint32_t k = wp[0];
        if (k > kmax) {
            if (status) *status = MCCL_HIP_ERR_SIZE;
            k = 0;
        }
        if (threadIdx.x < ws) {
            lo_s[r] = lower_bound_idx(wp + 1, k, (uint32_t)tstart);
        } else {
            hi_s[r] = lower_bound_idx(wp + 1, k, (uint32_t)(tstart + tlen));
            // the block that owns the bucket's last tile also checks the largest index
            if (tstart + tlen == bn && k > 0 && wp[1 + 2 * (uint64_t)(k - 1)] >= bn && status)
                *status = MCCL_HIP_ERR_INDEX;
        }
    }
    __syncthreads();
    for (int r = 0; r < ws; r++) {
        const uint32_t* pairs = (const uint32_t*)(wires.w[r] + (uint64_t)b * wire_stride) + 1;
        const uint32_t lo = lo_s[r], hi = hi_s[r];
        for (uint32_t p = lo + threadIdx.x; p < hi; p += kBlock) {
            const uint32_t off = pairs[2 * (uint64_t)p] - (uint32_t)tstart;
            const float v = u2f(pairs[2 * (uint64_t)p + 1]);
            if (off < tlen) tile[off] = tile[off] + v;
            else if (status) *status = MCCL_HIP_ERR_INDEX;  // unsorted payload
        }
        __syncthreads();
    }
    float* out = acc + bstart + tstart;
    if (tlen == kAccTile && (((uintptr_t)out & 15) == 0)) {
        for (int i = threadIdx.x; i < kAccTile / 4; i += kBlock) {
            u4a v;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float x = tile[4 * i + q];
                v[q] = f2u(apply_scale ? x * scale : x);
            }
            ((u4a*)out)[i] = v;
        }
    } else {
        for (uint32_t i = threadIdx.x; i < tlen; i += kBlock) {
            const float x = tile[i];
            out[i] = apply_scale ? x * scale : x;
        }
    }
}

// ---- tile bounds pre-pass ------------------------------------------------------
// start[(b * ws + r) * (tiles + 1) + t] = first pair of rank r's bucket-b payload
// whose index lies in tile t or later; entry t = tiles holds k.  A rank's entries
// are contiguous: interleaving the ranks put the entries that eight different
// blocks write into one 32-byte sector and made this kernel 40 % slower.  One
// thread per pair: pair p writes the
// entry of every tile that begins between pair p-1 and pair p (usually none), so
// each entry is written exactly once for a sorted payload; the entries of a gap of
// more than four tiles are shared by the wavefront, once a thread of it has found one (asked for behind every pair, nine
// ranks of 4 M elements at 1 % took 11.9 us instead of 11.7): one thread that wrote them took 25 ns for each, after all others.  us per call, one thread / so: two ranks of 6 M elements at 1 % whose pairs lie at the
// bucket's front 33.8 / 13.5, eight of 8 M in two buckets, the last a fifth as long, 32.7 / 14.3 (where entries past the
// last bucket's own tiles were written as well).  A thread takes eight consecutive pairs.  The pair loads do not wait for k: they stay inside the
// payload's stride and are masked afterwards.
__global__ __launch_bounds__(kBlock) void k_sparse_bounds(WirePtrs wires, int ws, uint64_t wire_stride,
                                                          uint64_t n_total, uint64_t bucket_elems, uint32_t tiles,
                                                          uint32_t* start, int* status) {
    const uint32_t b = blockIdx.y / (uint32_t)ws, r = blockIdx.y % (uint32_t)ws;
    const uint64_t bstart = (uint64_t)b * bucket_elems;
    const uint64_t bn = (n_total - bstart) < bucket_elems ? (n_total - bstart) : bucket_elems;
    const uint32_t* wp = (const uint32_t*)(wires.w[r] + (uint64_t)b * wire_stride);
    const uint32_t kmax = (uint32_t)((wire_stride - 4) / 8);
    constexpr int PP = 8;  // consecutive pairs per thread: four 16-byte loads, issued before the first use
    const uint32_t p0 = (blockIdx.x * kBlock + threadIdx.x) * PP;
    const u4u4* pv = (const u4u4*)(wp + 1);  // two (index, value) pairs per vector
    u4a v[PP / 2];
    uint32_t before = 0;  // index of pair p0 - 1
    if (p0 + PP <= kmax) {
#pragma unroll
        for (int j = 0; j < PP / 2; j++) v[j] = pv[p0 / 2 + j];
        if (p0 > 0) before = wp[1 + 2 * (uint64_t)(p0 - 1)];
    } else {
#pragma unroll
        for (int j = 0; j < PP / 2; j++) {
            v[j][0] = p0 + 2 * j < kmax ? wp[1 + 2 * (uint64_t)(p0 + 2 * j)] : 0u;
            v[j][2] = p0 + 2 * j + 1 < kmax ? wp[1 + 2 * (uint64_t)(p0 + 2 * j + 1)] : 0u;
        }
        if (p0 > 0 && p0 - 1 < kmax) before = wp[1 + 2 * (uint64_t)(p0 - 1)];
    }
    uint32_t k = wp[0];
    if (k > kmax) {
        if (status) *status = MCCL_HIP_ERR_SIZE;
        k = 0;
    }
    uint32_t* st = start + ((uint64_t)b * ws + r) * (tiles + 1);  // entry of tile t at st[t]
    if (k == 0) {
        for (uint32_t t = blockIdx.x * kBlock + threadIdx.x; t <= tiles; t += gridDim.x * kBlock) st[t] = 0;
        return;
    }
    // entries past the bucket's own tiles are read by nobody
    const uint32_t own_tiles = (uint32_t)((bn + kAccTile - 1) / kAccTile);
    const int lane = threadIdx.x & (kWave - 1);
    // The n entries from `from` on are `value`: those of pair p0 + j or, j = PP, the ones behind the bucket's last pair, if
    // the thread has that.
    struct Gap { uint32_t from, n, value; };
    auto index = [&](int j) { return v[j / 2][(j & 1) * 2]; };
    auto gap = [&](int j) {
        const bool behind = j == PP;
        const uint32_t p = behind ? k - 1 : p0 + (uint32_t)j;
        if (behind ? k - 1 - p0 >= (uint32_t)PP : p >= k) return Gap{0u, 0u, 0u};
        uint32_t at = behind ? 0u : index(j < PP ? j : 0);
        if (behind) {
#pragma unroll
            for (int i = 0; i < PP; i++)
                if (p0 + (uint32_t)i == p) at = index(i);
        }
        uint32_t to = at / kAccTile;  // the tile in which the pair lies
        if (to > own_tiles) to = own_tiles;
        if (behind) return Gap{to + 1, own_tiles - to, k};
        const uint32_t from = p == 0 ? 0u : (j ? index(j ? j - 1 : 0) : before) / kAccTile + 1;
        return Gap{from, from <= to ? to - from + 1 : 0u, p};
    };
    // a long gap - between clustered pairs, in front of the first, behind the last - is written by the whole wavefront
    constexpr uint32_t kAlone = 4;
    bool far = false;
#pragma unroll
    for (int j = 0; j <= PP; j++) {
        const Gap g = gap(j);
        if (g.n > kAlone) far = true;
        else
            for (uint32_t t = 0; t < g.n; t++) st[g.from + t] = g.value;
        if (j < PP && p0 + (uint32_t)j < k && status) {
            if (index(j) >= bn) *status = MCCL_HIP_ERR_INDEX;
            if (p0 + (uint32_t)j > 0 && (j ? index(j - 1) : before) >= index(j)) *status = MCCL_HIP_ERR_INDEX;  // not ascending
        }
    }
    if (!__ballot(far)) return;
#pragma unroll
    for (int j = 0; j <= PP; j++) {
        const Gap g = gap(j);
        for (uint64_t of = __ballot(g.n > kAlone); of; of &= of - 1) {
            const int l = __ffsll((long long)of) - 1;
            const uint32_t f = (uint32_t)__builtin_amdgcn_readlane((int)g.from, l), c = (uint32_t)__builtin_amdgcn_readlane((int)g.n, l);
            const uint32_t value = (uint32_t)__builtin_amdgcn_readlane((int)g.value, l);
            for (uint32_t i = (uint32_t)lane; i < c; i += kWave) st[f + i] = value;
        }
    }
}

// Accumulate with precomputed bounds: every block reads its 2 * ws bounds with one
// load per lane, then issues the loads of all its pairs (every rank) before the
// first LDS add; the adds run rank by rank.
__global__ __launch_bounds__(kAccThreads) void k_sparse_accumulate_b(float* acc, uint64_t n_total,
                                                                uint64_t bucket_elems, WirePtrs wires, int ws,
                                                                uint64_t wire_stride, uint32_t tiles,
                                                                const uint32_t* start, int apply_scale,
                                                                float scale, int* status) {
    __shared__ float tile[kAccTile];
    __shared__ uint32_t lo_s[MCCL_HIP_MAX_WORLD], hi_s[MCCL_HIP_MAX_WORLD];
    const uint32_t b = blockIdx.y, t = blockIdx.x;
    const uint64_t bstart = (uint64_t)b * bucket_elems;
    const uint64_t bn = (n_total - bstart) < bucket_elems ? (n_total - bstart) : bucket_elems;
    const uint64_t tstart = (uint64_t)t * kAccTile;
    if (tstart >= bn) return;
    const uint32_t tlen = (uint32_t)((bn - tstart) < kAccTile ? (bn - tstart) : kAccTile);
    const uint32_t kmax = (uint32_t)((wire_stride - 4) / 8);
    if (threadIdx.x < 2 * ws) {
        const int r = threadIdx.x < ws ? threadIdx.x : threadIdx.x - ws;
        uint32_t v = start[((uint64_t)b * ws + r) * (tiles + 1) + t + (threadIdx.x < ws ? 0 : 1)];
        if (v > kmax) v = kmax;  // stale bound of a malformed payload: stay inside the buffer
        if (threadIdx.x < ws) lo_s[r] = v; else hi_s[r] = v;
    }
    for (int i = threadIdx.x; i < kAccTile; i += kAccThreads) tile[i] = 0.0f;
    __syncthreads();
    constexpr int RB = 8;  // ranks whose pairs are in flight together
    for (int r0 = 0; r0 < ws; r0 += RB) {
        uint32_t off[RB], val[RB];
        bool have[RB];
#pragma unroll
        for (int j = 0; j < RB; j++) {
            const int r = r0 + j;
            have[j] = false;
            if (r < ws) {
                const uint32_t lo = lo_s[r], hi = hi_s[r];
                const uint32_t p = lo + threadIdx.x;
                if (p < hi) {
                    const uint32_t* pairs = (const uint32_t*)(wires.w[r] + (uint64_t)b * wire_stride) + 1;
                    off[j] = pairs[2 * (uint64_t)p] - (uint32_t)tstart;
                    val[j] = pairs[2 * (uint64_t)p + 1];
                    have[j] = true;
                }
            }
        }
#pragma unroll
        for (int j = 0; j < RB; j++) {
            const int r = r0 + j;
            if (r < ws) {
                if (have[j]) {
                    if (off[j] < tlen) tile[off[j]] = tile[off[j]] + u2f(val[j]);
                    else if (status) *status = MCCL_HIP_ERR_INDEX;
                }
                // a barrier between ranks keeps the adds to one element in rank order
                __syncthreads();
                // dense tiles (more than kAccThreads pairs of this rank): the rest, still in rank order
                if (hi_s[r] > lo_s[r] + kAccThreads) {  // block-uniform
                    const uint32_t lo = lo_s[r], hi = hi_s[r];
                    const uint32_t* pairs = (const uint32_t*)(wires.w[r] + (uint64_t)b * wire_stride) + 1;
                    for (uint32_t p = lo + kAccThreads + threadIdx.x; p < hi; p += kAccThreads) {
                        const uint32_t o = pairs[2 * (uint64_t)p] - (uint32_t)tstart;
                        if (o < tlen) tile[o] = tile[o] + u2f(pairs[2 * (uint64_t)p + 1]);
                        else if (status) *status = MCCL_HIP_ERR_INDEX;
                    }
                    __syncthreads();
                }
            }
        }
    }
    float* out = acc + bstart + tstart;
    if (tlen == kAccTile && (((uintptr_t)out & 15) == 0)) {
        for (int i = threadIdx.x; i < kAccTile / 4; i += kAccThreads) {
            u4a v;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float x = tile[4 * i + q];
                v[q] = f2u(apply_scale ? x * scale : x);
            }
            __builtin_nontemporal_store(v, (u4a*)out + i);
        }
    } else {
        for (uint32_t i = threadIdx.x; i < tlen; i += kAccThreads) {
            const float x = tile[i];
            out[i] = apply_scale ? x * scale : x;
        }
    }
}

// ---- runs of tiles, one wavefront each ------------------------------------------
// The kernels above pay for finding where a tile's pairs begin: a table that a
// pre-pass builds from a second read of every payload.  Here a wavefront owns a
// run of consecutive 2048-element tiles of one bucket (four tiles at 1 %
// density) and needs a position only where its run begins, and only to the
// nearest 80 pairs.  For each rank it requests three windows of 64 consecutive
// pairs (one pair per lane) when the run begins, all ranks at once, and keeps
// them in registers: every load of the run is issued before its first store
// (a load after stores would wait for their acknowledgements).  A pair belongs
// to the current tile exactly when its index lies inside it; pairs of earlier
// tiles are behind, pairs of later tiles wait in their window.  When the
// window's last index is below the tile's end the next window shifts in and is
// looked at for the same tile; a run denser than its three windows fetches
// further windows one at a time.  The tile sits in LDS (8 KiB per wavefront),
// ranks add in ascending order (the LDS executes one wavefront's operations in
// order, so no barrier is involved), and the tile goes out once, scaled, in
// 16-byte stores.  Everything that decides control flow (tile bounds, window
// ends, counts) lives in scalar registers.
//
// Where a run begins, when a block of a small call does not find it itself (block_starts): k_sparse_starts reads every 80th index (one 128-byte line
// in five) and writes, for every run w, the window that holds the last sampled
// index below the run's first element; every pair before that window belongs to
// an earlier run.
constexpr int kRunL = 2048;    // elements per tile of a wavefront (1024 and 4096 measured 4-5 % slower)
constexpr int kRunWaves = 8;   // wavefronts (= runs) per block: 64 KiB of LDS, two blocks per CU (4 measured 3 % slower, 2 slower still)
constexpr int kRunRanks = 12;  // ranks a wavefront holds windows for (12: 122 registers of 128); larger worlds use the tile kernels
constexpr int kWin = kWave;    // pairs per window
constexpr int kStride = 80;    // pairs between two sampled indices of the position table: five 128-byte lines,
                               // so a run begins with at most 79 pairs of an earlier run in its first window
constexpr int kRunWins = 3;    // windows of a rank a wavefront requests when its run begins
constexpr int kOwnSamples = 16;  // samples a lane holds where a block finds its runs' starts itself: 1024 a payload
constexpr uint64_t kOwnTotal = 2048;   // ... and over all ranks
constexpr uint64_t kOwnBlocks = 512;   // blocks the GPU holds at once: two per CU
constexpr uint64_t kFillWaves = 2048;  // eight wavefronts per CU
constexpr int kXcds = 8;       // accelerator dies of an MI355X; block B runs on die B mod 8

constexpr int kStartThreads = 1024;
constexpr uint32_t kStartSamples = 8192;  // samples of one payload the block keeps in LDS (32 KiB)

// One block per (bucket, rank).  The samples (every 80th index) are requested before k is known
// (inside the payload's capacity, masked afterwards), so the kernel is one round trip: samples
// into LDS, then every run finds by binary search how many samples lie below its first element.
__global__ __launch_bounds__(kStartThreads) void k_sparse_starts(WirePtrs wires, int ws, uint64_t wire_stride,
                                                                 uint32_t run_elems, uint32_t runs, uint32_t* start,
                                                                 int* status) {
    __shared__ uint32_t samp[kStartSamples];
    const uint32_t b = blockIdx.x / (uint32_t)ws, r = blockIdx.x % (uint32_t)ws;
    const uint32_t* wp = (const uint32_t*)(wires.w[r] + (uint64_t)b * wire_stride);
    const uint32_t kmax = (uint32_t)((wire_stride - 4) / 8);
    const uint32_t cap = (kmax + kStride - 1) / kStride;  // samples the payload can hold (at most kStartSamples)
    constexpr int kPer = kStartSamples / kStartThreads;
    uint32_t v[kPer];
#pragma unroll
    for (int i = 0; i < kPer; i++) {
        const uint32_t j = (uint32_t)i * kStartThreads + threadIdx.x;
        v[i] = j < cap ? wp[1 + 2 * (uint64_t)kStride * j] : 0u;
    }
    uint32_t k = wp[0];
    if (k > kmax) {
        if (status) *status = MCCL_HIP_ERR_SIZE;
        k = 0;
    }
    const uint32_t nsamp = (k + kStride - 1) / kStride;
#pragma unroll
    for (int i = 0; i < kPer; i++) {
        const uint32_t j = (uint32_t)i * kStartThreads + threadIdx.x;
        if (j < cap) samp[j] = v[i];
    }
    __syncthreads();
    uint32_t* st = start + ((uint64_t)b * ws + r) * runs;
    for (uint32_t w = threadIdx.x; w < runs; w += kStartThreads) {
        // samples below the run's first element; the last of them names the window to begin in.
        // (Unsorted samples give some window or other; the accumulate kernel trusts no entry.)
        const uint64_t first = (uint64_t)w * run_elems;
        uint32_t lo = 0, hi = nsamp;
        while (lo < hi) {
            const uint32_t mid = lo + ((hi - lo) >> 1);
            if (samp[mid] < first) lo = mid + 1;
            else hi = mid;
        }
        st[w] = lo ? (lo - 1) * kStride : 0u;
    }
}

typedef const __attribute__((address_space(1))) uint32_t* GlobalWords;  // loads compile to global_load, not flat_load

// One window of a rank's pairs: lane l asks for pair base + l.  The load is unconditional (no
// branch, so the loads of all ranks and windows are in flight together): positions past the
// payload's capacity are clamped to its last pair (kmax >= 1) and sorted out by window_index.
__device__ __forceinline__ u2a4 load_window(GlobalWords pairs, uint32_t base, uint32_t kmax, int lane) {
    uint32_t pos = base + (uint32_t)lane;
    if (pos > kmax - 1) pos = kmax - 1;
    return *(const __attribute__((address_space(1))) u2a4*)(pairs + 2 * (uint64_t)pos);
}

// The index a lane holds: lanes at or past k hold 0xFFFFFFFF, which lies in no tile.
__device__ __forceinline__ uint32_t window_index(u2a4 v, uint32_t base, uint32_t k, int lane) {
    return base + (uint32_t)lane < k ? v[0] : 0xFFFFFFFFu;
}

// The value the lane below holds (lane 0: `first`): one DPP move, no LDS traffic.
__device__ __forceinline__ uint32_t from_lane_below(uint32_t v, uint32_t first) {
    // wave_shr:1 - lane l reads lane l - 1 across the whole wavefront; lane 0 keeps `first`
    return (uint32_t)__builtin_amdgcn_update_dpp((int)first, (int)v, 0x138, 0xf, 0xf, false);
}

// Lanes (as a mask) whose pair breaks the rule: indices of a window ascend, continue the pair
// before the window (`before`), and stay inside the bucket.  `idx` is what was loaded, before
// the lanes past k are marked.
__device__ __forceinline__ uint64_t bad_lanes(uint32_t idx, uint32_t base, uint32_t k, uint32_t before, uint32_t bn) {
    const uint32_t up = from_lane_below(idx, before);
    uint64_t m = __ballot(up >= idx);
    if (base == 0) m &= ~1ull;  // the payload's first pair follows nothing
    m |= __ballot(idx >= bn);
    const uint32_t live = k > base ? k - base : 0u;  // lanes that hold a pair of the payload
    return live >= (uint32_t)kWin ? m : m & ((1ull << live) - 1);
}

// tile[off] += v as one LDS instruction that returns nothing.  The LDS adds in IEEE single
// precision, round to nearest even, subnormals kept, and executes one wavefront's instructions in
// the order they were issued, so successive ranks' adds to one element happen in rank order
// with no wait between them.
__device__ __forceinline__ void lds_add(float* p, float v) {
    (void)__hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}

__device__ __forceinline__ uint32_t lane_value(uint32_t v, int l) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, l);
}


// Where the block's runs begin in rank `wave`'s payload, found by that wavefront itself: it holds
// every kStride-th index in registers, and the samples below a run's first element are counted.
// Returns in lane q the start of run first_run + q (what k_sparse_starts would have written), and
// whether the samples are out of order.
__device__ __forceinline__ uint32_t block_starts(const uint8_t* wire, uint32_t kmax, uint64_t first_elem, uint64_t run_elems,
                                                 int lane, bool* unsorted) {
    GlobalWords wp = (GlobalWords)wire;
    const uint32_t cap = (kmax + kStride - 1) / kStride;
    uint32_t v[kOwnSamples];
#pragma unroll
    for (int i = 0; i < kOwnSamples; i++) {
        const uint32_t j = (uint32_t)(i * kWave + lane);
        v[i] = j < cap ? wp[1 + 2 * (uint64_t)kStride * j] : 0xFFFFFFFFu;
    }
    const uint32_t k = wp[0];
    const uint32_t nsamp = k > kmax ? 0u : (k + kStride - 1) / kStride;
    uint32_t prev = 0;
    uint64_t bad = 0;
#pragma unroll
    for (int i = 0; i < kOwnSamples; i++) {
        const uint32_t j = (uint32_t)(i * kWave + lane);
        bad |= __ballot(j > 0 && j < nsamp && from_lane_below(v[i], prev) >= v[i]);
        prev = lane_value(v[i], kWave - 1);
        if (j >= nsamp) v[i] = 0xFFFFFFFFu;  // below no run's first element
    }
    *unsorted = bad != 0;
    uint32_t mine = 0;
#pragma unroll
    for (int q = 0; q < kRunWaves; q++) {
        const uint64_t f = first_elem + (uint64_t)q * run_elems;
        const uint32_t first = f < 0xFFFFFFFFull ? (uint32_t)f : 0xFFFFFFFFu;
        uint32_t n = 0;
#pragma unroll
        for (int i = 0; i < kOwnSamples; i++) n += (uint32_t)__popcll(__ballot(v[i] < first));
        if (lane == q) mine = n ? (n - 1) * kStride : 0u;
    }
    return mine;
}

// NR: ranks the code is unrolled for (six ranks as eight, at 2 %: 94.6 us for 90 M elements, as six 85.8; 9 to 12 ranks,
// 50 M at 1 %: tile kernels 70 to 80 us, so 57 to 66) (ws <= NR; the ranks past ws read rank 0's payload as if
// its k were 0).  wire_stride holds at least one pair.  OWN: no position table, the block finds
// where its runs begin (one bucket, at most kOwnSamples * 64 samples a payload).
template <int NR, bool OWN>
__global__ __launch_bounds__(kRunWaves * kWave, 4) void k_sparse_accumulate_runs(
    float* acc, uint64_t n_total, uint64_t bucket_elems, WirePtrs wires, int ws, uint64_t wire_stride,
    uint32_t run_steps, uint32_t runs, uint32_t nbuckets, uint32_t blocks_per_xcd, const uint32_t* start,
    int apply_scale, float scale, int* status) {
    __shared__ __attribute__((aligned(16))) float tiles[kRunWaves][kRunL];
    const int lane = threadIdx.x & (kWave - 1);
    // the same in every lane; saying so keeps everything derived from it (the run, its tiles,
    // the window tests) in scalar registers and on the scalar unit
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    // blocks go to the XCDs in turn: block B runs on XCD B mod 8.  Each XCD takes one contiguous
    // eighth of the runs, in order, so the windows that neighbouring runs share are found in
    // that XCD's L2 and its stores move through memory in one direction.
    const uint32_t vblock = (blockIdx.x % kXcds) * blocks_per_xcd + blockIdx.x / kXcds;
    const uint64_t grun = (uint64_t)vblock * kRunWaves + (uint32_t)wave;
    __shared__ uint32_t own[kRunWaves][NR];
    if constexpr (OWN) {
        static_assert(NR <= kRunWaves, "a rank per wavefront");
        if (wave < ws) {
            const uint64_t run_elems = (uint64_t)run_steps * kRunL;
            bool unsorted;
            const uint32_t mine = block_starts(wires.w[wave], (uint32_t)((wire_stride - 4) / 8),
                                               (uint64_t)vblock * kRunWaves * run_elems, run_elems, lane, &unsorted);
            if (lane < kRunWaves) own[lane][wave] = mine;
            if (unsorted && status) *status = MCCL_HIP_ERR_INDEX;
        }
        __syncthreads();
    }
    if (grun >= (uint64_t)runs * nbuckets) return;  // whole wavefront; no block barrier follows
    const uint32_t b = (uint32_t)(grun / runs), run = (uint32_t)(grun % runs);
    const uint64_t bstart = (uint64_t)b * bucket_elems;
    const uint32_t bn = (uint32_t)((n_total - bstart) < bucket_elems ? (n_total - bstart) : bucket_elems);
    const uint64_t e0 = (uint64_t)run * run_steps * kRunL;
    if (e0 >= bn) return;
    const uint64_t e1w = e0 + (uint64_t)run_steps * kRunL;
    const uint32_t e1 = e1w < bn ? (uint32_t)e1w : bn;  // end of this run
    const uint32_t kmax = (uint32_t)((wire_stride - 4) / 8);
    float* tile = tiles[wave];
    {
        const u4a z = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int i = 0; i < kRunL / (4 * kWave); i++) ((u4a*)tile)[i * kWave + lane] = z;
    }

    uint64_t bad = 0;       // lanes that saw a pair out of order or out of range, reported once
    bool oversize = false;  // a k beyond the payload's capacity
    // first round trip: every rank's k and the window its pairs of this run begin in
    uint32_t kk[NR], wnext[NR];
    GlobalWords pairs[NR];
    {
        uint32_t kraw[NR], craw[NR];
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const int rr = r < ws ? r : 0;
            GlobalWords wp = (GlobalWords)(wires.w[rr] + (uint64_t)b * wire_stride);
            pairs[r] = wp + 1;
            kraw[r] = wp[0];
            craw[r] = OWN ? own[wave][rr] : ((GlobalWords)start)[((uint64_t)b * ws + rr) * runs + run];
        }
#pragma unroll
        for (int r = 0; r < NR; r++) {
            uint32_t k = kraw[r], c = craw[r];
            if (k > kmax) {
                oversize = true;
                k = 0;
            }
            if (r >= ws) k = 0;
            if (c >= k) c = k ? k - 1 : 0u;  // a table entry is never trusted
            kk[r] = __builtin_amdgcn_readfirstlane(k);
            wnext[r] = __builtin_amdgcn_readfirstlane(c);
        }
    }
    // second round trip: kRunWins windows of every rank at once; a run of the usual density needs
    // no other load
    u2a4 raw[NR][kRunWins];
    uint32_t before[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) {
        before[r] = pairs[r][2 * (uint64_t)(wnext[r] ? wnext[r] - 1 : 0u)];  // only used when the window is not the first
#pragma unroll
        for (int i = 0; i < kRunWins; i++) raw[r][i] = load_window(pairs[r], wnext[r] + (uint32_t)i * kWin, kmax, lane);
    }
    // wlast[r][i]: last index of window i, in a scalar register: whether a tile is done with a
    // window is decided without vector work
    uint32_t widx[NR][kRunWins], wval[NR][kRunWins], wlast[NR][kRunWins];
    int nreg[NR];  // windows of the rank still in registers
#pragma unroll
    for (int r = 0; r < NR; r++) {
        uint32_t prev = lane_value(before[r], 0);
        // The pair in front of the first window must lie before this run: a position-table entry
        // that points past the run's first pair (a table left by another call racing on shared
        // scratch, or sampled from a payload that is not ascending) would drop pairs silently.
        if (wnext[r] > 0 && kk[r] > 0 && prev >= (uint32_t)e0) bad |= 1ull;
#pragma unroll
        for (int i = 0; i < kRunWins; i++) {
            const uint32_t base = wnext[r] + (uint32_t)i * kWin;
            bad |= bad_lanes(raw[r][i][0], base, kk[r], prev, bn);
            widx[r][i] = window_index(raw[r][i], base, kk[r], lane);
            wval[r][i] = raw[r][i][1];
            prev = lane_value(widx[r][i], kWin - 1);  // 0xFFFFFFFF once the payload's end is in the window
            wlast[r][i] = prev;
        }
        wnext[r] += kRunWins * kWin;  // the first window not in registers
        nreg[r] = kRunWins;
    }

    for (uint64_t ts64 = e0; ts64 < e1; ts64 += kRunL) {  // 64-bit: the last tile of a 2^32-element bucket ends past 32 bits
        const uint32_t ts = (uint32_t)ts64;
        const uint32_t tlen = (e1 - ts) < (uint32_t)kRunL ? (e1 - ts) : (uint32_t)kRunL;
        const uint32_t tend = ts + tlen;
#pragma unroll
        for (int r = 0; r < NR; r++) {
            // slot 0 is the window the run has reached; the others wait behind it
            for (;;) {
                const uint32_t off = widx[r][0] - ts;
                if (off < tlen) lds_add(&tile[off], u2f(wval[r][0]));
                if (wlast[r][0] >= tend) break;  // the rest of the window belongs to later tiles
                // the window ends inside this tile: the next one may begin in it
                if (nreg[r] > 1) {
#pragma unroll
                    for (int i = 0; i + 1 < kRunWins; i++) {
                        widx[r][i] = widx[r][i + 1];
                        wval[r][i] = wval[r][i + 1];
                        wlast[r][i] = wlast[r][i + 1];
                    }
                    nreg[r]--;
                } else if (wnext[r] < kk[r]) {
                    // a dense stretch used up the windows requested at the start: further windows
                    // come one at a time, each waited for
                    const u2a4 v = load_window(pairs[r], wnext[r], kmax, lane);
                    bad |= bad_lanes(v[0], wnext[r], kk[r], wlast[r][0], bn);
                    widx[r][0] = window_index(v, wnext[r], kk[r], lane);
                    wval[r][0] = v[1];
                    wlast[r][0] = lane_value(widx[r][0], kWin - 1);
                    wnext[r] += kWin;
                } else {
                    wlast[r][0] = 0xFFFFFFFFu;  // the payload is finished
                    widx[r][0] = 0xFFFFFFFFu;
                    break;
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
        float* out = acc + bstart + ts;
        if (tlen == (uint32_t)kRunL && (((uintptr_t)out & 15) == 0)) {
            // all LDS reads first, so that one wait covers them; then the tile is cleared for the
            // next round and the stores go out
            constexpr int kVecs = kRunL / (4 * kWave);
            u4a v[kVecs];
#pragma unroll
            for (int i = 0; i < kVecs; i++) v[i] = ((u4a*)tile)[i * kWave + lane];
            const u4a z = {0u, 0u, 0u, 0u};
#pragma unroll
            for (int i = 0; i < kVecs; i++) ((u4a*)tile)[i * kWave + lane] = z;
            if (apply_scale) {
#pragma unroll
                for (int i = 0; i < kVecs; i++)
#pragma unroll
                    for (int q = 0; q < 4; q++) v[i][q] = f2u(u2f(v[i][q]) * scale);
            }
#pragma unroll
            for (int i = 0; i < kVecs; i++) {
                __builtin_nontemporal_store(v[i], (u4a*)out + i * kWave + lane);
            }
        } else {
            for (uint32_t i = (uint32_t)lane; i < tlen; i += kWave) {
                const float x = tile[i];
                tile[i] = 0.0f;
                out[i] = apply_scale ? x * scale : x;
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
    if (status) {
        if (bad) *status = MCCL_HIP_ERR_INDEX;
        if (oversize) *status = MCCL_HIP_ERR_SIZE;
    }
}

// Validates the arguments and enqueues the kernels; `workspace` (may be null:
// scratch-free kernel) is known to be large enough.  `shared_table`: it is not the caller's own.
int accumulate(float* acc, uint64_t n_total, uint64_t bucket_elems, const void* const* host_wires, int ws,
               uint64_t wire_stride, int apply_scale, float scale, int* status, void* workspace, bool shared_table,
               void* stream) {
    if (!acc || !host_wires || ws < 1 || ws > MCCL_HIP_MAX_WORLD) return MCCL_HIP_ERR_ARG;
    if (n_total == 0 || n_total > MCCL_HIP_MAX_ELEMS || bucket_elems == 0) return MCCL_HIP_ERR_ARG;
    if (wire_stride < 4 || (wire_stride & 3)) return MCCL_HIP_ERR_ARG;
    if (bucket_elems > n_total) bucket_elems = n_total;
    if (bucket_elems > 0xFFFFFFFFull) return MCCL_HIP_ERR_ARG;
    const uint64_t nb = (n_total + bucket_elems - 1) / bucket_elems;
    if (nb * (uint64_t)ws > 65535) return MCCL_HIP_ERR_ARG;
    WirePtrs wp;
    for (int r = 0; r < MCCL_HIP_MAX_WORLD; r++) wp.w[r] = nullptr;
    for (int r = 0; r < ws; r++) {
        if (!host_wires[r] || ((uintptr_t)host_wires[r] & 3)) return MCCL_HIP_ERR_ARG;
        wp.w[r] = (const uint8_t*)host_wires[r];
    }
    int rc = mccl_hip_init();
    if (rc) return rc;
    hipStream_t st = (hipStream_t)stream;
    const uint32_t tiles = (uint32_t)((bucket_elems + kAccTile - 1) / kAccTile);
    if (!workspace) {
        // no scratch: every block finds its ranges by binary search
        k_sparse_accumulate<<<dim3(tiles, (uint32_t)nb), kBlock, 0, st>>>(acc, n_total, bucket_elems, wp, ws,
                                                                           wire_stride, apply_scale, scale, status);
        return launch_status();
    }
    uint32_t* start = (uint32_t*)(((uintptr_t)workspace + 15) & ~(uintptr_t)15);
    const uint64_t kmax = (wire_stride - 4) / 8;
    // pairs of one rank in a 2048-element tile when the payload is full
    const uint64_t steps_bucket = (bucket_elems + kRunL - 1) / kRunL;
    const uint64_t per_tile = (kmax + steps_bucket - 1) / steps_bucket;
    const int path = tuning().sparse_path;
    const uint64_t samples = (kmax + kStride - 1) / kStride;
    bool runs_take = ws <= kRunRanks && path != 1 && per_tile <= 96 && kmax >= 1 && samples <= kStartSamples;
    uint64_t run_steps = 1, blocks = 0;
    uint32_t runs = 0;
    bool own = false;
    if (runs_take) {
        // a run is as many tiles as bring about 96 pairs of a rank: with up to 79 pairs of the run
        // before it in the first window, the three windows requested at its start (192 pairs) hold a
        // run of the usual density whole, and it never loads again
        run_steps = (uint64_t)tuning().sparse_run_steps;
        if (run_steps == 0) run_steps = per_tile ? 96 / per_tile : 8;
        if (run_steps > 8 && tuning().sparse_run_steps == 0) run_steps = 8;
        // ... but no more than leave every CU eight wavefronts: a wavefront's tiles follow one another,
        // 2-3 us each.  us per call, longer runs against this rule (1 %, position table): 8 ranks of
        // 1 M elements 18.5 / 12.4 (four tiles against one), of 6.5 M 20.4 / 16.6 (four against two);
        // one tile there 17.7
        const uint64_t spread = (steps_bucket * nb + kFillWaves - 1) / kFillWaves;
        if (run_steps > spread && tuning().sparse_run_steps == 0) run_steps = spread;
        if (run_steps < 1) run_steps = 1;
        if (run_steps > steps_bucket) run_steps = steps_bucket;
        runs = (uint32_t)((steps_bucket + run_steps - 1) / run_steps);
        blocks = ((uint64_t)runs * nb + kRunWaves - 1) / kRunWaves;
        // One bucket whose blocks all fit the GPU at once: a block finds its runs' starts itself, if
        // that takes it no more than some 2048 samples over all ranks - each is a memory sector.  us per
        // call, position table against this: 8 ranks of 1 M elements (1000 samples) 12.4 / 11.1, 4 of 2 M
        // (1000) 10.0 / 8.2, 2 of 3 M at 2 % (1500) 10.8 / 8.4, but 8 of 6.5 M (6552) 16.6 / 19.6
        own = nb == 1 && ws <= kRunWaves && blocks <= kOwnBlocks && samples <= (uint64_t)kOwnSamples * kWave &&
              samples * (uint64_t)ws <= kOwnTotal && path != 2;
        // Where the tile kernels take less time all the same: a wavefront's ranks follow one another, a block of theirs
        // has eight wavefronts for a tile.  That tells while the call leaves CUs idle or is dense, and for more ranks
        // than eight.  us per call, runs against tiles: at 1 % 8 ranks of 200,000 elements 10.9 / 9.9, of 4 M 13.2 / 11.3, of
        // 13 M 19.9 / 20.4, 5 ranks of 4 M 11.7 / 10.5, of 13 M 18.1 / 17.9, 3 of 2 M (which find their starts) 7.5 / 8.8, of 8 M
        // 14.1 / 12.3, 12 of 13 M 26.6 / 24.7, of 26 M 39.0 / 46.3; at 2 % 8 of 34 M 56.1 / 49.6, of 60 M 82.4 / 76.7, of 96.5 M
        // 117 / 113, 5 of 60 M 61.2 / 60.1, of 96.5 M 84.5 / 88.8, 9 of 96.5 M 135 / 121, 12 165 / 143; at 0.1 % 9 of 13 M 20.0 / 20.2,
        // and where a block finds its starts 5 of 2 M 9.6 / 10.9, 6 of 4 M 10.4 / 12.0, 8 of 2 M 11.1 / 11.6.
        const uint64_t few = per_tile > 32 ? 64u << 20 : ws > kRunWaves && per_tile > 8 ? 16u << 20 : 8u << 20;
        const bool alone = own && (ws < 5 || per_tile <= 8);  // finds its starts, and its ranks are few or short
        const bool tiles_faster = ws > kRunWaves && per_tile > 32 ? true : n_total <= few && ws >= 2 && !alone;
        // (calls that share a table keep to the runs, which notice a table that is not theirs, and to eight ranks)
        if (path == 0 && tuning().sparse_run_steps == 0) runs_take = shared_table ? ws <= kRunWaves : !tiles_faster;
    }
    if (runs_take) {
        if (!own)
            k_sparse_starts<<<(uint32_t)(nb * ws), kStartThreads, 0, st>>>(wp, ws, wire_stride,
                                                                            (uint32_t)(run_steps * kRunL), runs, start, status);
        const uint32_t per_xcd = (uint32_t)((blocks + kXcds - 1) / kXcds);
        // (more ranks than a block has wavefronts never find their starts: no kernel for those)
#define MCCLHIP_RUNS(NR)                                                                                     \
    (own ? k_sparse_accumulate_runs<(NR <= kRunWaves ? NR : 1), true>                                        \
         : k_sparse_accumulate_runs<NR, false>)<<<per_xcd * kXcds, kRunWaves * kWave, 0, st>>>(              \
        acc, n_total, bucket_elems, wp, ws, wire_stride, (uint32_t)run_steps, runs, (uint32_t)nb, per_xcd,   \
        start, apply_scale, scale, status)
        // Three ranks go as four where a run has two dense tiles: at 2 %, as three / as four, 96.5 M elements 80.6 / 77.1 us, 70 M
        // 62.3 / 59.8, 50 M 47.0 / 46.7; elsewhere as three: at 1 % 96.5 M 75.2 / 75.5, 70 M 60.1 / 61.5, at 3 % (runs of a tile) 91.8 / 96.7
        const bool two_dense = per_tile > 32 && run_steps == 2;
        if (ws == 1) MCCLHIP_RUNS(1);
        else if (ws == 2) MCCLHIP_RUNS(2);
        else if (ws == 3 && !two_dense) MCCLHIP_RUNS(3);
        else if (ws <= 4) MCCLHIP_RUNS(4);
        else if (ws <= 6) MCCLHIP_RUNS(6);
        else if (ws <= 8) MCCLHIP_RUNS(8);
        else if (ws <= 10) MCCLHIP_RUNS(10);
        else MCCLHIP_RUNS(12);
#undef MCCLHIP_RUNS
        return launch_status();
    }
    const uint32_t bx = clamp_u32((kmax + kBlock * 8 - 1) / (kBlock * 8), 1, 0x7FFFFFFF);
    k_sparse_bounds<<<dim3(bx, (uint32_t)(nb * ws)), kBlock, 0, st>>>(wp, ws, wire_stride, n_total, bucket_elems,
                                                                        tiles, start, status);
    k_sparse_accumulate_b<<<dim3(tiles, (uint32_t)nb), kAccThreads, 0, st>>>(acc, n_total, bucket_elems, wp, ws,
                                                                         wire_stride, tiles, start, apply_scale,
                                                                         scale, status);
    return launch_status();
}

}  // namespace

// Called by mccl_hip_init with `device` current, once per device: looks up the
// address of that device's copy of the static scratch array.
int sparse_static_setup(int device) {
    if (device < 0 || device >= kMaxDevices) return MCCL_HIP_OK;  // the static entry point reports it
    if (g_static_ptr[device]) return MCCL_HIP_OK;
    uint32_t* p = nullptr;
    MCCLHIP_TRY(hipGetSymbolAddress((void**)&p, HIP_SYMBOL(scratch)));
    g_static_ptr[device] = p;
    return MCCL_HIP_OK;
}

}  // namespace mcclhip

using namespace mcclhip;

extern "C" {

int mccl_hip_topk_decompress(const void* wire, uint64_t wire_bytes, float* dense, uint64_t count,
                             int* status, void* stream) {
    if (!wire || (!dense && count) || ((uintptr_t)wire & 3)) return MCCL_HIP_ERR_ARG;
    if (count > 0xFFFFFFFFull) return MCCL_HIP_ERR_ARG;
    if (wire_bytes < 4 || ((wire_bytes - 4) & 7)) return MCCL_HIP_ERR_SIZE;
    const uint64_t k64 = (wire_bytes - 4) / 8;
    if (k64 > 0xFFFFFFFFull) return MCCL_HIP_ERR_SIZE;
    int rc = mccl_hip_init();
    if (rc) return rc;
    hipStream_t st = (hipStream_t)stream;
    const uint64_t cap = (uint64_t)device_info().num_cus * (uint64_t)tuning().fold_blocks_per_cu;
    if (count) {
        k_fill_zero<<<clamp_u32((count / 4 + kBlock - 1) / kBlock, 1, cap), kBlock, 0, st>>>(dense, count);
    }
    k_scatter<<<clamp_u32((k64 + kBlock - 1) / kBlock, 1, cap), kBlock, 0, st>>>(
        (const uint32_t*)wire, (uint32_t)k64, dense, count, status);
    return launch_status();
}

int mccl_hip_topk_decompress_sorted(const void* wire, uint64_t wire_bytes, float* dense, uint64_t count,
                                    int* status, void* stream) {
    return mccl_hip_topk_decompress_sorted_flag(wire, wire_bytes, dense, count, status, nullptr, nullptr, stream);
}

int mccl_hip_topk_decompress_sorted_flag(const void* wire, uint64_t wire_bytes, float* dense, uint64_t count,
                                         int* status, const int* flag, int* flag_out, void* stream) {
    if (!wire || !dense || !status || ((uintptr_t)wire & 3) || !flag != !flag_out) return MCCL_HIP_ERR_ARG;
    if (count == 0 || count > 0xFFFFFFFFull) return MCCL_HIP_ERR_ARG;
    if (wire_bytes < 4 || ((wire_bytes - 4) & 7)) return MCCL_HIP_ERR_SIZE;
    const uint64_t k = (wire_bytes - 4) / 8;
    if (k > 0xFFFFFFFFull) return MCCL_HIP_ERR_SIZE;
    int rc = mccl_hip_init();
    if (rc) return rc;
    const uint64_t stride = k ? (k + kDecSamples - 1) / kDecSamples : 1;
    if (stride > kDecMaxStride) {
        if (flag) k_copy_word<<<1, 1, 0, (hipStream_t)stream>>>(flag, flag_out);
        return mccl_hip_topk_decompress(wire, wire_bytes, dense, count, status, stream);
    }
    k_decompress_sorted<false><<<(uint32_t)((count + kDecTile - 1) / kDecTile), kBlock, 0, (hipStream_t)stream>>>(
        (const uint32_t*)wire, (uint32_t)k, (uint32_t)stride, dense, count, status, flag, flag_out, Done{});
    return launch_status();
}

int mccl_hip_topk_decompress_sorted_done(const void* wire, uint64_t wire_bytes, float* dense, uint64_t count, const int* flag,
                                         void* counters, uint64_t* host_word, uint32_t ticket, void* stream) {
    if (!wire || !dense || !counters || !host_word || ((uintptr_t)wire & 3) || ((uintptr_t)counters & 7) || ((uintptr_t)host_word & 7))
        return MCCL_HIP_ERR_ARG;
    if (count == 0 || count > 0xFFFFFFFFull) return MCCL_HIP_ERR_ARG;
    if (wire_bytes < 4 || ((wire_bytes - 4) & 7)) return MCCL_HIP_ERR_SIZE;
    const uint64_t k = (wire_bytes - 4) / 8;
    if (k > 0xFFFFFFFFull) return MCCL_HIP_ERR_SIZE;
    const uint64_t stride = k ? (k + kDecSamples - 1) / kDecSamples : 1;
    if (stride > kDecMaxStride) return MCCL_HIP_ERR_CAPACITY;
    int rc = mccl_hip_init();
    if (rc) return rc;
    k_decompress_sorted<true><<<(uint32_t)((count + kDecTile - 1) / kDecTile), kBlock, 0, (hipStream_t)stream>>>(
        (const uint32_t*)wire, (uint32_t)k, (uint32_t)stride, dense, count, nullptr, flag, nullptr,
        Done{(uint64_t*)counters, host_word, ticket});
    return launch_status();
}

uint64_t mccl_hip_sparse_accumulate_workspace_bytes(uint64_t n_total, uint64_t bucket_elems, int ws) {
    if (n_total == 0 || bucket_elems == 0 || ws < 1 || ws > MCCL_HIP_MAX_WORLD) return 0;
    if (bucket_elems > n_total) bucket_elems = n_total;
    const uint64_t nb = (n_total + bucket_elems - 1) / bucket_elems;
    // one entry per 2048-element tile: room for the table of either kernel pair
    const uint64_t tiles = (bucket_elems + kRunL - 1) / kRunL;
    return nb * (uint64_t)ws * (tiles + 1) * 4 + 64;
}

int mccl_hip_sparse_accumulate(float* acc, uint64_t n_total, uint64_t bucket_elems,
                               const void* const* host_wires, int ws, uint64_t wire_stride,
                               int apply_scale, float scale, int* status, void* workspace,
                               uint64_t workspace_bytes, void* stream) {
    if (workspace && workspace_bytes < mccl_hip_sparse_accumulate_workspace_bytes(n_total, bucket_elems, ws))
        return MCCL_HIP_ERR_WORKSPACE;
    return accumulate(acc, n_total, bucket_elems, host_wires, ws, wire_stride, apply_scale, scale, status,
                      workspace, false, stream);
}

int mccl_hip_sparse_accumulate_static(float* acc, uint64_t n_total, uint64_t bucket_elems,
                                      const void* const* host_wires, int ws, uint64_t wire_stride,
                                      int apply_scale, float scale, int* status, void* stream) {
    const uint64_t need = mccl_hip_sparse_accumulate_workspace_bytes(n_total, bucket_elems, ws);
    if (need == 0) return MCCL_HIP_ERR_ARG;
    if (need > MCCL_HIP_SPARSE_STATIC_BYTES) return MCCL_HIP_ERR_WORKSPACE;
    int rc = mccl_hip_init();  // resolves this device's copy of the scratch array on first use
    if (rc) return rc;
    const int dev = device_info().device;
    if (dev < 0 || dev >= kMaxDevices || !g_static_ptr[dev]) return MCCL_HIP_ERR_RUNTIME;
    return accumulate(acc, n_total, bucket_elems, host_wires, ws, wire_stride, apply_scale, scale, status,
                      g_static_ptr[dev], true, stream);
}

}  // extern "C"
