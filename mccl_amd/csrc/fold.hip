// Chunk-fold kernels for gfx950: the reduction a ring allreduce / reduce-scatter
// applies to every inbound chunk, the AVG scale, the fused add+scale, and the
// W-way fold in ring-step order.
//
// All of them are HBM-bound streaming kernels: every lane moves 16 bytes per
// access (global_load/store_dwordx4), one tile per block in address order.
// The destination is peeled to 16-byte alignment; sources are read with element alignment only, because chunk views
// start at arbitrary element offsets (csrc/backend/ProcessGroupMCCL.cpp:1735-1741).
//
// Arithmetic follows the reference's CPU folds (csrc/metal/AccelerateOps.mm):
// one IEEE fp32 operation per element and step, never an FMA (this file is
// compiled with -ffp-contract=off); fp16/bf16 are widened, operated on in fp32
// and narrowed once with round-to-nearest-even.
#include "common.hip.h"
#include "fold_rows.h"
#include "runtime.h"

#include <algorithm>
#include <type_traits>
#include <vector>

namespace mcclhip {

namespace {

// Binary fold of two 96.5 M-element fp32 arrays that no cache holds: 176 us, 6.58 TB/s of 12 B/element
// (217 us with 256-thread blocks, a 64-bit index per lane and a grid capped at 65,536 blocks); the
// folds of a ring step as one list of 120: 178 us (223).
// Threads per block of the binary folds.  One wavefront per block, one 16-byte vector per lane and
// operand: the set of tiles in flight is one narrow address front, and what a wavefront executes
// beside its three memory instructions is kept to a handful of scalar ones - a block of this size
// moves 3 KiB, so every further instruction shows.  Measured on a bare dst += src over 402 MB
// arrays: 178 / 181 / 187 / 190 us with 64 / 128 / 256 / 1024 threads, 185 and 193 with two and
// four vectors per lane.
static_assert(kFoldBlock == kWave, "one wavefront per block");

template <bool NT>
__device__ __forceinline__ u4a load_vec_a(const u4a* p) {
    if constexpr (NT) return __builtin_nontemporal_load(p);
    else return *p;
}
template <int ES, bool NT>
__device__ __forceinline__ u4a load_vec_u(const void* p) {
    if constexpr (ES == 4) {
        if constexpr (NT) return __builtin_nontemporal_load((const u4u4*)p);
        else return *(const u4u4*)p;
    } else if constexpr (ES == 1) {
        if constexpr (NT) return __builtin_nontemporal_load((const u4u1*)p);
        else return *(const u4u1*)p;
    } else {
        if constexpr (NT) return __builtin_nontemporal_load((const u4u2*)p);
        else return *(const u4u2*)p;
    }
}
// The folds' output: streaming loads, but stores that stay in the memory-side cache (256 MB), which
// gathers them into longer write bursts between the reads and still holds them for the next call.
// Binary fold in place, against streaming stores, three buffer pairs in turn: 2 M elements 4.1 us
// (5.0), 6.5 M 11.0 (12.9), 13 M 20.1 (24.7), 20 M 29.8 (38.5), 26 M 47.9 (47.2), 96.5 M 174.7 (174);
// loads without the hint are 10-40 % slower from 13 M on.  Ring fold, 8 ranks of 96.5 M: 566 (582).
template <bool NT>
__device__ __forceinline__ void store_out(u4a* p, u4a v) {
    if constexpr (NT) store16_agent(p, v);
    else *p = v;
}

// ---- one element / one dword -------------------------------------------------

// KIND: 0 dst (op) src, 1 (dst + src) * scale, 2 dst * scale (src unused)
template <int DT, int OP, int KIND>
__device__ __forceinline__ float fold_f32(float d, float s, float scale) {
    if constexpr (KIND == 0) return op_f32<OP>(d, s);
    else if constexpr (KIND == 1) return (d + s) * scale;  // two roundings: no contraction
    else return d * scale;
}

template <int DT, int OP, int KIND>
__device__ __forceinline__ uint32_t fold_dword(uint32_t d, uint32_t s, float scale) {
    if constexpr (DT == MCCL_HIP_F32) {
        return f2u(fold_f32<DT, OP, KIND>(u2f(d), u2f(s), scale));
    } else {
        float lo = fold_f32<DT, OP, KIND>(widen16<DT>(d & 0xFFFFu), widen16<DT>(s & 0xFFFFu), scale);
        float hi = fold_f32<DT, OP, KIND>(widen16<DT>(d >> 16), widen16<DT>(s >> 16), scale);
        return narrow16<DT>(lo) | (narrow16<DT>(hi) << 16);
    }
}

template <int DT, int OP, int KIND>
__device__ __forceinline__ void fold_elem(void* dst, const void* src, uint64_t i, float scale) {
    if constexpr (DT == MCCL_HIP_F32) {
        float* d = (float*)dst;
        float s = KIND == 2 ? 0.0f : ((const float*)src)[i];
        d[i] = fold_f32<DT, OP, KIND>(d[i], s, scale);
    } else {
        uint16_t* d = (uint16_t*)dst;
        float s = KIND == 2 ? 0.0f : widen16<DT>(((const uint16_t*)src)[i]);
        d[i] = (uint16_t)narrow16<DT>(fold_f32<DT, OP, KIND>(widen16<DT>(d[i]), s, scale));
    }
}

// ---- integral types (DDP metadata, counters) ------------------------------------
// Wrap-around arithmetic, bool folded as raw uint8
// (csrc/metal/AccelerateOps.mm:206-236, csrc/metal/shaders.metal:554-731).
template <typename T, int OP>
__device__ __forceinline__ T fold_int(T d, T s) {
    typedef typename std::make_unsigned<T>::type UT;
    if constexpr (OP == kAdd) return (T)((UT)d + (UT)s);
    else if constexpr (OP == kMul) return (T)((UT)d * (UT)s);
    else if constexpr (OP == kMin) return s < d ? s : d;
    else return s > d ? s : d;
}

// ---- element kinds of a binary fold: 16 bytes and one element -----------------------
template <int DT, int OP, int KIND>
struct FoldFloat {
    static constexpr int size = ElemInfo<DT>::size;
    static constexpr bool needs_src = KIND != 2;
    static __device__ __forceinline__ u4a vec(u4a d, u4a s, float scale) {
        u4a r;
#pragma unroll
        for (int q = 0; q < 4; q++) r[q] = fold_dword<DT, OP, KIND>(d[q], s[q], scale);
        return r;
    }
    static __device__ __forceinline__ void elem(char* d, const char* s, float scale) {
        fold_elem<DT, OP, KIND>(d, s, 0, scale);
    }
};
template <typename T, int OP>
struct FoldInt {
    static constexpr int size = sizeof(T);
    static constexpr bool needs_src = true;
    static __device__ __forceinline__ u4a vec(u4a d, u4a s, float) {
        constexpr int N = 16 / sizeof(T);
        typedef T V __attribute__((ext_vector_type(N)));
        const V dv = __builtin_bit_cast(V, d), sv = __builtin_bit_cast(V, s);
        V r;
#pragma unroll
        for (int i = 0; i < N; i++) r[i] = fold_int<T, OP>(dv[i], sv[i]);
        return __builtin_bit_cast(u4a, r);
    }
    static __device__ __forceinline__ void elem(char* d, const char* s, float) {
        *(T*)d = fold_int<T, OP>(*(const T*)d, *(const T*)s);
    }
};

// ---- binary fold / scale / fused ----------------------------------------------
template <int ES, bool NT>
__device__ __forceinline__ u4a load_src(const void* p) {
    return load_vec_u<(ES == 2 ? 2 : (ES == 1 ? 1 : 4)), NT>(p);
}

// Block `block` of `nblocks` of one fold.
template <class F, bool NT>
__device__ __forceinline__ void fold_span_block(char* dst, const char* src, uint64_t nvec, uint32_t head, uint32_t tail,
                                                uint32_t lead, float scale, uint32_t block, uint32_t nblocks) {
    const uint32_t t = threadIdx.x;
    auto fold_vec = [&](uint64_t v) {
        char* const dp = dst + v * 16;
        const u4a d = load_vec_a<NT>((const u4a*)(dp + t * 16u));
        u4a s = d;
        if constexpr (F::needs_src) s = load_src<F::size, NT>(src + v * 16 + t * 16u);
        store_out<NT>((u4a*)(dp + t * 16u), F::vec(d, s, scale));
    };
    // (the launch gives a block one round unless the grid is capped)
    for (uint64_t v = (uint64_t)block * kFoldBlock; v < nvec; v += (uint64_t)nblocks * kFoldBlock) {
        if (v >= lead && v + kFoldBlock <= nvec) fold_vec(v);  // (uniform)
        else if (v + t >= lead && v + t < nvec) fold_vec(v);
    }
    if (block + 1 == nblocks && (head | tail)) {  // scalars: at most 15 in front of the body, 15 behind it
        constexpr uint32_t EPV = 16 / F::size;
        if (t < head) {
            const int64_t o = (int64_t)lead * 16 - (int64_t)((head - t) * F::size);
            F::elem(dst + o, F::needs_src ? src + o : nullptr, scale);
        } else if (t >= EPV && t - EPV < tail) {
            const uint64_t o = nvec * 16 + (uint64_t)(t - EPV) * F::size;
            F::elem(dst + o, F::needs_src ? src + o : nullptr, scale);
        }
    }
}

template <class F, bool NT>
__global__ __launch_bounds__(kFoldBlock) void k_fold2(char* dst, const char* src, uint64_t nvec, uint32_t head,
                                                      uint32_t tail, uint32_t lead, float scale) {
    fold_span_block<F, NT>(dst, src, nvec, head, tail, lead, scale, blockIdx.x, gridDim.x);
}

// ---- a list of independent binary folds in one launch ---------------------------
// blockIdx.y = fold, blockIdx.x = tile of it (strided where the grid is capped).  The table is read where
// the launch put it, in the kernel-argument segment, one 32-byte scalar load per block (indexing
// the by-value parameter would make the compiler copy it to per-lane scratch memory first): it
// is therefore the only parameter.
constexpr int kFoldBatch = 120;  // folds per launch: the kernel arguments stay below 4 KiB
struct FoldBatch {
    FoldSpan f[kFoldBatch];
};
template <class F, bool NT>
__global__ __launch_bounds__(kFoldBlock) void k_fold2_batch(FoldBatch) {
    typedef const __attribute__((address_space(4))) FoldBatch* Arg;
    const Arg fb = (Arg)__builtin_amdgcn_kernarg_segment_ptr();
    const uint32_t y = blockIdx.y;
    fold_span_block<F, NT>(fb->f[y].dst, fb->f[y].src, fb->f[y].nvec, fb->f[y].head, fb->f[y].tail, fb->f[y].lead,
                           1.0f, blockIdx.x, gridDim.x);
}

// T(float(x) * scale): int32 rounds half away from zero, int64 / uint8 truncate
// (csrc/metal/shaders.metal:622-665).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_scale_int(T* buf, uint64_t n, float scale) {
    for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (uint64_t)gridDim.x * kBlock) {
        float v = (float)buf[i] * scale;
        if constexpr (sizeof(T) == 4) buf[i] = (T)roundf(v);
        else buf[i] = (T)v;
    }
}

// ---- W-way fold in ring-step order --------------------------------------------
// in[i] = buffer of rank i % ws for i < 2 * ws: the ws buffers in ring order
// starting at any rank are ws consecutive entries, which a block fetches with
// one wide scalar load instead of ws dependent ones.
struct RingPtrs {
    const void* in[2 * MCCL_HIP_MAX_WORLD];
};

// blockIdx = (tile, chunk, bucket).  A row of blocks folds one chunk of one bucket, so the first
// rank of the fold is uniform over the block.
// Measured over 96.5 M fp32 elements per rank, 25 MiB buckets, buffers that no cache holds (TB/s, against
// 256-thread blocks with up to eight vectors per lane and rank whose tiles began with the chunk):
// W = 2: 6.6 (6.2), 3: 6.5 (6.2), 4: 6.4 (6.0), 5: 6.3 (6.0), 6: 6.3 (5.7), 7: 6.2 (5.6), 8: 6.2 (5.9);
// bf16 W = 4: 6.5 (6.1), W = 8: 6.4 (5.9).  What bounds it is HBM with reads and writes mixed; the wait
// for the rank pointers behind the computation of the cut was worth 4 % at W = 8.
// WSC > 0 fixes the world size at compile time, so the rank loop unrolls and
// all WSC * ring_unroll(WSC) loads of a thread are in flight together; WSC == 0 reads
// it at run time.
template <int DT, int OP, bool NT, int WSC>
__global__ __launch_bounds__(kFoldBlock) void k_ring_fold(void* out, RingPtrs ptrs, RingCut cut, int ws_rt, float scale,
                                                          int apply_scale, int stepwise) {
    constexpr int ES = ElemInfo<DT>::size;
    constexpr int EPV = ElemInfo<DT>::per_vec;
    constexpr int U = ring_unroll(WSC);
    const int ws = WSC > 0 ? WSC : ws_rt;
    const uint32_t bucket = blockIdx.z, c = blockIdx.y;
    // basic: c < ws; chunked: (c + 1) / 2 <= ws
    const int half = (int)((c + 1) >> 1);
    const int first = cut.chunked ? (half == ws ? 0 : half) : (int)c;
    const void* rp[WSC > 0 ? WSC : 1];  // rank buffers in fold order (compile-time world sizes)
    if constexpr (WSC > 0) {
#pragma unroll
        for (int j = 0; j < WSC; j++) rp[j] = ptrs.in[first + j];
    }
    const RingRow row = ring_row(cut, (uint64_t)(uintptr_t)out, ES, bucket, c);
    const uint64_t e0 = row.e0, len = row.len, head = row.head, nvec = row.nvec;
    const uint32_t lead = row.lead;
    const uint64_t voff = (e0 + head) * ES - lead * 16u;  // byte offset of the first tile

    const uint64_t tile = (uint64_t)kFoldBlock * U;
    auto rank_ptr = [&](int j, int r) -> const char* {
        if constexpr (WSC > 0) return (const char*)rp[j];
        else return (const char*)ptrs.in[r];
    };
    const uint64_t base = (uint64_t)blockIdx.x * tile;
    // (the pointers' load is under way while the cut is computed, not started behind the branch)
    if constexpr (WSC > 0) {
#pragma unroll
        for (int j = 0; j < WSC; j++) asm volatile("" : "+s"(rp[j]));
    }
    if (nvec && base + tile > lead && base < nvec + lead) {
        // byte offsets from the tile's start; outside the chunk its first or last vector is folded and not stored
        const uint32_t end = (uint32_t)(nvec + lead - base < tile ? nvec + lead - base : tile);
        const uint32_t begin = base < lead ? (uint32_t)(lead - base) : 0u;
        uint32_t off[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const uint32_t i = (uint32_t)u * kFoldBlock + threadIdx.x;
            off[u] = (i < begin ? begin : (i < end ? i : end - 1)) * 16u;
        }
        if constexpr (DT == MCCL_HIP_F32) {
            float acc[U][4];
            {
                const char* p = rank_ptr(0, first) + voff + base * 16;
#pragma unroll
                for (int u = 0; u < U; u++) {
                    u4a v = load_vec_u<ES, NT>(p + off[u]);
#pragma unroll
                    for (int q = 0; q < 4; q++) acc[u][q] = u2f(v[q]);
                }
            }
            int r = first;
#pragma unroll
            for (int j = 1; j < ws; j++) {
                r = (r + 1 == ws) ? 0 : r + 1;
                const char* p = rank_ptr(j, r) + voff + base * 16;
                u4a v[U];
#pragma unroll
                for (int u = 0; u < U; u++) v[u] = load_vec_u<ES, NT>(p + off[u]);
#pragma unroll
                for (int u = 0; u < U; u++)
#pragma unroll
                    for (int q = 0; q < 4; q++) acc[u][q] = op_f32<OP>(u2f(v[u][q]), acc[u][q]);
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                u4a rv;
#pragma unroll
                for (int q = 0; q < 4; q++) rv[q] = f2u(apply_scale ? acc[u][q] * scale : acc[u][q]);
                if (off[u] == (uint32_t)(u * kFoldBlock + threadIdx.x) * 16u) store_out<NT>((u4a*)((char*)out + voff + base * 16 + off[u]), rv);
            }
        } else {
            float acc[U][8];
            {
                const char* p = rank_ptr(0, first) + voff + base * 16;
#pragma unroll
                for (int u = 0; u < U; u++) {
                    u4a v = load_vec_u<ES, NT>(p + off[u]);
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        acc[u][2 * q] = widen16<DT>(v[q] & 0xFFFFu);
                        acc[u][2 * q + 1] = widen16<DT>(v[q] >> 16);
                    }
                }
            }
            int r = first;
#pragma unroll
            for (int j = 1; j < ws; j++) {
                r = (r + 1 == ws) ? 0 : r + 1;
                const char* p = rank_ptr(j, r) + voff + base * 16;
                u4a v[U];
#pragma unroll
                for (int u = 0; u < U; u++) v[u] = load_vec_u<ES, NT>(p + off[u]);
#pragma unroll
                for (int u = 0; u < U; u++)
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        float lo = op_f32<OP>(widen16<DT>(v[u][q] & 0xFFFFu), acc[u][2 * q]);
                        float hi = op_f32<OP>(widen16<DT>(v[u][q] >> 16), acc[u][2 * q + 1]);
                        if (stepwise) {
                            lo = widen16<DT>(narrow16<DT>(lo));
                            hi = widen16<DT>(narrow16<DT>(hi));
                        }
                        acc[u][2 * q] = lo;
                        acc[u][2 * q + 1] = hi;
                    }
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                u4a rv;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    float lo = apply_scale ? acc[u][2 * q] * scale : acc[u][2 * q];
                    float hi = apply_scale ? acc[u][2 * q + 1] * scale : acc[u][2 * q + 1];
                    rv[q] = narrow16<DT>(lo) | (narrow16<DT>(hi) << 16);
                }
                if (off[u] == (uint32_t)(u * kFoldBlock + threadIdx.x) * 16u) store_out<NT>((u4a*)((char*)out + voff + base * 16 + off[u]), rv);
            }
        }
    }

    // scalar head and tail of the chunk
    if (blockIdx.x != 0 || (head == 0 && nvec * EPV == len)) return;
    const uint64_t g = threadIdx.x;
    const uint64_t tail = head + nvec * EPV;
    uint64_t i = len;  // element (relative to the chunk) this thread folds, if any
    if (g < head) i = g;
    else if (g >= (uint64_t)EPV && g < 2u * EPV && tail + (g - EPV) < len) i = tail + (g - EPV);
    if (i < len) {
        const uint64_t e = e0 + i;
        float acc;
        if constexpr (DT == MCCL_HIP_F32) acc = ((const float*)ptrs.in[first])[e];
        else acc = widen16<DT>(((const uint16_t*)ptrs.in[first])[e]);
        int r = first;
        for (int j = 1; j < ws; j++) {
            r = (r + 1 == ws) ? 0 : r + 1;
            float x;
            if constexpr (DT == MCCL_HIP_F32) x = ((const float*)ptrs.in[r])[e];
            else x = widen16<DT>(((const uint16_t*)ptrs.in[r])[e]);
            acc = op_f32<OP>(x, acc);
            if constexpr (DT != MCCL_HIP_F32)
                if (stepwise) acc = widen16<DT>(narrow16<DT>(acc));
        }
        if (apply_scale) acc = acc * scale;
        if constexpr (DT == MCCL_HIP_F32) ((float*)out)[e] = acc;
        else ((uint16_t*)out)[e] = (uint16_t)narrow16<DT>(acc);
    }
}

// ---- launch helpers -----------------------------------------------------------

// Blocks for `work_tiles` tiles: one tile per block in address order; the cap only bounds the grid
// for very large arrays (the kernels stride when it applies).
uint32_t stream_blocks(uint64_t work_tiles) {
    const uint64_t cap = (uint64_t)device_info().num_cus * (uint64_t)tuning().fold_blocks_per_cu;
    return clamp_u32(work_tiles, 1, cap);
}

FoldSpan fold_span(void* dst, const void* src, uint64_t n, int es) {
    uint64_t head = ((16 - ((uintptr_t)dst & 15)) & 15) / es;
    if (head > n) head = n;
    const uint64_t body = (n - head) * es / 16;
    FoldSpan f;
    f.head = (uint16_t)head;
    f.tail = (uint16_t)(n - head - body * 16 / es);
    f.lead = body ? (uint32_t)(((uintptr_t)dst + head * es) >> 4) & (kGroupVecs - 1) : 0u;
    f.dst = (char*)dst + head * es - f.lead * 16u;
    f.src = src ? (const char*)src + head * es - f.lead * 16u : nullptr;
    f.nvec = body ? body + f.lead : 0;
    return f;
}

template <class F>
int launch_fold2_f(void* dst, const void* src, uint64_t n, float scale, hipStream_t st) {
    const FoldSpan f = fold_span(dst, src, n, F::size);
    const uint32_t blocks = stream_blocks((f.nvec + kFoldBlock - 1) / kFoldBlock);
    if (tuning().nontemporal)
        k_fold2<F, true><<<blocks, kFoldBlock, 0, st>>>(f.dst, f.src, f.nvec, f.head, f.tail, f.lead, scale);
    else
        k_fold2<F, false><<<blocks, kFoldBlock, 0, st>>>(f.dst, f.src, f.nvec, f.head, f.tail, f.lead, scale);
    return launch_status();
}
template <int DT, int OP, int KIND>
int launch_fold2_t(void* dst, const void* src, uint64_t n, float scale, hipStream_t st) {
    return launch_fold2_f<FoldFloat<DT, OP, KIND>>(dst, src, n, scale, st);
}

// At most kFoldBatch folds a launch (fold_rows.h: how a ragged list is parted).
template <class F>
int launch_fold2_batch_f(void* const* dsts, const void* const* srcs, const uint64_t* counts, uint32_t nfolds,
                         hipStream_t st) {
    const uint64_t cap = (uint64_t)device_info().num_cus * (uint64_t)tuning().fold_blocks_per_cu;
    const bool nt = tuning().nontemporal != 0;
    FoldSpan spans[kFoldBatch];
    uint32_t n = 0;
    auto flush = [&]() {
        if (n) fold_rows(spans, n, [&](const FoldSpan* f, uint32_t m, uint64_t gx) {
            FoldBatch fb = {};
            std::copy(f, f + m, fb.f);
            if (m > 1) gx = (gx + kXcds - 1) / kXcds * kXcds;  // every fold starts on the same XCD
            const dim3 grid(clamp_u32(gx, 1, cap / m > 0 ? cap / m : 1), m, 1);
            if (nt) k_fold2_batch<F, true><<<grid, kFoldBlock, 0, st>>>(fb);
            else k_fold2_batch<F, false><<<grid, kFoldBlock, 0, st>>>(fb);
        });
        n = 0;
    };
    for (uint32_t i = 0; i < nfolds; i++) {
        if (counts[i] == 0) continue;
        spans[n] = fold_span(dsts[i], srcs[i], counts[i], F::size);
        if (++n == (uint32_t)kFoldBatch) flush();
    }
    flush();
    return launch_status();
}

// Calls fn(F{}) with the fold kind of an element type and op.
template <class Fn>
int with_fold_kind(int dtype, int opi, Fn&& fn) {
#define MCCLHIP_KINDS(K)                                       \
    switch (opi) {                                             \
        case kAdd: return fn(K(kAdd){});                       \
        case kMul: return fn(K(kMul){});                       \
        case kMin: return fn(K(kMin){});                       \
        default: return fn(K(kMax){});                         \
    }
#define MCCLHIP_K_F32(OP) FoldFloat<MCCL_HIP_F32, OP, 0>
#define MCCLHIP_K_F16(OP) FoldFloat<MCCL_HIP_F16, OP, 0>
#define MCCLHIP_K_BF16(OP) FoldFloat<MCCL_HIP_BF16, OP, 0>
#define MCCLHIP_K_I32(OP) FoldInt<int32_t, OP>
#define MCCLHIP_K_I64(OP) FoldInt<int64_t, OP>
#define MCCLHIP_K_U8(OP) FoldInt<uint8_t, OP>
    switch (dtype) {
        case MCCL_HIP_F32: MCCLHIP_KINDS(MCCLHIP_K_F32)
        case MCCL_HIP_F16: MCCLHIP_KINDS(MCCLHIP_K_F16)
        case MCCL_HIP_BF16: MCCLHIP_KINDS(MCCLHIP_K_BF16)
        case MCCL_HIP_I32: MCCLHIP_KINDS(MCCLHIP_K_I32)
        case MCCL_HIP_I64: MCCLHIP_KINDS(MCCLHIP_K_I64)
        case MCCL_HIP_BOOL:
        case MCCL_HIP_U8: MCCLHIP_KINDS(MCCLHIP_K_U8)
        default: return MCCL_HIP_ERR_DTYPE;
    }
#undef MCCLHIP_KINDS
#undef MCCLHIP_K_F32
#undef MCCLHIP_K_F16
#undef MCCLHIP_K_BF16
#undef MCCLHIP_K_I32
#undef MCCLHIP_K_I64
#undef MCCLHIP_K_U8
}

template <typename T>
int launch_scale_int(void* buf, uint64_t n, float scale, hipStream_t st) {
    const uint32_t blocks = stream_blocks((n + kBlock - 1) / kBlock);
    k_scale_int<T><<<blocks, kBlock, 0, st>>>((T*)buf, n, scale);
    return launch_status();
}

template <int DT, int OP>
int launch_ring_t(void* out, const RingPtrs& ptrs, int ws, uint64_t n_total, uint64_t bucket_elems,
                  int schedule, uint32_t nchunks, uint32_t nbuckets, float scale, int apply_scale,
                  int stepwise, hipStream_t st) {
    const RingCut cut = ring_cut(n_total, bucket_elems, nbuckets, nchunks, schedule == MCCL_HIP_RING_CHUNKED);
    const uint64_t tiles = ring_tiles(cut, (uint64_t)(uintptr_t)out, ElemInfo<DT>::size, nchunks, ring_tile_vecs(ws));
    // One tile per block, x fastest: blocks are dispatched in address order, so
    // the set of tiles in flight is one contiguous front per rank buffer.  A
    // persistent grid looping inside each chunk row scatters the front over all
    // rows and costs about 13 % of the bandwidth on MI355X.
    if (tiles > 0xFFFFFFFFull / kFoldBlock) return MCCL_HIP_ERR_ARG;  // more than 2^32 threads in a row: a chunk of 68 GB
    dim3 grid((uint32_t)tiles, nchunks, nbuckets);
#define MCCLHIP_RING_LAUNCH(NT, WSC)                                                                  \
    k_ring_fold<DT, OP, NT, WSC><<<grid, kFoldBlock, 0, st>>>(out, ptrs, cut, ws, scale, apply_scale, stepwise)
    const bool nt = tuning().nontemporal != 0;
    switch (ws) {
        // world sizes 2..8 have an unrolled instance each: all loads of a thread are in flight
        // before the first add (the run-time loop measured 0.69 of peak at 6 ranks)
        case 2: if (nt) MCCLHIP_RING_LAUNCH(true, 2); else MCCLHIP_RING_LAUNCH(false, 2); break;
        case 3: if (nt) MCCLHIP_RING_LAUNCH(true, 3); else MCCLHIP_RING_LAUNCH(false, 3); break;
        case 4: if (nt) MCCLHIP_RING_LAUNCH(true, 4); else MCCLHIP_RING_LAUNCH(false, 4); break;
        case 5: if (nt) MCCLHIP_RING_LAUNCH(true, 5); else MCCLHIP_RING_LAUNCH(false, 5); break;
        case 6: if (nt) MCCLHIP_RING_LAUNCH(true, 6); else MCCLHIP_RING_LAUNCH(false, 6); break;
        case 7: if (nt) MCCLHIP_RING_LAUNCH(true, 7); else MCCLHIP_RING_LAUNCH(false, 7); break;
        case 8: if (nt) MCCLHIP_RING_LAUNCH(true, 8); else MCCLHIP_RING_LAUNCH(false, 8); break;
        default: if (nt) MCCLHIP_RING_LAUNCH(true, 0); else MCCLHIP_RING_LAUNCH(false, 0); break;
    }
#undef MCCLHIP_RING_LAUNCH
    return launch_status();
}

template <int DT>
int launch_ring_dt(void* out, const RingPtrs& p, int ws, uint64_t n_total, uint64_t bucket_elems,
                   int schedule, uint32_t nchunks, uint32_t nbuckets, int opi, float scale,
                   int apply_scale, int stepwise, hipStream_t st) {
    switch (opi) {
        case kAdd: return launch_ring_t<DT, kAdd>(out, p, ws, n_total, bucket_elems, schedule, nchunks, nbuckets, scale, apply_scale, stepwise, st);
        case kMul: return launch_ring_t<DT, kMul>(out, p, ws, n_total, bucket_elems, schedule, nchunks, nbuckets, scale, apply_scale, stepwise, st);
        case kMin: return launch_ring_t<DT, kMin>(out, p, ws, n_total, bucket_elems, schedule, nchunks, nbuckets, scale, apply_scale, stepwise, st);
        default: return launch_ring_t<DT, kMax>(out, p, ws, n_total, bucket_elems, schedule, nchunks, nbuckets, scale, apply_scale, stepwise, st);
    }
}

int check_common(const void* a, uint64_t n) {
    if (n == 0) return 1;  // nothing to do
    if (!a || n > MCCL_HIP_MAX_ELEMS) return MCCL_HIP_ERR_ARG;
    return 0;
}

}  // namespace
}  // namespace mcclhip

using namespace mcclhip;

extern "C" {

int mccl_hip_fold2(void* dst, const void* src, uint64_t n, int dtype, int op, void* stream) {
    const int opi = op_index(op);
    if (opi < 0) return MCCL_HIP_ERR_OP;
    int c = check_common(dst, n);
    if (c) return c < 0 ? c : MCCL_HIP_OK;
    if (!src) return MCCL_HIP_ERR_ARG;
    int rc = mccl_hip_init();
    if (rc) return rc;
    hipStream_t st = (hipStream_t)stream;
    return with_fold_kind(dtype, opi, [&](auto f) { return launch_fold2_f<decltype(f)>(dst, src, n, 1.0f, st); });
}

int mccl_hip_fold2_batch(void* const* host_dsts, const void* const* host_srcs, const uint64_t* host_counts,
                         uint32_t nfolds, int dtype, int op, void* stream) {
    const int opi = op_index(op);
    if (opi < 0) return MCCL_HIP_ERR_OP;
    if (nfolds == 0) return MCCL_HIP_OK;
    if (!host_dsts || !host_srcs || !host_counts) return MCCL_HIP_ERR_ARG;
    int es;
    switch (dtype) {
        case MCCL_HIP_F32: case MCCL_HIP_I32: es = 4; break;
        case MCCL_HIP_F16: case MCCL_HIP_BF16: es = 2; break;
        case MCCL_HIP_I64: es = 8; break;
        case MCCL_HIP_BOOL: case MCCL_HIP_U8: es = 1; break;
        default: return MCCL_HIP_ERR_DTYPE;
    }
    for (uint32_t i = 0; i < nfolds; i++) {
        if (host_counts[i] == 0) continue;
        if (!host_dsts[i] || !host_srcs[i] || host_counts[i] > MCCL_HIP_MAX_ELEMS) return MCCL_HIP_ERR_ARG;
    }
    // the folds of one call run in no particular order: a destination may not overlap any other
    // fold's destination or source.  Destinations in address order that do not overlap their
    // neighbours overlap none; a source then has to be compared with those it reaches into.
    struct Range {
        uintptr_t lo, hi;
        uint32_t fold;
    };
    std::vector<Range> d;
    d.reserve(nfolds);
    bool sorted = true;
    for (uint32_t i = 0; i < nfolds; i++) {
        if (host_counts[i] == 0) continue;
        const uintptr_t lo = (uintptr_t)host_dsts[i];
        if (!d.empty() && lo < d.back().lo) sorted = false;
        d.push_back({lo, lo + host_counts[i] * (uint64_t)es, i});
    }
    if (!sorted) std::sort(d.begin(), d.end(), [](const Range& a, const Range& b) { return a.lo < b.lo; });
    for (size_t i = 1; i < d.size(); i++)
        if (d[i].lo < d[i - 1].hi) return MCCL_HIP_ERR_ARG;
    for (uint32_t i = 0; i < nfolds; i++) {
        if (host_counts[i] == 0) continue;
        const uintptr_t lo = (uintptr_t)host_srcs[i], hi = lo + host_counts[i] * (uint64_t)es;
        // the first destination that ends behind the source's start, and those after it
        auto it = std::partition_point(d.begin(), d.end(), [&](const Range& r) { return r.hi <= lo; });
        for (; it != d.end() && it->lo < hi; ++it)
            if (it->fold != i) return MCCL_HIP_ERR_ARG;
    }
    int rc = mccl_hip_init();
    if (rc) return rc;
    hipStream_t st = (hipStream_t)stream;
    return with_fold_kind(dtype, opi, [&](auto f) {
        return launch_fold2_batch_f<decltype(f)>(host_dsts, host_srcs, host_counts, nfolds, st);
    });
}

int mccl_hip_scale(void* buf, uint64_t n, int dtype, float scale, void* stream) {
    int c = check_common(buf, n);
    if (c) return c < 0 ? c : MCCL_HIP_OK;
    int rc = mccl_hip_init();
    if (rc) return rc;
    hipStream_t st = (hipStream_t)stream;
    switch (dtype) {
        case MCCL_HIP_F32: return launch_fold2_t<MCCL_HIP_F32, kAdd, 2>(buf, nullptr, n, scale, st);
        case MCCL_HIP_F16: return launch_fold2_t<MCCL_HIP_F16, kAdd, 2>(buf, nullptr, n, scale, st);
        case MCCL_HIP_BF16: return launch_fold2_t<MCCL_HIP_BF16, kAdd, 2>(buf, nullptr, n, scale, st);
        case MCCL_HIP_I32: return launch_scale_int<int32_t>(buf, n, scale, st);
        case MCCL_HIP_I64: return launch_scale_int<int64_t>(buf, n, scale, st);
        case MCCL_HIP_BOOL:
        case MCCL_HIP_U8: return launch_scale_int<uint8_t>(buf, n, scale, st);
        default: return MCCL_HIP_ERR_DTYPE;
    }
}

int mccl_hip_fold2_scale(void* dst, const void* src, uint64_t n, int dtype, float scale,
                         void* stream) {
    int c = check_common(dst, n);
    if (c) return c < 0 ? c : MCCL_HIP_OK;
    if (!src) return MCCL_HIP_ERR_ARG;
    int rc = mccl_hip_init();
    if (rc) return rc;
    hipStream_t st = (hipStream_t)stream;
    switch (dtype) {
        case MCCL_HIP_F32: return launch_fold2_t<MCCL_HIP_F32, kAdd, 1>(dst, src, n, scale, st);
        case MCCL_HIP_F16: return launch_fold2_t<MCCL_HIP_F16, kAdd, 1>(dst, src, n, scale, st);
        case MCCL_HIP_BF16: return launch_fold2_t<MCCL_HIP_BF16, kAdd, 1>(dst, src, n, scale, st);
        case MCCL_HIP_I32:
        case MCCL_HIP_I64:
        case MCCL_HIP_BOOL:
        case MCCL_HIP_U8:
            // Integral AVG: the add kernel then the scale kernel, as the
            // reference does (csrc/metal/MetalKernels.mm:629-635).
            rc = mccl_hip_fold2(dst, src, n, dtype, MCCL_HIP_SUM, stream);
            if (rc) return rc;
            return mccl_hip_scale(dst, n, dtype, scale, stream);
        default: return MCCL_HIP_ERR_DTYPE;
    }
}

int mccl_hip_ring_fold(void* out, const void* const* host_in, int ws, uint64_t n_total,
                       uint64_t bucket_elems, int schedule, int dtype, int op, int apply_scale,
                       float scale, int stepwise, void* stream) {
    const int opi = op_index(op);
    if (opi < 0) return MCCL_HIP_ERR_OP;
    if (dtype != MCCL_HIP_F32 && dtype != MCCL_HIP_F16 && dtype != MCCL_HIP_BF16) return MCCL_HIP_ERR_DTYPE;
    if (ws < 1 || ws > MCCL_HIP_MAX_WORLD || !host_in) return MCCL_HIP_ERR_ARG;
    if (schedule != MCCL_HIP_RING_BASIC && schedule != MCCL_HIP_RING_CHUNKED) return MCCL_HIP_ERR_ARG;
    int c = check_common(out, n_total);
    if (c) return c < 0 ? c : MCCL_HIP_OK;
    if (bucket_elems == 0) return MCCL_HIP_ERR_ARG;
    RingPtrs ptrs;
    for (int r = 0; r < 2 * MCCL_HIP_MAX_WORLD; r++) ptrs.in[r] = nullptr;
    for (int r = 0; r < ws; r++) {
        if (!host_in[r]) return MCCL_HIP_ERR_ARG;
        ptrs.in[r] = host_in[r];
        ptrs.in[ws + r] = host_in[r];
    }
    int rc = mccl_hip_init();
    if (rc) return rc;
    if (bucket_elems > n_total) bucket_elems = n_total;
    const uint64_t nbuckets64 = (n_total + bucket_elems - 1) / bucket_elems;
    const uint32_t nchunks = (uint32_t)(schedule == MCCL_HIP_RING_CHUNKED ? 2 * ws : ws);
    if (nbuckets64 * nchunks > 65535) return MCCL_HIP_ERR_ARG;  // grid rows
    const uint32_t nb = (uint32_t)nbuckets64;
    hipStream_t st = (hipStream_t)stream;
    switch (dtype) {
        case MCCL_HIP_F32: return launch_ring_dt<MCCL_HIP_F32>(out, ptrs, ws, n_total, bucket_elems, schedule, nchunks, nb, opi, scale, apply_scale, stepwise, st);
        case MCCL_HIP_F16: return launch_ring_dt<MCCL_HIP_F16>(out, ptrs, ws, n_total, bucket_elems, schedule, nchunks, nb, opi, scale, apply_scale, stepwise, st);
        default: return launch_ring_dt<MCCL_HIP_BF16>(out, ptrs, ws, n_total, bucket_elems, schedule, nchunks, nb, opi, scale, apply_scale, stepwise, st);
    }
}

}  // extern "C"
