// fp32 <-> fp16 transport casts of the FP16 compressor for gfx950
// (csrc/compression/FP16Compression.cpp:16-112).
//
// Semantics are those of the reference's target platform (its NEON branch):
// IEEE round-to-nearest-even with gradual underflow, overflow to infinity, and
// NaN kept NaN with the top mantissa bits and the quiet bit set
// (sign | 0x7C00 | mant >> 13 | 0x200, the rule its portable branch spells out
// at :47-51).  The portable branch (:38-73, :96-111: the one a non-ARM build of
// the reference runs) differs in two places: half subnormals are flushed to
// zero in both directions, and widening passes a NaN's mantissa bits through
// without setting the quiet bit.  The tuning key "fp16_portable" selects that
// behaviour, for bit-identical results with such a build.
//
// Both kernels stream with one tile per block in address order.  A lane owns
// 4 consecutive elements (16 bytes one side, 8 the other), or two such groups a
// block apart; every access of a wavefront covers consecutive addresses.
#include "common.hip.h"
#include "runtime.h"

namespace mcclhip {

namespace {

__device__ __forceinline__ uint32_t f32_to_f16_transport(uint32_t bits) {
    const float f = u2f(bits);
    _Float16 v = (_Float16)f;
    uint16_t h;
    __builtin_memcpy(&h, &v, 2);
    uint32_t r = h;
    if (f != f) r = ((bits >> 16) & 0x8000u) | 0x7C00u | ((bits & 0x7FFFFFu) >> 13) | 0x200u;
    return r;
}

// The portable branch: anything below the smallest normal half becomes a signed zero, also
// what round-to-nearest would have carried up to it.
__device__ __forceinline__ uint32_t f32_to_f16_portable(uint32_t bits) {
    if (((bits >> 23) & 0xFFu) <= 112u) return (bits >> 16) & 0x8000u;
    return f32_to_f16_transport(bits);
}

__device__ __forceinline__ uint32_t f16_to_f32_portable(uint32_t h) {
    const uint32_t sign = (h & 0x8000u) << 16, e = (h >> 10) & 0x1Fu, m = h & 0x3FFu;
    if (e == 0) return sign;
    if (e == 31) return sign | 0x7F800000u | (m << 13);
    return sign | ((e + 112u) << 23) | (m << 13);
}

template <bool PORTABLE>
__device__ __forceinline__ uint32_t narrow_transport(uint32_t bits) {
    return PORTABLE ? f32_to_f16_portable(bits) : f32_to_f16_transport(bits);
}

template <bool PORTABLE>
__device__ __forceinline__ uint32_t widen_transport(uint32_t h) {
    return PORTABLE ? f16_to_f32_portable(h) : f2u(widen_f16(h));
}

// Measured with three buffer pairs in turn, us for 1.6 M / 6.5 M / 26 M / 96.5 M elements (6 B each):
//   narrowing  two groups, one wavefront per block      3.0   6.4  22.2  87.8
//              one group                                3.2   7.3  23.7  84.2
//              8 elements per lane, 256 threads           -   8.2     -  93.2
//   widening   two groups, one wavefront per block      3.0   6.6  22.5  91.6
//              one group, four wavefronts               3.1   7.0  23.3  85.9
//              two groups, four wavefronts, streamed      -   7.4     -  94.3
// Streaming loads throughout, and stores that stay in the memory-side cache, where whoever takes
// the payload reads them.  From kCastLarge elements on neither side fits there, and the shapes of
// the right-hand column win.
constexpr uint64_t kCastLarge = 48u << 20;

template <bool PORTABLE, int THREADS, int GROUPS>
__global__ __launch_bounds__(THREADS) void k_cast_f32_f16(const float* __restrict__ src, uint16_t* __restrict__ dst, uint64_t n) {
    const uint64_t nquad = n / 4;
    uint64_t q0 = (uint64_t)blockIdx.x * (THREADS * GROUPS);
    for (; q0 < nquad; q0 += (uint64_t)gridDim.x * (THREADS * GROUPS)) {
        const float* sp = src + q0 * 4;
        uint16_t* dp = dst + q0 * 4;
        u4a v[GROUPS];
#pragma unroll
        for (int j = 0; j < GROUPS; j++)
            if (q0 + j * THREADS + threadIdx.x < nquad) v[j] = __builtin_nontemporal_load((const u4u4*)(sp + 4 * (j * THREADS + threadIdx.x)));
#pragma unroll
        for (int j = 0; j < GROUPS; j++)
            if (q0 + j * THREADS + threadIdx.x < nquad)
                store8_agent(dp + 4 * (j * THREADS + threadIdx.x),
                             u2a{narrow_transport<PORTABLE>(v[j][0]) | (narrow_transport<PORTABLE>(v[j][1]) << 16),
                                 narrow_transport<PORTABLE>(v[j][2]) | (narrow_transport<PORTABLE>(v[j][3]) << 16)});
    }
    if (blockIdx.x == 0 && threadIdx.x < (n & 3)) dst[nquad * 4 + threadIdx.x] = (uint16_t)narrow_transport<PORTABLE>(f2u(src[nquad * 4 + threadIdx.x]));
}

template <bool PORTABLE, int THREADS, int GROUPS>
__global__ __launch_bounds__(THREADS) void k_cast_f16_f32(const uint16_t* __restrict__ src, float* __restrict__ dst, uint64_t n) {
    const uint64_t nquad = n / 4;
    uint64_t q0 = (uint64_t)blockIdx.x * (THREADS * GROUPS);
    for (; q0 < nquad; q0 += (uint64_t)gridDim.x * (THREADS * GROUPS)) {
        const uint16_t* sp = src + q0 * 4;
        float* dp = dst + q0 * 4;
        u2a h[GROUPS];
#pragma unroll
        for (int j = 0; j < GROUPS; j++)
            if (q0 + j * THREADS + threadIdx.x < nquad) h[j] = __builtin_nontemporal_load((const u2u2*)(sp + 4 * (j * THREADS + threadIdx.x)));
#pragma unroll
        for (int j = 0; j < GROUPS; j++)
            if (q0 + j * THREADS + threadIdx.x < nquad)
                store16_agent(dp + 4 * (j * THREADS + threadIdx.x),
                              u4a{widen_transport<PORTABLE>(h[j][0] & 0xFFFFu), widen_transport<PORTABLE>(h[j][0] >> 16),
                                  widen_transport<PORTABLE>(h[j][1] & 0xFFFFu), widen_transport<PORTABLE>(h[j][1] >> 16)});
    }
    if (blockIdx.x == 0 && threadIdx.x < (n & 3)) dst[nquad * 4 + threadIdx.x] = u2f(widen_transport<PORTABLE>(src[nquad * 4 + threadIdx.x]));
}

uint32_t cast_blocks(uint64_t n, uint64_t per_block) {
    const uint64_t cap = (uint64_t)device_info().num_cus * (uint64_t)tuning().fold_blocks_per_cu;
    return clamp_u32((n + per_block - 1) / per_block, 1, cap);
}

template <bool PORTABLE>
void launch_narrow(const float* src, uint16_t* dst, uint64_t n, hipStream_t st) {
    if (n < kCastLarge) k_cast_f32_f16<PORTABLE, 64, 2><<<cast_blocks(n, 8 * 64), 64, 0, st>>>(src, dst, n);
    else k_cast_f32_f16<PORTABLE, 64, 1><<<cast_blocks(n, 4 * 64), 64, 0, st>>>(src, dst, n);
}
template <bool PORTABLE>
void launch_widen(const uint16_t* src, float* dst, uint64_t n, hipStream_t st) {
    if (n < kCastLarge) k_cast_f16_f32<PORTABLE, 64, 2><<<cast_blocks(n, 8 * 64), 64, 0, st>>>(src, dst, n);
    else k_cast_f16_f32<PORTABLE, 256, 1><<<cast_blocks(n, 4 * 256), 256, 0, st>>>(src, dst, n);
}

}  // namespace
}  // namespace mcclhip

using namespace mcclhip;

extern "C" {

int mccl_hip_cast_f32_to_f16(const float* src, void* dst, uint64_t n, void* stream) {
    if (n == 0) return MCCL_HIP_OK;
    if (!src || !dst || n > MCCL_HIP_MAX_ELEMS || ((uintptr_t)src & 3) || ((uintptr_t)dst & 1)) return MCCL_HIP_ERR_ARG;
    int rc = mccl_hip_init();
    if (rc) return rc;
    if (tuning().fp16_portable) launch_narrow<true>(src, (uint16_t*)dst, n, (hipStream_t)stream);
    else launch_narrow<false>(src, (uint16_t*)dst, n, (hipStream_t)stream);
    return launch_status();
}

int mccl_hip_cast_f16_to_f32(const void* src, float* dst, uint64_t n, void* stream) {
    if (n == 0) return MCCL_HIP_OK;
    if (!src || !dst || n > MCCL_HIP_MAX_ELEMS || ((uintptr_t)dst & 3) || ((uintptr_t)src & 1)) return MCCL_HIP_ERR_ARG;
    int rc = mccl_hip_init();
    if (rc) return rc;
    if (tuning().fp16_portable) launch_widen<true>((const uint16_t*)src, dst, n, (hipStream_t)stream);
    else launch_widen<false>((const uint16_t*)src, dst, n, (hipStream_t)stream);
    return launch_status();
}

}  // extern "C"
