// Shared definitions for the FACE hot-path kernels (gfx950, wave64).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/face_hip.h"

#define FACE_LAUNCH_CHECK()                               \
    do {                                                  \
        hipError_t e_ = hipGetLastError();                \
        if (e_ != hipSuccess) return (int)e_;             \
    } while (0)

namespace face {

constexpr int kWave = 64;

// Rank of each of the 20 symmetric monomials (1 | x y z | 6 rank-2 | 10 rank-3).
__host__ __device__ constexpr int rank_of(int x) { return x == 0 ? 0 : (x < 4 ? 1 : (x < 10 ? 2 : 3)); }

// Edge range of receiver atom i: CSR row_ptr, or the uniform padded stride M when row_ptr is null.
__device__ __forceinline__ void row_range(const int32_t* __restrict__ row_ptr, int64_t i, int M, int64_t& e0,
                                          int64_t& e1) {
    if (row_ptr) {
        e0 = row_ptr[i];
        e1 = row_ptr[i + 1];
    } else {
        e0 = i * (int64_t)M;
        e1 = e0 + M;
    }
}

// Butterfly sum over aligned groups of `width` lanes (width a power of two <= 64); every
// lane of the group ends with the group total.
__device__ __forceinline__ float group_sum(float v, int width) {
    for (int o = width >> 1; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
    return v;
}

// Cross-lane data movement on the VALU (DPP), no LDS round trip: the value of the lane that the
// DPP control selects within the lane's 16-lane row (all lanes of the row active).
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}

// Sum over each aligned group of 16 lanes, every lane ending with its group's total: lane ^ 1 and
// lane ^ 2 (quad permutes), then the other quad of the half row (row_half_mirror, 7 - i) and the
// other half row (row_mirror, 15 - i), which after the first two steps hold the same partial sums
// that lane ^ 4 and lane ^ 8 would: the pairing and rounding of group_sum(v, 16), bit for bit,
// in four VALU instructions instead of four LDS permutes.
__device__ __forceinline__ float row16_sum(float v) {
    v += dpp_f<0xB1>(v);                                 // quad_perm [1, 0, 3, 2]
    v += dpp_f<0x4E>(v);                                 // quad_perm [2, 3, 0, 1]
    v += dpp_f<0x141>(v);                                // row_half_mirror
    v += dpp_f<0x140>(v);                                // row_mirror
    return v;
}

// fp32 matrix-core helpers. v_mfma_f32_16x16x4f32 operand layouts (wave64): A[i][k] in lane
// i + 16k, B[k][j] in lane j + 16k, D[4q + r][j] in register r of lane j + 16q.
typedef float v4f __attribute__((ext_vector_type(4)));

__device__ __forceinline__ v4f mfma_16x16x4(float a, float b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// fp32 products on the bf16 matrix cores. x = h + m + l with h = bf16(x), m = bf16(x - h),
// l = bf16(x - h - m), each rounded to nearest: the three limbs hold the 24 bits of x, and
// x w = xh wh + (xh wm + xm wh) + (xm wm + xh wl + xl wh) up to the three products left out, together below
// 2^-24 of |x w|, half an ulp of fp32 (1.98 2^-25 at x = w = 0x1.00ff8p0; of random pairs one in 700 passes
// 2^-25). Six v_mfma_f32_32x32x16_bf16 do the work of sixteen 16x16x4 fp32 products of the same
// shape in 192 cycles instead of 512 (register-only loops: 1300-1580 / 6 = 217-263 against 110-137
// TFLOP/s), and with fp32 accumulation over fewer, longer dot products their sums are closer to
// 64 bits (relative error of a K = 160 / 512 / 1024 sum 1.7e-7 / 3.4e-7 / 4.9e-7 against 2.2e-7 /
// 4.0e-7 / 5.8e-7). Both ends of the range: values past the largest bf16 (and infinities) have a NaN limb;
// below |x| = 2^-110 the low limb ends at bf16's smallest subnormal, and x is held to 2^-134 only.
// Operand layouts (wave64): A[i][k], k = 8 (lane >> 5) + e in element e of lane i + 32 (k >> 3);
// B[k][j] likewise by j; D[8 (r >> 2) + 4 (lane >> 5) + (r & 3)][lane & 31] in register r.
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

struct Split8 {                                              // eight consecutive k of one row, in limbs
    v8bf h, m, l;
};
__device__ __forceinline__ uint32_t bf16_pair(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((v2f){a, b}, v2bf));
}
__device__ __forceinline__ Split8 split8(v4f a, v4f b) {
    v4u h, m, l;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const float x0 = p < 2 ? a[2 * p] : b[2 * p - 4], x1 = p < 2 ? a[2 * p + 1] : b[2 * p - 3];
        h[p] = bf16_pair(x0, x1);
        const float r0 = x0 - __builtin_bit_cast(float, h[p] << 16);
        const float r1 = x1 - __builtin_bit_cast(float, h[p] & 0xffff0000u);
        m[p] = bf16_pair(r0, r1);
        l[p] = bf16_pair(r0 - __builtin_bit_cast(float, m[p] << 16), r1 - __builtin_bit_cast(float, m[p] & 0xffff0000u));
    }
    return {__builtin_bit_cast(v8bf, h), __builtin_bit_cast(v8bf, m), __builtin_bit_cast(v8bf, l)};
}
__device__ __forceinline__ v16f mfma_32x32x16(v8bf a, v8bf b, v16f c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ v4f ld4(const float* p) { return *reinterpret_cast<const v4f*>(p); }

// float4 read of an LDS image (16-byte aligned base) at a float offset that is a multiple of 4:
// one ds_read_b128. A plain pointer cast at a runtime offset leaves the alignment unknown to
// the compiler, which then splits the read into 32-bit pairs (ds_read2_b32).
__device__ __forceinline__ v4f lds4_at(const float* base, int off) {
    return reinterpret_cast<const v4f*>(__builtin_assume_aligned(base, 16))[off >> 2];
}
__device__ __forceinline__ void st4(float* p, v4f v) { *reinterpret_cast<v4f*>(p) = v; }

// Workgroup copy of n float4 items, put(v, src(v)) for v < n, U loads per thread issued before
// their U stores: a staging loop that stores each item before loading the next one waits a
// full memory latency per round.
template <int U, typename Src, typename Put>
__device__ __forceinline__ void stage4(int n, Src src, Put put) {
    const int tid = threadIdx.x, nthr = blockDim.x;
    for (int v0 = 0; v0 < n; v0 += U * nthr) {
        v4f b[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int v = v0 + u * nthr + tid;
            if (v < n) b[u] = src(v);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int v = v0 + u * nthr + tid;
            if (v < n) put(v, b[u]);
        }
    }
}

// Attribute of the current device, cached per device and attribute slot (fallback if the
// query fails).
template <int Slot>
static inline int device_attr(hipDeviceAttribute_t a, int fallback) {
    constexpr int kMaxDev = 64;
    static int cache[kMaxDev];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDev) return fallback;
    int& v = cache[dev];
    if (v <= 0 && (hipDeviceGetAttribute(&v, a, dev) != hipSuccess || v <= 0)) v = fallback;
    return v;
}
static inline int device_cu_count() { return device_attr<0>(hipDeviceAttributeMultiprocessorCount, 256); }
static inline int device_max_lds() { return device_attr<1>(hipDeviceAttributeMaxSharedMemoryPerBlock, 65536); }

}  // namespace face
