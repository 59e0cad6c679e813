// Shared by the kernels that walk edge lists: rank blocks of the pooled tensors, equal shares of the
// edges, and per-edge linear layers as split bf16 products.
#pragma once
#include "common.h"

namespace face {

__host__ __device__ constexpr int rank_start(int l) { return l == 0 ? 0 : (l == 1 ? 1 : (l == 2 ? 4 : 10)); }

struct RankOut {
    float* p[4];
    int64_t sa, sx;
    __device__ __forceinline__ float* at(int64_t i, int x) const {
        float* b = x < 1 ? p[0] : (x < 4 ? p[1] : (x < 10 ? p[2] : p[3]));
        return b + i * sa + (int64_t)(x - rank_start(rank_of(x))) * sx;
    }
};
struct RankIn {
    const float* p[4];
    int64_t sa, sx;
    __device__ __forceinline__ const float* at(int64_t i, int x) const {
        const float* b = x < 1 ? p[0] : (x < 4 ? p[1] : (x < 10 ? p[2] : p[3]));
        return b + i * sa + (int64_t)(x - rank_start(rank_of(x))) * sx;
    }
};

// Smallest r in [0, n] with a[r] >= target (a nondecreasing, a[n] >= target), the 64 lanes of
// the wave probing 64 points per pass; the result is wave-uniform.
__device__ __forceinline__ int64_t wave_lower_bound(const int32_t* __restrict__ a, int64_t n, int64_t target,
                                                    int lane) {
    int64_t lo = 0, hi = n;
    while (lo < hi) {
        const int64_t step = (hi - lo + kWave - 1) / kWave;
        const int64_t p = min(lo + (int64_t)lane * step, hi);
        const uint64_t m = __ballot(a[p] >= target);      // a[hi] >= target: clamped probes are true
        if (m == 0) {
            lo += (int64_t)(kWave - 1) * step + 1;
        } else {
            const int f = __ffsll((unsigned long long)m) - 1;
            const int64_t pf = min(lo + (int64_t)f * step, hi);
            if (f > 0) lo += (int64_t)(f - 1) * step + 1;
            hi = pf;
        }
    }
    return lo < n ? lo : n;
}

// A wave-uniform 64-bit value held in scalar registers.
__device__ __forceinline__ int64_t uniform64(int64_t v) {
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)v >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
}

// Rank-block descriptors from the C-ABI arguments; every rank the NX monomials touch needs a pointer.
static inline bool rank_out(float* const* p, int64_t sa, int64_t sx, int NX, RankOut& r) {
    const int nr = NX == 20 ? 4 : 2;
    for (int l = 0; l < 4; ++l) r.p[l] = (p && l < nr) ? p[l] : nullptr;
    r.sa = sa;
    r.sx = sx;
    for (int l = 0; l < nr; ++l)
        if (!r.p[l]) return false;
    return sa > 0 && sx > 0;
}
static inline bool rank_in(const float* const* p, int64_t sa, int64_t sx, int NX, RankIn& r) {
    const int nr = NX == 20 ? 4 : 2;
    for (int l = 0; l < 4; ++l) r.p[l] = (p && l < nr) ? p[l] : nullptr;
    r.sa = sa;
    r.sx = sx;
    for (int l = 0; l < nr; ++l)
        if (!r.p[l]) return false;
    return sa > 0 && sx > 0;
}

static inline bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// ------------------------------------------------------------------ per-edge linear layers
// One product of 32 edges by 32 output features, K = 16 HB <= 64 inputs, as six bf16 products per 16
// inputs (Split8, common.h). The features' weights sit in LDS as limbs in operand order,
// [16-input step][limb][64 lanes] of 16 bytes, so every operand is one conflict-free ds_read_b128.
// The order of the six products is the same in every kernel and for either operand role, so a layer
// gives the same bits wherever it is computed.
template <int HB>
constexpr int kLimbImage = HB * 3 * kWave;                   // 16-byte items of 32 features

// Largest magnitude of the values (NaN ignored: it reaches the result either way).
__device__ __forceinline__ float max_abs8(v4f a, v4f b, float m) {
#pragma unroll
    for (int i = 0; i < 4; ++i) m = fmaxf(m, fmaxf(fabsf(a[i]), fabsf(b[i])));
    return m;
}
// Past the largest bf16 a value has no finite limb: such tiles are recomputed in plain fp32.
constexpr float kLimbMax = 3.38953139e38f;

// Limb image of `nblk` blocks of 32 features; row(blk, f) -> the feature's K weights (16-byte aligned)
// or null (zeros). True in the threads that met a value past kLimbMax.
template <int HB, typename Row>
__device__ __forceinline__ bool stage_limbs(v8bf* img, int nblk, Row row) {
    float big = 0.f;
    for (int v = threadIdx.x; v < nblk * HB * kWave; v += blockDim.x) {
        const int ln = v & (kWave - 1), s = (v / kWave) % HB, blk = v / (kWave * HB);
        const float* p = row(blk, ln & 31);
        v4f a = {0.f, 0.f, 0.f, 0.f}, b = a;
        if (p) {
            a = ld4(p + 16 * s + 8 * (ln >> 5));
            b = ld4(p + 16 * s + 8 * (ln >> 5) + 4);
        }
        big = max_abs8(a, b, big);
        const Split8 x = split8(a, b);
        v8bf* d = img + (blk * HB + s) * 3 * kWave + ln;
        d[0] = x.h;
        d[kWave] = x.m;
        d[2 * kWave] = x.l;
    }
    return big > kLimbMax;
}

// acc[l] += x w_l over all 16-input steps for NL feature blocks (images img(l)), EDGES the rows (A operand)
// or the columns (B operand) of D. One operand's registers hold the next operand as soon as its last
// product is issued, so every read has 3 to 5 products (96 to 160 cycles) to arrive and the weights take
// 12 registers; the barriers keep that order (left to itself the compiler waits for each read).
template <int HB, int NL, bool EDGES_ARE_ROWS, typename Img>
__device__ __forceinline__ void limb_products(const Split8 (&x)[HB], Img img, int lane, v16f (&acc)[NL]) {
    v8bf w0 = img(0)[lane], w1 = img(0)[kWave + lane], w2 = img(0)[2 * kWave + lane];
#pragma unroll
    for (int i = 0; i < HB * NL; ++i) {
        const int s = i / NL, l = i % NL;
        const bool more = i + 1 < HB * NL;
        const v8bf* nx = img((i + 1) % NL) + (more ? (i + 1) / NL : 0) * 3 * kWave + lane;
        auto mm = [&](v8bf xe, v8bf we) __attribute__((always_inline)) {
            acc[l] = EDGES_ARE_ROWS ? mfma_32x32x16(xe, we, acc[l]) : mfma_32x32x16(we, xe, acc[l]);
        };
        mm(x[s].h, w2);
        if (more) w2 = nx[2 * kWave];
        __builtin_amdgcn_sched_barrier(0);
        mm(x[s].m, w1);
        mm(x[s].h, w1);
        if (more) w1 = nx[kWave];
        __builtin_amdgcn_sched_barrier(0);
        mm(x[s].l, w0);
        mm(x[s].m, w0);
        mm(x[s].h, w0);
        if (more) w0 = nx[0];
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Row (of 32) that register r of a lane holds in the layout of D.
__device__ __forceinline__ constexpr int d_row(int r) { return 8 * (r >> 2) + (r & 3); }   // + 4 (lane >> 5)

}  // namespace face
