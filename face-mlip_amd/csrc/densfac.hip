// Factor density D[i, x, b, k] = sum_{e in row i} phi[e, b] msg[m(e), k] Y[e, x] of 20 monomials and B = 16
// radial functions (face/kernels.py:22-118, 135-178): on split bf16 products.
#include "densfac.h"

#include <algorithm>

namespace face {

constexpr int kDfWaves = 4;                                  // 5 monomials each
constexpr int kDfX = 20 / kDfWaves;
constexpr int kDfRow = 36;                                   // floats per edge in LDS: 20 Y, 16 phi

// acc += a b, limbs of b in LDS or registers
__device__ __forceinline__ v16f six(const Split8& a, const v8bf bh, const v8bf bm, const v8bf bl, v16f acc) {
    acc = mfma_32x32x16(a.h, bl, acc);
    acc = mfma_32x32x16(a.m, bm, acc);
    acc = mfma_32x32x16(a.h, bm, acc);
    acc = mfma_32x32x16(a.l, bh, acc);
    acc = mfma_32x32x16(a.m, bh, acc);
    return mfma_32x32x16(a.h, bh, acc);
}

// Forward. Workgroup = atom, wave w = the rows (x, b) of monomials 5w .. 5w + 4 in three blocks of 32, all K
// channels: D = F^T m with F[e, (x, b)] = Y[e, x] phi[e, b] formed and split in the lane (Y and phi of the chunk
// transposed in LDS, 8 edges per operand) and the message rows split once per atom into LDS. Steps of 16
// edges, chunks of kDfSteps of them. Bound by the write of D and, for short rows, by one chain of loads
// per atom; at K = 48 and 64 two waves per SIMD without spills beat three with them (25,000 atoms of 70
// edges, K = 64: 0.79 against 1.04 ms). Against the fp32 matrix-core kernel it replaced: that shape 1.06 ->
// 0.79 ms (2.6 TB/s of writes), 3000 atoms of 37 slots, K = 32, 45 -> 33 us, 864 atoms of 18 edges 12.9 -> 11.8.
constexpr int kDfSteps = 6;
constexpr int kDfCol = 16 * kDfSteps + 4;                    // floats per transposed row in LDS

template <int KS>
__global__ __launch_bounds__(kDfWaves * kWave) __attribute__((amdgpu_waves_per_eu(KS >= 3 ? 2 : 3))) void density_fwd_limb_kernel(
    const float* __restrict__ phi, int ld_phi, const float* __restrict__ msg, int ld_msg,
    const int32_t* __restrict__ msg_row, const float* __restrict__ Y, int ld_Y, const int32_t* __restrict__ row_ptr,
    int M, RankOut D) {
    constexpr int K = 16 * KS, KT = (KS + 1) / 2, S = kDfSteps, EC = 16 * S, kThr = kDfWaves * kWave;
    __shared__ __attribute__((aligned(16))) float tr[36 * kDfCol];               // 20 rows of Y, 16 of phi
    __shared__ v8bf img[S * KT * 3 * kWave];
    const int x_w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) * kDfX;
    const int lane = threadIdx.x & (kWave - 1), half = lane >> 5, el = lane & 31;
    const int64_t i = blockIdx.x;
    int64_t e0, e_end;
    row_range(row_ptr, i, M, e0, e_end);
    const int64_t e_beg = e0;
    v16f acc[3][KT];
#pragma unroll
    for (int rb = 0; rb < 3; ++rb)
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[rb][kt][r] = 0.f;
    float mx = 0.f;
    for (; e0 < e_end; e0 += EC) {
        const int n = (int)min((int64_t)EC, e_end - e0), ns = (n + 15) >> 4;
        if (e0 != e_beg) __syncthreads();
        int tid = threadIdx.x;                               // through an empty asm: no address is held across chunks
        asm volatile("" : "+v"(tid));
        // message rows: one operand (16 edges x 32 channels) per wave and turn
        constexpr int kUm = (S * KT + kDfWaves - 1) / kDfWaves;
        float mv[kUm][8];
#pragma unroll
        for (int u = 0; u < kUm; ++u) {
            const int it = u * kDfWaves + __builtin_amdgcn_readfirstlane(tid / kWave), s = it / KT, kt = it % KT;
            if (s < ns) {
                const int k = min(32 * kt + (tid & 31), K - 1), eb = 16 * s + 8 * ((tid >> 5) & 1);
                int64_t row[8];
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const int64_t e = e0 + min(eb + q, n - 1);
                    row[q] = msg_row ? (int64_t)msg_row[e] : e;
                }
#pragma unroll
                for (int q = 0; q < 8; ++q) mv[u][q] = msg[row[q] * ld_msg + k];
            }
        }
        const int ey = tid / 20, fy = tid - 20 * ey, ep = tid >> 4, fp = tid & 15;
        float yv[S * 16 / 12], pv[S];
#pragma unroll
        for (int u = 0; u < S * 16 / 12; ++u) yv[u] = 12 * u < n ? Y[(e0 + min(12 * u + ey, n - 1)) * ld_Y + fy] : 0.f;
#pragma unroll
        for (int u = 0; u < S; ++u) pv[u] = 16 * u < n ? phi[(e0 + min(16 * u + ep, n - 1)) * ld_phi + fp] : 0.f;
        __builtin_amdgcn_sched_barrier(0);
        float fx = 0.f;                                      // Y phi has limbs when both are within sqrt(kLimbMax)
#pragma unroll
        for (int u = 0; u < S * 16 / 12; ++u) {
            fx = fmaxf(fx, fabsf(yv[u]));
            if (tid < 240) tr[fy * kDfCol + 12 * u + ey] = 12 * u + ey < n ? yv[u] : 0.f;
        }
#pragma unroll
        for (int u = 0; u < S; ++u) {
            fx = fmaxf(fx, fabsf(pv[u]));
            tr[(20 + fp) * kDfCol + 16 * u + ep] = 16 * u + ep < n ? pv[u] : 0.f;
        }
        if (fx > 1.84e19f) mx = 2.f * kLimbMax;
#pragma unroll
        for (int u = 0; u < kUm; ++u) {
            const int it = u * kDfWaves + __builtin_amdgcn_readfirstlane(tid / kWave), s = it / KT, kt = it % KT;
            if (s < ns) {
                const int eb = 16 * s + 8 * ((tid >> 5) & 1);
                const bool in = 32 * kt + (tid & 31) < K;
                v4f a, b;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    a[q] = in && eb + q < n ? mv[u][q] : 0.f;
                    b[q] = in && eb + 4 + q < n ? mv[u][4 + q] : 0.f;
                }
                mx = max_abs8(a, b, mx);
                const Split8 x = split8(a, b);
                v8bf* d = img + it * 3 * kWave + (tid & (kWave - 1));
                d[0] = x.h;
                d[kWave] = x.m;
                d[2 * kWave] = x.l;
            }
        }
        __syncthreads();
        const float* const pb = tr + (20 + (el & 15)) * kDfCol + 8 * half;
#pragma unroll 1
        for (int s = 0; s < ns; ++s) {
            v8bf b[KT][3];
#pragma unroll
            for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                for (int q = 0; q < 3; ++q) b[kt][q] = img[((s * KT + kt) * 3 + q) * kWave + lane];
            const v4f p0 = lds4_at(pb, 16 * s), p1 = lds4_at(pb, 16 * s + 4);
#pragma unroll
            for (int rb = 0; rb < 3; ++rb) {
                const int x = x_w + 2 * rb + (rb < 2 ? el >> 4 : 0);
                const v4f y0 = lds4_at(tr + x * kDfCol + 8 * half, 16 * s);
                const v4f y1 = lds4_at(tr + x * kDfCol + 8 * half, 16 * s + 4);
                const Split8 f = split8(y0 * p0, y1 * p1);
#pragma unroll
                for (int kt = 0; kt < KT; ++kt) acc[rb][kt] = six(f, b[kt][0], b[kt][1], b[kt][2], acc[rb][kt]);
            }
        }
    }
#pragma unroll
    for (int rb = 0; rb < 3; ++rb)
#pragma unroll
        for (int xi = 0; xi < (rb < 2 ? 2 : 1); ++xi) {
            float* const d = D.at(i, x_w + 2 * rb + xi);
#pragma unroll
            for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                for (int r = 0; r < 8; ++r)
                    if (32 * kt + el < K) d[(d_row(r) + 4 * half) * K + 32 * kt + el] = acc[rb][kt][8 * xi + r];
        }
    // values past the limbs' range (or an infinity): the atom once more in plain fp32
    if (__syncthreads_or(mx > kLimbMax)) {
        for (int v = threadIdx.x; v < 320 * K; v += kThr) {
            const int xb = v / K, k = v - xb * K;
            float s = 0.f;
            for (int64_t e = e_beg; e < e_end; ++e)
                s = fmaf(Y[e * ld_Y + (xb >> 4)] * phi[e * ld_phi + (xb & 15)],
                         msg[(msg_row ? (int64_t)msg_row[e] : e) * ld_msg + k], s);
            D.at(i, xb >> 4)[(xb & 15) * K + k] = s;
        }
    }
}

int launch_density_fwd_limb(const float* phi, int ld_phi, const float* msg, int ld_msg, const int32_t* msg_row,
                            const float* Y, int ld_Y, const int32_t* row_ptr, int64_t N, int M, int K, const RankOut& D,
                            hipStream_t st) {
#define FACE_DFL(KS_)                                                                                             \
    hipLaunchKernelGGL((density_fwd_limb_kernel<KS_>), dim3((unsigned)N), dim3(kDfWaves * kWave), 0, st, phi, ld_phi, \
                       msg, ld_msg, msg_row, Y, ld_Y, row_ptr, M, D)
    switch (K / 16) {
        case 1: FACE_DFL(1); break;
        case 2: FACE_DFL(2); break;
        case 3: FACE_DFL(3); break;
        default: FACE_DFL(4); break;
    }
#undef FACE_DFL
    FACE_LAUNCH_CHECK();
    return 0;
}

// Workgroup = atom, wave w = monomials 5w .. 5w + 4 (80 rows (x, b) of the atom's G, three blocks of 32); the row's edges in
// chunks of 32 T, Y, phi and the limbs of the message rows in LDS.
//   1. W[(x, b), e] = sum_k G[x, b, k] m[e, k] with G read once in rows, split in registers and used for
//      all the chunk's edges; D has an edge per lane and 8 b of two monomials in its registers, so
//      dY[e, x] = sum_b W phi and dphi[e, b] = sum_x W Y are multiply-adds in the lane. dphi is summed
//      over the waves through LDS.
//   2. dm[e, k] = sum_{x, b} G[x, b, k] (Y[e, x] phi[e, b]): one 16-step of the product per monomial,
//      Y phi formed and split in the lane; the waves' parts are summed through LDS, wave order, 32
//      edges at a time.
// G is read twice (the second time from L2); the split of G is shared by the edges of the chunk, so T covers
// the longest row in as few chunks as possible (host). Four waves of five monomials, not five of four: the
// waves of a five-wave workgroup do not fill the four SIMDs evenly and only one workgroup fits a CU (155
// against 79 us at 3000 atoms). Three waves per SIMD where the registers allow it, two for the large tiles
// (100,000 atoms, K = 64: 7.6 against 6.5 ms). Bound by the chain of load, product and reduction phases of an atom.
// Against the fp32 matrix-core kernels it replaced: 3000 atoms of 37 slots, K = 32, 100 -> 77 us; 864 atoms of
// 18 edges 28.4 -> 21.5; 100,000 atoms of 70 edges, K = 64, 8.65 -> 5.25 ms.
template <int KS, int T>
__global__ __launch_bounds__(kDfWaves * kWave) __attribute__((amdgpu_waves_per_eu(KS >= 3 || T == 3 ? 2 : 3))) void density_bwd_limb_kernel(
    const float* __restrict__ phi, int ld_phi, const float* __restrict__ msg, int ld_msg,
    const int32_t* __restrict__ msg_row, const float* __restrict__ Y, int ld_Y, const int32_t* __restrict__ row_ptr,
    int M, RankIn G, float* __restrict__ dphi, int ld_dphi, float* __restrict__ dmsg, int ld_dmsg,
    float* __restrict__ dY, int ld_dY) {
    constexpr int K = 16 * KS, KT = (KS + 1) / 2, PS = 36;
    constexpr int kImg = T * KS * 3 * kWave * 16, kDphi = (kDfWaves * 16 + 20) * T * 32 * 4, kDm = kDfWaves * 32 * PS * 4;
    constexpr int kUnion = kImg > kDphi ? (kImg > kDm ? kImg : kDm) : (kDphi > kDm ? kDphi : kDm);
    __shared__ __attribute__((aligned(16))) float yp[T * 32 * kDfRow];
    __shared__ __attribute__((aligned(16))) char uni[kUnion];
    v8bf* const img = reinterpret_cast<v8bf*>(uni);
    float* const part = reinterpret_cast<float*>(uni);
    float* const dyl = part + kDfWaves * T * 32 * 16;        // dY rows behind the waves' dphi parts
    constexpr int kThr = kDfWaves * kWave, kUm = (T * KS * kWave + kThr - 1) / kThr, kUy = (T * 32 + 11) / 12;
    const int x_w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) * kDfX;
    const int64_t i = blockIdx.x;
    int64_t e0, e_end;
    row_range(row_ptr, i, M, e0, e_end);
    for (; e0 < e_end; e0 += 32 * T) {
        const int n = (int)min((int64_t)(32 * T), e_end - e0), nt = (n + 31) >> 5;
        int tid = threadIdx.x;                               // through an empty asm: no address is held across chunks
        asm volatile("" : "+v"(tid));
        const int lane = tid & (kWave - 1), half = lane >> 5, el = lane & 31;
        // row (x, b) of this lane in block rb, from input 8 half on
        auto g_row = [&](int rb) __attribute__((always_inline)) {
            const int x = x_w + 2 * rb;                      // (the last block holds one monomial, twice)
            return (el >> 4 && rb < 2 ? G.at(i, x + 1) : G.at(i, x)) + (el & 15) * K + 8 * half;
        };
        v4f raw[2 * KS];
        auto load_g = [&](const float* p) __attribute__((always_inline)) {
#pragma unroll
            for (int s = 0; s < KS; ++s) raw[2 * s] = ld4(p + 16 * s), raw[2 * s + 1] = ld4(p + 16 * s + 4);
        };
        // every load of the chunk before the first wait: message row indices, G, Y and phi, message rows
        // (edges past the row's end load its last one and are zeroed)
        const float* mp[kUm];
#pragma unroll
        for (int u = 0; u < kUm; ++u) {
            const int v = u * kThr + tid, ln = v & (kWave - 1), s = (v / kWave) % KS, t = v / (kWave * KS);
            const int64_t e = e0 + min(32 * t + (ln & 31), n - 1);
            mp[u] = msg + (msg_row ? (int64_t)msg_row[e] : e) * ld_msg + 16 * s + 8 * (ln >> 5);
        }
        load_g(g_row(0));
        float yv[kUy], pv[2 * T];
        const int ey = tid / 20, fy = tid - 20 * ey, ep = tid >> 4, fp = tid & 15;
#pragma unroll
        for (int u = 0; u < kUy; ++u) yv[u] = Y[(e0 + min(12 * u + ey, n - 1)) * ld_Y + fy];
#pragma unroll
        for (int u = 0; u < 2 * T; ++u) pv[u] = phi[(e0 + min(16 * u + ep, n - 1)) * ld_phi + fp];
        v4f ma[kUm], mb[kUm];
#pragma unroll
        for (int u = 0; u < kUm; ++u) ma[u] = ld4(mp[u]), mb[u] = ld4(mp[u] + 4);
        float mx = 0.f;
        __builtin_amdgcn_sched_barrier(0);
        // Y phi has limbs when both are within the square root of kLimbMax
        float fx = 0.f;
#pragma unroll
        for (int u = 0; u < kUy; ++u) fx = fmaxf(fx, fabsf(yv[u]));
#pragma unroll
        for (int u = 0; u < 2 * T; ++u) fx = fmaxf(fx, fabsf(pv[u]));
        if (fx > 1.84e19f) mx = 2.f * kLimbMax;
#pragma unroll
        for (int u = 0; u < kUy; ++u)
            if (tid < 240 && 12 * u + ey < 32 * T) yp[(12 * u + ey) * kDfRow + fy] = 12 * u + ey < n ? yv[u] : 0.f;
#pragma unroll
        for (int u = 0; u < 2 * T; ++u) yp[(16 * u + ep) * kDfRow + 20 + fp] = 16 * u + ep < n ? pv[u] : 0.f;
#pragma unroll
        for (int u = 0; u < kUm; ++u) {
            const int v = u * kThr + tid, ln = v & (kWave - 1), st = v / kWave;
            const bool in = 32 * (st / KS) + (ln & 31) < n;
            const v4f z = {0.f, 0.f, 0.f, 0.f};
            const v4f a = in ? ma[u] : z, b = in ? mb[u] : z;
            mx = max_abs8(a, b, mx);
            if (st < T * KS) {
                const Split8 x = split8(a, b);
                v8bf* d = img + st * 3 * kWave + ln;
                d[0] = x.h;
                d[kWave] = x.m;
                d[2 * kWave] = x.l;
            }
        }
        __syncthreads();
        // 1. W, dY, dphi
        float dph[T][8];
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int j = 0; j < 8; ++j) dph[t][j] = 0.f;
        float dy[3][T];
#pragma unroll
        for (int rb = 0; rb < 3; ++rb) {
            __builtin_amdgcn_sched_barrier(0);
            v16f acc[T];
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;
            const float* const next = g_row(rb < 2 ? rb + 1 : 2);
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                __builtin_amdgcn_sched_barrier(0);
                const Split8 a = split8(raw[2 * s], raw[2 * s + 1]);
                mx = max_abs8(raw[2 * s], raw[2 * s + 1], mx);
                if (rb < 2) raw[2 * s] = ld4(next + 16 * s), raw[2 * s + 1] = ld4(next + 16 * s + 4);
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    if (t < nt) {
                        const v8bf* b = img + (t * KS + s) * 3 * kWave + lane;
                        acc[t] = six(a, b[0], b[kWave], b[2 * kWave], acc[t]);
                    }
                }
            }
            const int xa = x_w + 2 * rb;
#pragma unroll
            for (int t = 0; t < T; ++t) {
                __builtin_amdgcn_sched_barrier(0);
                if (t < nt) {
                    const float* row = yp + (32 * t + el) * kDfRow;
                    const float ya = row[xa], yb = rb < 2 ? row[xa + 1] : 0.f;
                    const v4f p0 = lds4_at(yp, (32 * t + el) * kDfRow + 20 + 4 * half);
                    const v4f p1 = lds4_at(yp, (32 * t + el) * kDfRow + 28 + 4 * half);
                    float da = 0.f, db = 0.f;
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        const float p = j < 4 ? p0[j] : p1[j - 4];
                        da = fmaf(acc[t][j], p, da);
                        db = fmaf(acc[t][8 + j], p, db);
                        dph[t][j] = fmaf(acc[t][j], ya, fmaf(acc[t][8 + j], yb, dph[t][j]));
                    }
                    // the lower half keeps xa and is given the upper half's part, which keeps xb
                    const float got = __shfl_xor(half ? da : db, 32, kWave);
                    dy[rb][t] = (half ? db : da) + got;
                }
            }
        }
        float gc[2][8];                                      // G by channel for part 2: the lane's channel, 8 b
        auto load_gc = [&](int kt, int xi, float (&g)[8]) __attribute__((always_inline)) {
            const float* p = G.at(i, x_w + xi) + (8 * half * K + min(32 * kt + el, K - 1));
#pragma unroll
            for (int b = 0; b < 8; ++b) g[b] = p[b * K];
        };
        if (dmsg) load_gc(0, 0, gc[0]);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();                                     // the limbs are done with
#pragma unroll
        for (int t = 0; t < T; ++t) {
            if (t < nt) {
                float* d = part + ((x_w / kDfX) * T * 32 + 32 * t + el) * 16 + 4 * half;
                st4(d, (v4f){dph[t][0], dph[t][1], dph[t][2], dph[t][3]});
                st4(d + 8, (v4f){dph[t][4], dph[t][5], dph[t][6], dph[t][7]});
#pragma unroll
                for (int rb = 0; rb < 3; ++rb)
                    if (rb < 2 || !half) dyl[(32 * t + el) * 20 + x_w + 2 * rb + half] = dy[rb][t];
            }
        }
        __syncthreads();
        if (dphi)
            for (int v = tid; v < n * 16; v += kThr) {
                float s = 0.f;
#pragma unroll
                for (int w = 0; w < kDfWaves; ++w) s += part[w * T * 32 * 16 + v];
                dphi[(e0 + (v >> 4)) * ld_dphi + (v & 15)] = s;
            }
        if (dY)
            for (int v = tid; v < n * 20; v += kThr) {
                const int e = v / 20;
                dY[(e0 + e) * ld_dY + v - 20 * e] = dyl[v];
            }
        // 2. dm
        if (dmsg) {
#pragma unroll 1
            for (int kt = 0; kt < KT; ++kt) {                // 32 channels at a time: registers for 12 waves per CU
                v16f acc[T];
#pragma unroll
                for (int t = 0; t < T; ++t)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;
#pragma unroll
                for (int xi = 0; xi < kDfX; ++xi) {
                    __builtin_amdgcn_sched_barrier(0);
                    float (&g)[8] = gc[xi & 1];
                    const Split8 a = split8((v4f){g[0], g[1], g[2], g[3]}, (v4f){g[4], g[5], g[6], g[7]});
                    if (xi + 1 < kDfX) load_gc(kt, xi + 1, gc[(xi + 1) & 1]);
#pragma unroll
                    for (int t = 0; t < T; ++t) {
                        __builtin_amdgcn_sched_barrier(0);
                        if (t < nt) {
                            const float y = yp[(32 * t + el) * kDfRow + x_w + xi];
                            const v4f f0 = y * lds4_at(yp, (32 * t + el) * kDfRow + 20 + 8 * half);
                            const v4f f1 = y * lds4_at(yp, (32 * t + el) * kDfRow + 24 + 8 * half);
                            const Split8 f = split8(f0, f1);
                            acc[t] = six(a, f.h, f.m, f.l, acc[t]);
                        }
                    }
                }
                if (kt + 1 < KT) load_gc(kt + 1, 0, gc[0]);
                __builtin_amdgcn_sched_barrier(0);
                const int kw = min(32, K - 32 * kt) / 4;     // float4s of a row in this block
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    if (t < nt) {
                        __syncthreads();
#pragma unroll
                        for (int g = 0; g < 4; ++g)
                            if (2 * g < kw)
                                st4(part + ((x_w / kDfX) * 32 + el) * PS + 8 * g + 4 * half,
                                    (v4f){acc[t][4 * g], acc[t][4 * g + 1], acc[t][4 * g + 2], acc[t][4 * g + 3]});
                        __syncthreads();
                        const int m = min(32, n - 32 * t);
                        for (int v = tid; v < m * kw; v += kThr) {
                            const int e = v / kw, k = 4 * (v - e * kw);
                            v4f s = lds4_at(part, e * PS + k);
#pragma unroll
                            for (int w = 1; w < kDfWaves; ++w) s += lds4_at(part, (w * 32 + e) * PS + k);
                            float* d = dmsg + (e0 + 32 * t + e) * ld_dmsg + 32 * kt + k;
                            d[0] = s[0], d[1] = s[1], d[2] = s[2], d[3] = s[3];
                        }
                    }
                }
            }
        }
        // values past the limbs' range (or an infinity): the chunk once more in plain fp32
        if (__syncthreads_or(mx > kLimbMax)) {
            for (int v = tid; v < n * K && dmsg; v += kThr) {
                const int e = v / K, k = v - e * K;
                float s = 0.f;
                for (int xb = 0; xb < 320; ++xb)
                    s = fmaf(G.at(i, xb >> 4)[(xb & 15) * K + k],
                             yp[e * kDfRow + (xb >> 4)] * yp[e * kDfRow + 20 + (xb & 15)], s);
                dmsg[(e0 + e) * ld_dmsg + k] = s;
            }
            for (int v = tid; v < n * 36; v += kThr) {
                const int e = v / 36, f = v - 36 * e;        // dY of monomial f, or dphi of b = f - 20
                const float* me = msg + (msg_row ? (int64_t)msg_row[e0 + e] : e0 + e) * ld_msg;
                float s = 0.f;
                for (int o = 0; o < (f < 20 ? 16 : 20); ++o) {
                    const float* g = f < 20 ? G.at(i, f) + o * K : G.at(i, o) + (f - 20) * K;
                    float w = 0.f;
                    for (int k = 0; k < K; ++k) w = fmaf(g[k], me[k], w);
                    s = fmaf(w, yp[e * kDfRow + (f < 20 ? 20 + o : o)], s);
                }
                if (f < 20 && dY) dY[(e0 + e) * ld_dY + f] = s;
                if (f >= 20 && dphi) dphi[(e0 + e) * ld_dphi + f - 20] = s;
            }
            __syncthreads();                                 // LDS is staged anew
        }
    }
}

int launch_density_bwd_limb(const float* phi, int ld_phi, const float* msg, int ld_msg, const int32_t* msg_row,
                            const float* Y, int ld_Y, const int32_t* row_ptr, int64_t N, int M, int max_row, int K,
                            const RankIn& G, float* dphi, int ld_dphi, float* dmsg, int ld_dmsg, float* dY, int ld_dY,
                            hipStream_t st) {
    const int chunks = (max_row + 95) / 96, T = std::min(3, (max_row + 32 * chunks - 1) / (32 * chunks));
#define FACE_DBL(KS_, T_)                                                                                        \
    hipLaunchKernelGGL((density_bwd_limb_kernel<KS_, T_>), dim3((unsigned)N), dim3(kDfWaves * kWave), 0, st, phi, \
                       ld_phi, msg, ld_msg, msg_row, Y, ld_Y, row_ptr, M, G, dphi, ld_dphi, dmsg, ld_dmsg, dY, ld_dY)
#define FACE_DBL_T(KS_)                 \
    switch (T) {                        \
        case 1: FACE_DBL(KS_, 1); break; \
        case 2: FACE_DBL(KS_, 2); break; \
        default: FACE_DBL(KS_, 3); break; \
    }
    switch (K / 16) {
        case 1: FACE_DBL_T(1); break;
        case 2: FACE_DBL_T(2); break;
        case 3: FACE_DBL_T(3); break;
        default: FACE_DBL_T(4); break;
    }
#undef FACE_DBL_T
#undef FACE_DBL
    FACE_LAUNCH_CHECK();
    return 0;
}

}  // namespace face
