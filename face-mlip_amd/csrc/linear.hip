// Per-edge linear layers on the matrix cores (gfx950; forward as split bf16 products), for layers whose input is a
// per-edge feature row of K <= 64 values and whose output is a per-edge row of F values:
//
//   forward   Y[e] = X[e] W^T + b + T[idx[e]]                            (E, F)
//   backward  dX[e] = dY[e] W                                            (E, K)
//             dT[n] = sum of dY[e] over the edges e with idx[e] = n      (N, F), idx = col
//
// Users: the CP columns of the last radial layer, R = h2 W_cp^T + b_cp (face/model.py:469,
// :496-497; no table), and the pass message gather(msg(h)) + dir_mix(d) (face/model.py:488-493:
// X = d, T = msg(h), idx = col). The backward's table reduction walks each atom's reverse
// edges (rev) the way the gather backward does, so no atomics are needed and the sums are
// bitwise reproducible; the same pass applies W to each visited edge.
#include "edges.h"

#include <algorithm>

namespace face {

// ------------------------------------------------------------------ forward
// D = W . X^T in 32 x 32 blocks as split bf16 products (edges.h): the weight blocks of the workgroup's
// features sit in LDS as limbs, each wave splits the X rows of 32 edges once and walks the blocks, lane
// e holding features 8 g + 4 (lane >> 5) + 0..3 of edge e, one float4 store each. Bound by the write of
// Y; six blocks of 64 inputs (72 KB) leave room for two workgroups per CU (1.25 M edges, 64 -> 160 with
// gathered table rows: 400 us as on fp32 instructions; the form is the one cp_radial_fwd shares).
constexpr int kLinWaves = 4, kLinBlocks = 6;

template <int KB, bool HAS_T>
__global__ __launch_bounds__(kLinWaves * kWave) __attribute__((amdgpu_waves_per_eu(2))) void edge_linear_fwd_kernel(
    const float* __restrict__ X, int ld_X, int64_t E, const float* __restrict__ w, const float* __restrict__ b,
    int F, int nblk, const float* __restrict__ T, int ld_T, const int32_t* __restrict__ idx, float* __restrict__ Y,
    int ld_Y) {
    constexpr int K = 16 * KB;
    extern __shared__ v8bf sW[];                             // nblk limb images, then 32 nblk bias values
    float* const sb = reinterpret_cast<float*>(sW + nblk * kLimbImage<KB>);
    const int tid = threadIdx.x, lane = tid & (kWave - 1), half = lane >> 5;
    const int f_beg = blockIdx.y * nblk * 32;
    const int nf = min(nblk * 32, F - f_beg);                // a multiple of 16
    bool big = stage_limbs<KB>(sW, (nf + 31) / 32, [&](int blk, int f) {
        const int ff = 32 * blk + f;
        return ff < nf ? w + (int64_t)(f_beg + ff) * K : nullptr;
    });
    for (int f = tid; f < nf; f += blockDim.x) sb[f] = b ? b[f_beg + f] : 0.f;
    big = __syncthreads_or(big);
    const int64_t ntile = (E + 31) / 32, stride = (int64_t)gridDim.x * kLinWaves;
    int64_t t = (int64_t)blockIdx.x * kLinWaves + __builtin_amdgcn_readfirstlane(tid / kWave);
    if (t >= ntile) return;
    // rows past E repeat edge E - 1 (never stored); the next tile's rows are loaded while the current
    // one computes
    v4f xn[2 * KB];
    int64_t rn = 0;
    auto load_tile = [&](int64_t tt) __attribute__((always_inline)) {
        const int64_t e = min(tt * 32 + (lane & 31), E - 1);
#pragma unroll
        for (int s = 0; s < KB; ++s) {
            xn[2 * s] = ld4(X + e * ld_X + 16 * s + 8 * half);
            xn[2 * s + 1] = ld4(X + e * ld_X + 16 * s + 8 * half + 4);
        }
        if (HAS_T) rn = idx ? (int64_t)idx[e] : e;
    };
    load_tile(t);
    for (; t < ntile; t += stride) {
        const int64_t e = t * 32 + (lane & 31);
        Split8 x[KB];
        float mx = 0.f;
#pragma unroll
        for (int s = 0; s < KB; ++s) {
            x[s] = split8(xn[2 * s], xn[2 * s + 1]);
            mx = max_abs8(xn[2 * s], xn[2 * s + 1], mx);
        }
        const bool plain = big || __any(mx > kLimbMax);
        const float* const Tr = HAS_T ? T + rn * ld_T + f_beg + 4 * half : nullptr;
        if (t + stride < ntile) load_tile(t + stride);
        float* const Ye = Y + e * ld_Y + f_beg + 4 * half;
#pragma unroll 1
        for (int f0 = 0; f0 < nf; f0 += 32) {
            const int ng = nf - f0 < 32 ? 2 : 4;             // groups of 8 features
            v4f tv[4];
            if (HAS_T) {
#pragma unroll
                for (int g = 0; g < 4; ++g) tv[g] = ld4(Tr + f0 + (g < ng ? 8 * g : 0));
            }
            v16f ac[1];
#pragma unroll
            for (int r = 0; r < 16; ++r) ac[0][r] = 0.f;
            limb_products<KB, 1, false>(
                x, [&](int) __attribute__((always_inline)) { return sW + (f0 / 32) * kLimbImage<KB>; }, lane, ac);
            v16f& acc = ac[0];
            if (plain) {
                const float* xe = X + min(e, E - 1) * ld_X;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float* wf = w + (int64_t)(f_beg + min(f0 + d_row(r) + 4 * half, nf - 1)) * K;
                    float s = 0.f;
#pragma unroll 1
                    for (int k = 0; k < K; ++k) s = fmaf(xe[k], wf[k], s);
                    acc[r] = s;
                }
            }
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                if (g < ng) {
                    const v4f bs = lds4_at(sb, f0 + 8 * g + 4 * half);
                    v4f y;
#pragma unroll
                    for (int i = 0; i < 4; ++i) y[i] = acc[4 * g + i] + bs[i];
                    if (HAS_T) y += tv[g];
                    if (e < E) st4(Ye + f0 + 8 * g, y);
                }
            }
        }
    }
}

// ------------------------------------------------------------------ backward
// One wave per atom n (persistent waves): the edges with idx = n are rev[e] for the edges e of
// row n. Per tile of 16 such edges the wave loads their dY rows as B operands (K index q of
// instruction r of chunk fc = output feature 16 fc + 4q + r), adds them into per-lane partial
// sums of dT[n], and multiplies them by W^T (A operand from an LDS image W^T[k][f], row stride
// F + 4) into dX: D = W^T . dY^T holds input feature 4q + r of edge j in register r of lane
// j + 16q. The 16 edge lanes of the partial sums are reduced once per atom.
constexpr int kLinBwdWaves = 8;

template <int KB, int FCB>
__global__ __launch_bounds__(kLinBwdWaves * kWave) void edge_linear_bwd_kernel(
    const float* __restrict__ dY, int ld_dY, const float* __restrict__ w, int F, const int32_t* __restrict__ row_ptr,
    const int32_t* __restrict__ rev, int64_t N, float* __restrict__ dX, int ld_dX, float* __restrict__ dT,
    int ld_dT) {
    constexpr int K = 16 * KB;
    extern __shared__ float sWT[];
    const int SW = F + 4;
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    if (dX) {
        for (int v0 = 0; v0 < K * F; v0 += 4 * (int)blockDim.x) {
            float buf[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int v = v0 + u * (int)blockDim.x + tid;             // v = c * K + k: coalesced reads of w
                if (v < K * F) buf[u] = w[v];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int v = v0 + u * (int)blockDim.x + tid;
                if (v < K * F) sWT[(v % K) * SW + v / K] = buf[u];
            }
        }
        __syncthreads();
    }
    const int j = lane & 15, q = lane >> 4;
    const int nfc = F / 16;
    const int wv_id = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int64_t stride = (int64_t)gridDim.x * kLinBwdWaves;
    const v4f z4 = {0.f, 0.f, 0.f, 0.f};
    for (int64_t n = (int64_t)blockIdx.x * kLinBwdWaves + wv_id; n < N; n += stride) {
        const int64_t a = row_ptr[n], bnd = row_ptr[n + 1];
        v4f sums[FCB];
#pragma unroll
        for (int fc = 0; fc < FCB; ++fc) sums[fc] = z4;
        // the reverse-edge index of the next tile is loaded before this tile's stores: on gfx9 a
        // wait for a load also waits for every store issued before it
        int64_t ep_next = a + j < bnd ? (int64_t)rev[a + j] : 0;
        for (int64_t t0 = a; t0 < bnd; t0 += 16) {
            const int64_t er = t0 + j;
            const bool ok = er < bnd;
            const int64_t ep = ep_next;
            ep_next = t0 + 16 + j < bnd ? (int64_t)rev[t0 + 16 + j] : 0;
            v4f acc[KB];
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) acc[kb] = z4;
#pragma unroll
            for (int fc = 0; fc < FCB; ++fc) {
                if (fc < nfc) {
                    const v4f g = ok ? ld4(dY + ep * ld_dY + 16 * fc + 4 * q) : z4;
                    sums[fc] += g;
                    if (dX) {
#pragma unroll
                        for (int kb = 0; kb < KB; ++kb) {
                            const v4f wa = lds4_at(sWT, (16 * kb + j) * SW + 16 * fc + 4 * q);
#pragma unroll
                            for (int r = 0; r < 4; ++r) acc[kb] = mfma_16x16x4(wa[r], g[r], acc[kb]);
                        }
                    }
                }
            }
            if (dX && ok) {
#pragma unroll
                for (int kb = 0; kb < KB; ++kb) st4(dX + ep * ld_dX + 16 * kb + 4 * q, acc[kb]);
            }
        }
        if (dT) {
#pragma unroll
            for (int fc = 0; fc < FCB; ++fc) {
                if (fc < nfc) {
                    v4f s = sums[fc];
#pragma unroll
                    for (int o = 1; o < 16; o <<= 1) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) s[r] += __shfl_xor(s[r], o, kWave);
                    }
                    if (j == 0) st4(dT + n * ld_dT + 16 * fc + 4 * q, s);
                }
            }
        }
    }
}

}  // namespace face

using namespace face;

extern "C" int face_edge_linear_fwd(const float* x, int32_t ld_x, int64_t E, int32_t K, const float* w, const float* b,
                                    int32_t F, const float* tab, int32_t ld_tab, const int32_t* idx, float* y,
                                    int32_t ld_y, void* stream) {
    if (E < 0 || K < 16 || K > 64 || K % 16 || F < 16 || F % 16 || ld_x < K || ld_y < F || (tab && ld_tab < F))
        return FACE_ERR_ARG;
    if (E == 0) return 0;
    if (!x || !w || !y) return FACE_ERR_ARG;
    if (ld_x % 4 || ld_y % 4 || (tab && ld_tab % 4) || !aligned16(x) || !aligned16(w) || !aligned16(y) ||
        (b && !aligned16(b)) || (tab && !aligned16(tab)))
        return FACE_ERR_UNSUPPORTED;
    const int all = (F + 31) / 32, parts = (all + kLinBlocks - 1) / kLinBlocks, nblk = (all + parts - 1) / parts;
    const size_t lds = (size_t)nblk * (K / 16 * 3 * kWave * 16 + 32 * sizeof(float));
    if ((int64_t)lds > device_max_lds()) return FACE_ERR_UNSUPPORTED;
    int64_t wgs = std::max<int64_t>(1, 2 * (int64_t)device_cu_count() / parts);   // persistent, two workgroups per CU
    const int64_t need = ((E + 31) / 32 + kLinWaves - 1) / kLinWaves;
    if (need < wgs) wgs = need;
    const dim3 grid((unsigned)wgs, (unsigned)((all + nblk - 1) / nblk)), block(kLinWaves * kWave);
    const hipStream_t st = (hipStream_t)stream;
#define FACE_LINF(KB_)                                                                                        \
    do {                                                                                                      \
        auto kern = tab ? edge_linear_fwd_kernel<KB_, true> : edge_linear_fwd_kernel<KB_, false>;             \
        if (lds > 65536 &&                                                                                    \
            hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) !=    \
                hipSuccess)                                                                                   \
            return FACE_ERR_UNSUPPORTED;                                                                      \
        hipLaunchKernelGGL(kern, grid, block, lds, st, x, ld_x, E, w, b, F, nblk, tab, ld_tab, idx, y, ld_y); \
    } while (0)
    switch (K / 16) {
        case 1: FACE_LINF(1); break;
        case 2: FACE_LINF(2); break;
        case 3: FACE_LINF(3); break;
        default: FACE_LINF(4); break;
    }
#undef FACE_LINF
    FACE_LAUNCH_CHECK();
    return 0;
}

extern "C" int face_edge_linear_bwd(const float* dy, int32_t ld_dy, int32_t F, const float* w, int32_t K,
                                    const int32_t* row_ptr, const int32_t* rev, int64_t N, float* dx, int32_t ld_dx,
                                    float* dtab, int32_t ld_dtab, void* stream) {
    if (N < 0 || K < 16 || K > 64 || K % 16 || F < 16 || F > 256 || F % 16 || ld_dy < F ||
        (dx && ld_dx < K) || (dtab && ld_dtab < F))
        return FACE_ERR_ARG;
    if (N == 0 || (!dx && !dtab)) return 0;
    if (!dy || !row_ptr || !rev || (dx && !w)) return FACE_ERR_ARG;
    if (ld_dy % 4 || (dx && ld_dx % 4) || (dtab && ld_dtab % 4) || !aligned16(dy) || (dx && !aligned16(dx)) ||
        (dtab && !aligned16(dtab)))
        return FACE_ERR_UNSUPPORTED;
    const size_t lds = dx ? (size_t)K * (F + 4) * sizeof(float) : 0;
    if ((int64_t)lds > device_max_lds()) return FACE_ERR_UNSUPPORTED;
    int64_t wgs = (int64_t)device_cu_count() * 2;
    const int64_t need = (N + kLinBwdWaves - 1) / kLinBwdWaves;
    if (need < wgs) wgs = need;
    const dim3 grid((unsigned)wgs), block(kLinBwdWaves * kWave);
    const hipStream_t st = (hipStream_t)stream;
    const int nfc = F / 16;
    const int fcb = nfc <= 2 ? nfc : (nfc <= 4 ? 4 : (nfc <= 8 ? 8 : (nfc <= 10 ? 10 : 16)));
#define FACE_LINB(KB_, FCB_)                                                                                   \
    do {                                                                                                       \
        auto kern = edge_linear_bwd_kernel<KB_, FCB_>;                                                         \
        if (lds > 65536 &&                                                                                     \
            hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) !=     \
                hipSuccess)                                                                                    \
            return FACE_ERR_UNSUPPORTED;                                                                       \
        hipLaunchKernelGGL(kern, grid, block, lds, st, dy, ld_dy, w, F, row_ptr, rev, N, dx, ld_dx, dtab, ld_dtab); \
    } while (0)
#define FACE_LINB_K(FCB_)                 \
    switch (K / 16) {                     \
        case 1: FACE_LINB(1, FCB_); break; \
        case 2: FACE_LINB(2, FCB_); break; \
        case 3: FACE_LINB(3, FCB_); break; \
        default: FACE_LINB(4, FCB_); break; \
    }
    switch (fcb) {
        case 1: FACE_LINB_K(1); break;
        case 2: FACE_LINB_K(2); break;
        case 4: FACE_LINB_K(4); break;
        case 8: FACE_LINB_K(8); break;
        case 10: FACE_LINB_K(10); break;
        default: FACE_LINB_K(16); break;
    }
#undef FACE_LINB_K
#undef FACE_LINB
    FACE_LAUNCH_CHECK();
    return 0;
}
