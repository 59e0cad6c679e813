// Row-block linear layers of the node features on the matrix cores (gfx950), fp32 in and out:
//
//   y[m, :] = (beta y0[m, :] + (op(x)[m, :] * xs[m, :]) W^T + bias) * ys[m, :]    (per problem)
//
// for the tall activations of a pass, (k_l N, C) blocks against weights of at most a few
// hundred columns: mix, tmix and proj (face/model.py:498-533, :537-544), the readout layers
// (face/model.py:331-339) and their input gradients. xs / ys are per-atom scale rows picked by the
// atom's element (the elem_scale factor of face/model.py:530-533) and are optional, as are beta and
// bias. Up to eight problems share one launch.
//
// The products are six bf16 matrix products of the operands' three-way splits (common.h). A
// workgroup of NW waves owns a tile of 32 NW rows and a slice of NSB = 32 NB output columns; each
// wave keeps its 32 x NSB outputs in registers over the whole K loop. The x rows stream from memory
// straight into the waves' A operands (lane i + 32 h holds columns 8 h .. 8 h + 7 of row i; a chunk of 32
// columns is one 128-byte line per row), loaded one chunk ahead, scaled or transformed and split in
// registers. The weight slice streams through LDS in chunks of 32 k, double-buffered, split once per
// workgroup as it is staged and held in the order the B operands are read (one conflict-free
// ds_read_b128 per limb and 32 columns); the loads of the next chunk are in flight during the current
// one's products, one barrier per chunk. A slice streamed this way leaves room for two or more
// workgroups per CU, whose prologues and stores hide under each other's products, and costs the same
// for any K. D holds 32 columns of a row in 32 lanes: the stores are whole 128-byte lines.
//
// Every output of the staged kernel is the same sequence of products whatever the tile, slice and
// grid, so results do not depend on the launch shape or on the number of rows; launches small enough
// for the direct kernel below (rows_shape) sum K in four parts.
#pragma once
#include "common.h"

namespace face {

constexpr int kGemmRows = 32;                   // rows per wave
constexpr int kGemmK = 32;                      // k per staged chunk
constexpr int kGemmMaxProbs = 8;                // problems per launch
constexpr int kGemmMaxGroups = 64;              // scale-table rows (elements)
constexpr int64_t kGemmMaxLd = (int64_t)1 << 25; // row stride of the staged kernel: 31 rows within 32 bits of bytes

struct GemmProb {
    const float* x;
    int64_t ld_x, m;
    const float* w;
    int64_t ld_w;
    float* y;
    int64_t ld_y;
    int n, k, s_off, slices;               // slices of 32 NB columns
    float beta;
    const float* x2;                       // input columns k >= k1 (column k - k1), or x
    int64_t ld_x2;
    int k1, x_op;                          // x_op on columns < k1: 0 none, 1 silu, 2 * silu'(xz)
    const float* xz;
    int64_t ld_xz;
    const float* w2;                       // weights of the columns k >= k1 (w itself if not given)
    int64_t ld_w2;
    const float* bias;
    const float* bias_row;                 // per-row factor of the bias, or null
    const float* sum_row;                  // per-row factor of the sum before the bias, or null
    const float* y0;                       // initial sum beta * y0 (columns < n_y0), null: y
    int64_t ld_y0;
    int n_y0;
    int64_t first_block;                   // first work item of this problem
    int64_t w_off;                         // its split weights in the workspace (bytes)
    int turn0, turn1;                      // chunks of negated weights (see flip_sign)
};

// The matrix instruction cuts each addend, aligned to the largest of the sum, below 2^-8 of an ulp towards
// minus infinity, so a long sum drifts: its mean error over random operands was -1.1e-8 of the results' rms at
// K = 160 and -2.7e-8 at 512, the same sign in every output, which a sum over atoms collects (fp32
// instructions: none). Chunks [turn0, turn1) of 32 k therefore enter with negated weights into accumulators
// whose sign is turned before and after, so that two parts of the sum drift in opposite directions. A step of
// 16 k drifts as the accumulators grow, by the square root of its number, the first one 6.5 times the unit (its
// last product is larger than the sum so far), and all alike where the sum starts at y: turn_chunks (gemm.hip)
// puts half of the whole between the turns. What is left is about 1e-9 from K = 80 on, 3e-9 at 64, 5e-9 at 48;
// one chunk keeps its 7e-9.
__device__ __forceinline__ v4f flip_sign(v4f v, uint32_t sign) {
    return __builtin_bit_cast(v4f, __builtin_bit_cast(v4u, v) ^ sign);
}

// Logistic function (and one minus it) with the hardware exp2 and reciprocal, each corrected to first order:
// e = exp(-x) from the rounded exponent t and what its rounding and that of log2(e) left over, 1 / (1 + e) by
// one Newton step. Uncorrected, x < 0 came out 0.3 to 0.8 ulp too large on average (silu: mean -0.30 ulp,
// rms 0.90). |x| is cut at 80, where exp(-|x|) is 2e-35 and all intermediate values are finite.
__device__ __forceinline__ float gemm_sigmoid(float x, float& rest) {
    constexpr float kL = 0x1.715476p+0f, kLow = 0x1.4ae0cp-26f;           // log2(e) = kL + kLow
    const float a = __builtin_amdgcn_fmed3f(x, -80.f, 80.f), t = -kL * a;
    const float lo = fmaf(-kLow, a, fmaf(-kL, a, -t));
    float e = __builtin_amdgcn_exp2f(t);
    e = fmaf(e, 0.693147181f * lo, e);
    const float d = 1.f + e;
    float r = __builtin_amdgcn_rcpf(d);
    r = fmaf(fmaf(-d, r, 1.f), r, r);
    rest = e * r;
    return r;
}
__device__ __forceinline__ float gemm_op(float x, float z, int op) {
    float rest;
    if (op == 1) return x * gemm_sigmoid(x, rest);
    if (op == 2) {                                                     // x * d silu(z) / dz
        const float sg = gemm_sigmoid(z, rest);
        return x * (sg * fmaf(z, rest, 1.f));
    }
    return x;
}
__device__ __forceinline__ v4f gemm_op4(v4f x, v4f z, int op) {
    v4f o;
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = gemm_op(x[r], z[r], op);
    return o;
}

struct GemmArgs {
    GemmProb p[kGemmMaxProbs];
    int n_probs, w_kn;
    const float *xs, *ys;
    int ld_s, n_groups;
    const int32_t* group;
    int64_t period;
    int kmax, side_lds;                    // largest K; the scale tables fit in LDS
    int xcd_order;                         // items in XCD-contiguous ranges
    const char* work;                      // split weights (PS kernels), else null
};

// A uniform base and a 32-bit byte offset per lane: one scalar address pair per access.
__device__ __forceinline__ float* at_off(float* u, uint32_t bytes) {
    return reinterpret_cast<float*>(reinterpret_cast<char*>(u) + bytes);
}
__device__ __forceinline__ const float* at_off(const float* u, uint32_t bytes) {
    return reinterpret_cast<const float*>(reinterpret_cast<const char*>(u) + bytes);
}
__device__ __forceinline__ v4f ld4_off(const float* u, uint32_t bytes) { return ld4(at_off(u, bytes)); }

// LDS after the two weight buffers: the row groups of every wave (32 ints each), then the scale rows of the slice's columns (ys) and of the problem's inputs (xs).
static inline size_t gemm_lds(int NB, int NW, int64_t side_floats) {
    return (size_t)2 * NB * 6144 + 4 * ((size_t)NW * kGemmRows + (size_t)side_floats);
}

// One row of a problem in plain fp32 products, for operands that do not split: columns n0 .. n0 + ns by
// the lanes of a wave.
template <int XM>
__device__ __forceinline__ void plain_row(const GemmArgs& A, const GemmProb& P, int64_t r, int n0, int ns, int lane) {
    if (r >= P.m) return;
    const int64_t g = A.group ? A.group[r % A.period] : 0;
#pragma unroll 1
    for (int c = lane; c < ns; c += kWave) {
        float s = 0.f;
        if (P.beta != 0.f && n0 + c < P.n_y0)
            s = P.beta * (P.y0 ? P.y0[r * P.ld_y0 + n0 + c] : P.y[r * P.ld_y + n0 + c]);
#pragma unroll 1
        for (int k = 0; k < P.k; ++k) {
            const bool second = k >= P.k1;
            float x = second ? P.x2[r * P.ld_x2 + k - P.k1] : P.x[r * P.ld_x + k];
            if (XM == 1) x *= A.xs[g * A.ld_s + P.s_off + k];
            if (XM == 3 && !second) x = gemm_op(x, P.x_op == 2 ? P.xz[r * P.ld_xz + k] : 0.f, P.x_op);
            const float* w = second ? P.w2 : P.w;
            const int64_t ld = second ? P.ld_w2 : P.ld_w, kk = second ? k - P.k1 : k;
            s = fmaf(x, A.w_kn ? w[kk * ld + n0 + c] : w[(n0 + c) * ld + kk], s);
        }
        if (P.sum_row) s *= P.sum_row[r];
        if (P.bias) s = fmaf(P.bias_row ? P.bias_row[r] : 1.f, P.bias[n0 + c], s);
        if (A.ys) s *= A.ys[g * A.ld_s + P.s_off + n0 + c];
        P.y[r * P.ld_y + n0 + c] = s;
    }
}

// XM: input mode -- 0 plain, 1 the per-group x scale (xs), 2 split input (x2, w2) or y0, 3 these and the
// transform x_op
// PS: the weights come split from the workspace (split_weights_kernel)
//
// The loads ahead have no branches: past an edge (last chunk, last column, last row) they read the last
// valid place again, whose products are not formed or not stored. (With guarded loads the compiler
// waited for each before issuing the next.)
template <int NB, int NW, int XM, bool PS>
__global__ __launch_bounds__(NW * kWave, NB <= 2 ? 3 : 2) void rows_gemm_kernel(GemmArgs A) {
    constexpr bool XS = XM == 1, XO = XM >= 2, XF = XM == 3;
    constexpr int NSB = 32 * NB, NT = NW * kWave, BUF = NB * 6144;
    constexpr int WI = (NSB * 4 + NT - 1) / NT;               // (column, 8 k) items per thread and chunk
    constexpr int WU = PS ? (6 * NB + NW - 1) / NW : 2 * WI;  // 16-byte loads per thread and chunk
    extern __shared__ __attribute__((aligned(16))) char smem[];
    int* sgrp = reinterpret_cast<int*>(smem + 2 * BUF);
    float* sys = reinterpret_cast<float*>(sgrp + NW * kGemmRows);
    float* sxs = sys + (A.ys ? A.n_groups * NSB : 0);
    const int tid = threadIdx.x, lane = tid & (kWave - 1), j = lane & 31, hf = lane >> 5;
    const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
    // item -> (problem, row tile, column slice), slices fastest. In XCD order (workgroup b runs on
    // XCD b % 8) each XCD takes a contiguous range, so the slices of a tile read its rows from one L2.
    int it = blockIdx.x;
    if (A.xcd_order) {
        const int nbk = gridDim.x, xcd = it & 7, per = nbk >> 3, rem = nbk & 7;
        it = xcd * per + min(xcd, rem) + (it >> 3);
    }
    int pi = 0;
#pragma unroll 1
    for (int k = 1; k < A.n_probs; ++k)
        if (it >= A.p[k].first_block) pi = k;
    const GemmProb& P = A.p[pi];
    const int slices = P.slices, local = it - (int)P.first_block, tile = local / slices;
    const int K = P.k, N = P.n, k1 = P.k1, x_op = XF ? P.x_op : 0;
    const int n0 = (local - tile * slices) * NSB;
    const int ns = min(NSB, N - n0);                          // a multiple of 16
    const int ncb = (N + 31) >> 5;                            // 32-column blocks
    const int turn0 = P.turn0, turn1 = P.turn1;
    const int64_t M = P.m, m0 = ((int64_t)tile * NW + wv) * kGemmRows;
    const int64_t mb = min(m0, M - 1);                        // first row read (waves past m: the last row)
    const int jr = (int)min((int64_t)j, M - 1 - mb);          // this lane's input row - mb
    const int64_t ld_x = P.ld_x, ld_x2 = P.ld_x2, ld_xz = P.ld_xz;
    const float *xb = P.x + mb * ld_x, *x2b = P.x2 + mb * ld_x2, *xzb = P.xz + mb * ld_xz;
    const uint32_t xo = 4 * (uint32_t)(jr * (int)ld_x + 8 * hf), x2o = 4 * (uint32_t)(jr * (int)ld_x2 + 8 * hf);
    const uint32_t xzo = 4 * (uint32_t)(jr * (int)ld_xz + 8 * hf);
    const int grp = A.group ? A.group[(mb + jr) % A.period] : 0;
    const float *wsrc = P.w, *w2src = P.w2;
    const int64_t ld_w = P.ld_w, ld_w2 = P.ld_w2;
    const bool w_kn = A.w_kn != 0;
    const char* wwork = PS ? A.work + P.w_off + (int64_t)(n0 >> 5) * 3072 : nullptr;
    int woff[WU];                                             // of this wave's 1 KB pieces of a chunk
#pragma unroll
    for (int u = 0; u < WU; ++u) {
        const int f = min(wv + u * NW, 6 * NB - 1), s = f >= 3 * NB;
        woff[u] = s * ncb * 3072 + min(f - s * 3 * NB, 3 * (ncb - (n0 >> 5)) - 1) * 1024;
    }

    auto load_x = [&](int c, v4f (&xv)[4], v4f (&zv)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int k0 = min(kGemmK * c + 16 * s, K - 16);  // uniform
            const bool second = XO && k0 >= k1;
            const float* u = second ? x2b + (k0 - k1) : xb + k0;
            const uint32_t o = second ? x2o : xo;
            xv[2 * s] = ld4_off(u, o);
            xv[2 * s + 1] = ld4_off(u, o + 16);
            if (XF && x_op == 2 && !second) {
                zv[2 * s] = ld4_off(xzb + k0, xzo);
                zv[2 * s + 1] = ld4_off(xzb + k0, xzo + 16);
            }
        }
    };
    // weight item v of a chunk: 8 consecutive k (group kg) of one column; a wave's loads cover whole
    // lines (4 groups of 16 columns, or 32 columns of 8 rows of a (k, n) weight)
    auto item = [&](int u, int& col, int& kg) __attribute__((always_inline)) {
        const int v = min(u * NT + tid, NSB * 4 - 1);
        if (w_kn) col = 32 * (v >> 7) + (v & 31), kg = (v >> 5) & 3;
        else col = 16 * (v >> 6) + (v & 15), kg = (v >> 4) & 3;
    };
    // LDS image of a chunk: [16-k step][column block][limb][64 lanes] of 16 bytes
    auto load_w = [&](int c, v4f (&bw)[WU]) __attribute__((always_inline)) {
        if (PS) {
#pragma unroll
            for (int u = 0; u < WU; ++u)
                bw[u] = ld4_off(reinterpret_cast<const float*>(wwork + (int64_t)c * (ncb * 6144) + woff[u]), 16 * lane);
        } else if (w_kn) {
#pragma unroll
            for (int u = 0; u < WI; ++u) {
                int col, kg;
                item(u, col, kg);
                const int k = min(kGemmK * c + 8 * kg, K - 8);
                const bool second = XO && k >= k1;
                const int64_t ld = second ? ld_w2 : ld_w;
                const float* p = (second ? w2src + (k - k1) * ld : wsrc + k * ld) + n0 + min(col, ns - 1);
#pragma unroll
                for (int r = 0; r < 4; ++r) bw[2 * u][r] = p[r * ld];
#pragma unroll
                for (int r = 0; r < 4; ++r) bw[2 * u + 1][r] = p[(r + 4) * ld];
            }
        } else {
#pragma unroll
            for (int u = 0; u < WI; ++u) {
                int col, kg;
                item(u, col, kg);
                const int64_t k = min(kGemmK * c + 8 * kg, K - 8), f = n0 + min(col, ns - 1);
                const float* p = XO && k >= k1 ? w2src + f * ld_w2 + (k - k1) : wsrc + f * ld_w + k;
                bw[2 * u] = ld4(p);
                bw[2 * u + 1] = ld4(p + 4);
            }
        }
    };
    auto store_w = [&](int c, int buf, const v4f (&bw)[WU]) __attribute__((always_inline)) {
        if (PS) {
#pragma unroll
            for (int u = 0; u < WU; ++u)
                st4(reinterpret_cast<float*>(smem + buf * BUF + min(wv + u * NW, 6 * NB - 1) * 1024) + 4 * lane, bw[u]);
        } else {
#pragma unroll
            for (int u = 0; u < WI; ++u) {
                int col, kg;
                item(u, col, kg);
                const uint32_t sg = c >= turn0 && c < turn1 ? 0x80000000u : 0u;     // uniform
                const Split8 w = split8(flip_sign(bw[2 * u], sg), flip_sign(bw[2 * u + 1], sg));
                v8bf* d = reinterpret_cast<v8bf*>(smem + buf * BUF + ((kg >> 1) * NB + (col >> 5)) * 3072) + (kg & 1) * 32 +
                          (col & 31);
                d[0] = w.h;
                d[64] = w.m;
                d[128] = w.l;
            }
        }
    };

    v4f xn[4], zn[4], bw[WU];
    load_w(0, bw);
    load_x(0, xn, zn);
    if (hf == 0) sgrp[wv * kGemmRows + j] = grp;
    if (A.side_lds && A.ys) {
        for (int v = tid; v < A.n_groups * NSB; v += NT) {
            const int g = v / NSB, c = v - g * NSB;
            sys[v] = A.ys[(int64_t)g * A.ld_s + P.s_off + n0 + min(c, ns - 1)];
        }
    }
    if (XS && A.side_lds) {
        for (int v = tid; v < A.n_groups * K; v += NT) {
            const int g = v / K, k = v - g * K;
            sxs[g * A.kmax + k] = A.xs[(int64_t)g * A.ld_s + P.s_off + k];
        }
    }
    store_w(0, 0, bw);
    // output element (row 8 (r >> 2) + 4 hf + (r & 3), column 32 nb + j) of the wave: a uniform base per
    // (r, nb) and one byte offset per lane
    const int64_t ld_y = P.ld_y;
    float* yb = P.y + m0 * ld_y + n0;
    const uint32_t yo = 4 * (uint32_t)(4 * hf * (int)ld_y + j);
    const bool full = m0 + kGemmRows <= M;
    auto row_ok = [&](int r) __attribute__((always_inline)) { return m0 + 8 * (r >> 2) + (r & 3) + 4 * hf < M; };
    // beta y0 of a column block. A sum onto y starts there, its loads under the first x rows'; the forms with
    // an initial sum of their own (a residual, larger than what is added to it) add it after the products,
    // which then round at their own size (readout, d h: 3.5e-7 with the residual first, 0.7e-7).
    const float beta = P.beta;
    auto initial = [&](int nb, v16f& v) __attribute__((always_inline)) {
        const float* y0 = P.y0 ? P.y0 : P.y;
        const int64_t ld0 = P.y0 ? P.ld_y0 : ld_y;
        const float* y0b = y0 + m0 * ld0 + n0;
        const uint32_t o0 = 4 * (uint32_t)(4 * hf * (int)ld0 + j);
        const int n_y0 = min(P.n_y0 - n0, ns);
        if (full && 32 * nb + 32 <= n_y0) {                   // uniform
#pragma unroll
            for (int r = 0; r < 16; ++r) v[r] = beta * *at_off(y0b + (8 * (r >> 2) + (r & 3)) * ld0 + 32 * nb, o0);
        } else if (32 * nb < n_y0 && m0 < M) {
            const int64_t c = min(32 * nb + j, n_y0 - 1);
#pragma unroll
            for (int r = 0; r < 16; ++r) {                    // at the nearest valid place, zero outside
                const int64_t rr = min(m0 + 8 * (r >> 2) + (r & 3) + 4 * hf, M - 1);
                const float x = y0[rr * ld0 + n0 + c];
                v[r] = (32 * nb + j < n_y0 && row_ok(r)) ? beta * x : 0.f;
            }
        }
    };
    v16f acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[nb][r] = 0.f;
    if (!XO && beta != 0.f) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) initial(nb, acc[nb]);
    }
    __syncthreads();
    const int nchunk = (K + kGemmK - 1) / kGemmK;
#pragma unroll 1
    for (int c = 0, part = 0; part < 3; ++part) {
        const int end = part == 0 ? turn0 : (part == 1 ? turn1 : nchunk);
#pragma unroll 1
        for (; c < end; ++c) {
            const int buf = c & 1, cn = min(c + 1, nchunk - 1);
            load_w(cn, bw);
            Split8 xq[2];
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const int k0 = min(kGemmK * c + 16 * s, K - 16);
                v4f a = xn[2 * s], b = xn[2 * s + 1];
                if (XS) {
                    if (A.side_lds) {
                        a *= lds4_at(sxs, grp * A.kmax + k0 + 8 * hf);
                        b *= lds4_at(sxs, grp * A.kmax + k0 + 8 * hf + 4);
                    } else {
                        const float* t = A.xs + (int64_t)grp * A.ld_s + P.s_off + k0 + 8 * hf;
                        a *= ld4(t);
                        b *= ld4(t + 4);
                    }
                }
                if (XF && x_op && k0 < k1) {
                    a = gemm_op4(a, zn[2 * s], x_op);
                    b = gemm_op4(b, zn[2 * s + 1], x_op);
                }
                xq[s] = split8(a, b);
            }
            load_x(cn, xn, zn);
            __builtin_amdgcn_sched_barrier(0);                    // the loads ahead are issued before the products
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                if (s && kGemmK * c + 16 >= K) break;
                const v8bf* wf = reinterpret_cast<const v8bf*>(smem + buf * BUF + s * NB * 3072) + lane;
                const Split8& x = xq[s];
                // the limbs of the next column block are read ahead; the smallest products first
                v8bf w[3];
#pragma unroll
                for (int q = 0; q < 3; ++q) w[q] = wf[q * 64];
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    v8bf wn[3];
#pragma unroll
                    for (int q = 0; q < 3; ++q) wn[q] = nb + 1 < NB ? wf[(nb + 1) * 192 + q * 64] : w[q];
                    acc[nb] = mfma_32x32x16(x.l, w[0], acc[nb]);
                    acc[nb] = mfma_32x32x16(x.h, w[2], acc[nb]);
                    acc[nb] = mfma_32x32x16(x.m, w[1], acc[nb]);
                    acc[nb] = mfma_32x32x16(x.m, w[0], acc[nb]);
                    acc[nb] = mfma_32x32x16(x.h, w[1], acc[nb]);
                    acc[nb] = mfma_32x32x16(x.h, w[0], acc[nb]);
#pragma unroll
                    for (int q = 0; q < 3; ++q) w[q] = wn[q];
                }
                // issue order: the reads of blocks 0 and 1, then per block its products and the reads of the
                // block after the next one
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    if (nb == 0) __builtin_amdgcn_sched_group_barrier(0x100, NB > 1 ? 6 : 3, 0);
                    __builtin_amdgcn_sched_group_barrier(0x008, 6, 0);
                    if (nb + 2 < NB) __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
                }
            }
            store_w(cn, buf ^ 1, bw);
            __syncthreads();
        }
        if (part < 2) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[nb][r] = -acc[nb][r];
        }
    }
    // Operands that round to a bf16 infinity have a NaN limb, which every product they enter carries into
    // the sums: a row with a sum that is not finite is formed again in plain fp32 products (and not stored
    // below); the others of the wave keep theirs.
    float chk = 0.f;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int r = 0; r < 16; ++r) chk = fmaf(acc[nb][r], 0.f, chk);
    uint32_t redo = 0;                                        // rows of the tile, uniform
    if (__any(chk != chk)) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float c = 0.f;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) c = fmaf(acc[nb][r], 0.f, c);
            const uint64_t b = __ballot(c != c);
            const int row = 8 * (r >> 2) + (r & 3);
            redo |= ((uint32_t)b ? 1u : 0u) << row | ((b >> 32) ? 1u : 0u) << (row + 4);
        }
#pragma unroll 1
        for (int i = 0; i < kGemmRows; ++i)
            if (redo >> i & 1) plain_row<XM>(A, P, m0 + i, n0, ns, lane);
    }
    // epilogue: initial sum, bias and y scale, then stores of 128 bytes per row
    if (XO && beta != 0.f) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            v16f v;
#pragma unroll
            for (int r = 0; r < 16; ++r) v[r] = 0.f;
            initial(nb, v);
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[nb][r] += v[r];
        }
    }
    if (XF && P.sum_row) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float f = P.sum_row[min(m0 + 8 * (r >> 2) + (r & 3) + 4 * hf, M - 1)];
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) acc[nb][r] *= f;
        }
    }
    if (P.bias) {
        const float* br = P.bias_row;
        float f[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) f[r] = br ? br[min(m0 + 8 * (r >> 2) + (r & 3) + 4 * hf, M - 1)] : 1.f;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            const float b = P.bias[n0 + min(32 * nb + j, ns - 1)];
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[nb][r] = fmaf(f[r], b, acc[nb][r]);
        }
    }
    if (A.ys) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int g = sgrp[wv * kGemmRows + 8 * (r >> 2) + 4 * hf + (r & 3)];
            if (A.side_lds) {
                const float* t = sys + g * NSB + j;
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) acc[nb][r] *= t[32 * nb];
            } else {
                const float* t = A.ys + (int64_t)g * A.ld_s + P.s_off + n0;
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) acc[nb][r] *= t[min(32 * nb + j, ns - 1)];
            }
        }
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        if (full && !redo && 32 * nb + 32 <= ns) {            // uniform
#pragma unroll
            for (int r = 0; r < 16; ++r) *at_off(yb + (8 * (r >> 2) + (r & 3)) * ld_y + 32 * nb, yo) = acc[nb][r];
        } else {
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (32 * nb + j < ns && row_ok(r) && !(redo >> (8 * (r >> 2) + (r & 3) + 4 * hf) & 1))
                    *at_off(yb + (8 * (r >> 2) + (r & 3)) * ld_y + 32 * nb, yo) = acc[nb][r];
        }
    }
}

// Small launches: no staging. Each wave loads its columns' weights straight into its B operands (lane
// j + 32 h: 8 consecutive k of column j), splits them itself and runs D steps of 16 k ahead, without LDS
// or barriers in the loop; the four waves of a workgroup share a 32-row tile, each a contiguous
// part of K, and add their sums through LDS in wave order. What bounds these launches is the chain of a
// wave -- split, products that wait for each other, 0.4 us per 16 k with one wave per SIMD -- times the
// length of K, not the products or the memory: a quarter of K per wave takes 21 rows of 864 -> 192 from 22 us
// (staged) to 9.1, and 1,344 rows from 22 to 11.5.
constexpr int kDirectWaves = 4;
template <int NB, int XM>
__global__ __launch_bounds__(kDirectWaves * kWave, 2) void rows_gemm_direct_kernel(GemmArgs A) {
    constexpr bool XS = XM == 1, XO = XM >= 2, XF = XM == 3;
    constexpr int NSB = 32 * NB, D = 3, KW = kDirectWaves, NR = 16 / KW;
    __shared__ float ssum[KW * NB * 16 * kWave];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), j = lane & 31, hf = lane >> 5;
    const int kp = __builtin_amdgcn_readfirstlane(tid / kWave), it = blockIdx.x;
    int pi = 0;
#pragma unroll 1
    for (int k = 1; k < A.n_probs; ++k)
        if (it >= A.p[k].first_block) pi = k;
    const GemmProb& P = A.p[pi];
    const int slices = P.slices, local = it - (int)P.first_block, tile = local / slices;
    const int K = P.k, N = P.n, k1 = P.k1, x_op = XF ? P.x_op : 0, nk = K >> 4;
    const int n0 = (local - tile * slices) * NSB, ns = min(NSB, N - n0);
    const int64_t M = P.m, m0 = (int64_t)tile * kGemmRows;
    const int64_t row = min(m0 + j, M - 1);
    const float *xr = P.x + row * P.ld_x + 8 * hf, *x2r = P.x2 + row * P.ld_x2 + 8 * hf;
    const float* xzr = P.xz + row * P.ld_xz + 8 * hf;
    const int grp = A.group ? A.group[row % A.period] : 0;
    const float* xsr = XS ? A.xs + (int64_t)grp * A.ld_s + P.s_off + 8 * hf : nullptr;
    const bool w_kn = A.w_kn != 0;
    const int64_t ld_w = P.ld_w, ld_w2 = P.ld_w2;
    int64_t wo[NB], wo2[NB];                                  // this lane's column (and k half) in w and w2
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const int64_t f = n0 + min(32 * nb + j, ns - 1);
        wo[nb] = w_kn ? 8 * hf * ld_w + f : f * ld_w + 8 * hf;
        wo2[nb] = w_kn ? 8 * hf * ld_w2 + f : f * ld_w2 + 8 * hf;
    }
    struct Step {
        v4f x[2], z[2], s[2], w[NB][2];
    };
    auto load = [&](int st, Step& b) __attribute__((always_inline)) {
        const int k0 = 16 * min(st, nk - 1);                  // uniform
        const bool second = XO && k0 >= k1;
        const float* p = second ? x2r + (k0 - k1) : xr + k0;
        b.x[0] = ld4(p);
        b.x[1] = ld4(p + 4);
        if (XF && x_op == 2 && !second) {
            b.z[0] = ld4(xzr + k0);
            b.z[1] = ld4(xzr + k0 + 4);
        }
        if (XS) {
            b.s[0] = ld4(xsr + k0);
            b.s[1] = ld4(xsr + k0 + 4);
        }
        const float* w = second ? P.w2 : P.w;
        const int64_t ld = second ? ld_w2 : ld_w, kk = second ? k0 - k1 : k0;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            const float* q = w + (second ? wo2[nb] : wo[nb]) + (w_kn ? kk * ld : kk);
            if (w_kn) {
#pragma unroll
                for (int r = 0; r < 8; ++r) b.w[nb][r >> 2][r & 3] = q[r * ld];
            } else {
                b.w[nb][0] = ld4(q);
                b.w[nb][1] = ld4(q + 4);
            }
        }
    };
    const int s0 = nk * kp / KW, s1 = nk * (kp + 1) / KW;
    const uint32_t sg = kp == 1 || kp == 2 ? 0x80000000u : 0u;   // the middle parts drift the other way (see flip_sign)
    Step b[D];
#pragma unroll
    for (int d = 0; d < D; ++d) load(s0 + d, b[d]);
    v16f acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[nb][r] = 0.f;
    const float beta = P.beta;
    const float* y0 = P.y0 ? P.y0 : P.y;
    const int64_t ld_y = P.ld_y, ld0 = P.y0 ? P.ld_y0 : ld_y;
    auto out_row = [&](int r) __attribute__((always_inline)) { return m0 + 8 * (r >> 2) + (r & 3) + 4 * hf; };
    const int n_y0 = min(P.n_y0 - n0, ns);
    if (!XO && beta != 0.f && kp == 0) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            if (32 * nb >= n_y0) break;
            const int64_t c = n0 + min(32 * nb + j, n_y0 - 1);
#pragma unroll
            for (int r = 0; r < 16; ++r) {                    // at the nearest valid place, zero outside
                const float v = y0[min(out_row(r), M - 1) * ld0 + c];
                acc[nb][r] = (32 * nb + j < n_y0 && out_row(r) < M) ? beta * v : 0.f;
            }
        }
    }
    for (int st = s0; st < s1; st += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            if (st + d >= s1) break;                          // uniform
            Step& c = b[d];
            if (XS) c.x[0] *= c.s[0], c.x[1] *= c.s[1];
            if (XF && x_op && 16 * (st + d) < k1) {
                c.x[0] = gemm_op4(c.x[0], c.z[0], x_op);
                c.x[1] = gemm_op4(c.x[1], c.z[1], x_op);
            }
            const Split8 x = split8(flip_sign(c.x[0], sg), flip_sign(c.x[1], sg));
            Split8 w[NB];
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) w[nb] = split8(c.w[nb][0], c.w[nb][1]);
            load(st + d + D, c);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) acc[nb] = mfma_32x32x16(x.l, w[nb].h, acc[nb]);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) acc[nb] = mfma_32x32x16(x.h, w[nb].l, acc[nb]);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) acc[nb] = mfma_32x32x16(x.m, w[nb].m, acc[nb]);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) acc[nb] = mfma_32x32x16(x.m, w[nb].h, acc[nb]);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) acc[nb] = mfma_32x32x16(x.h, w[nb].m, acc[nb]);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) acc[nb] = mfma_32x32x16(x.h, w[nb].h, acc[nb]);
        }
    }
    // the NR accumulator registers this wave finishes, of rows out_row(NR kp + i)
    const int rb = NR * kp;
    float v[NB][NR];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int r = 0; r < 16; ++r) ssum[((kp * NB + nb) * 16 + r) * kWave + lane] = acc[nb][r];
    __syncthreads();
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            v[nb][i] = ssum[(nb * 16 + rb + i) * kWave + lane];
#pragma unroll
            for (int k = 1; k < KW; ++k) {
                const float p = ssum[((k * NB + nb) * 16 + rb + i) * kWave + lane];
                v[nb][i] += k == 1 || k == 2 ? -p : p;
            }
        }
    if (XO && beta != 0.f) {                                  // after the products, as in the staged kernel
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            if (32 * nb >= n_y0) break;
            const int64_t c = n0 + min(32 * nb + j, n_y0 - 1);
#pragma unroll
            for (int i = 0; i < NR; ++i) {
                const float x = y0[min(out_row(rb + i), M - 1) * ld0 + c];
                v[nb][i] += (32 * nb + j < n_y0 && out_row(rb + i) < M) ? beta * x : 0.f;
            }
        }
    }
    uint32_t redo = 0;                                        // rows formed again, as in the staged kernel: bits i, i + 16
#pragma unroll
    for (int i = 0; i < NR; ++i) {
        float c = 0.f;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) c = fmaf(v[nb][i], 0.f, c);
        const uint64_t b = __ballot(c != c);
        redo |= ((uint32_t)b ? 1u : 0u) << i | ((b >> 32) ? 1u : 0u) << (i + 16);
    }
    if (redo) {
#pragma unroll 1
        for (int i = 0; i < 2 * NR; ++i)
            if (redo >> ((i >> 1) + 16 * (i & 1)) & 1)
                plain_row<XM>(A, P, m0 + 8 * ((rb + (i >> 1)) >> 2) + ((rb + (i >> 1)) & 3) + 4 * (i & 1), n0, ns, lane);
    }
#pragma unroll
    for (int i = 0; i < NR; ++i) {
        const int64_t r = out_row(rb + i), rc = min(r, M - 1);
        const float f = P.bias_row ? P.bias_row[rc] : 1.f, sr = XF && P.sum_row ? P.sum_row[rc] : 1.f;
        const float* t = A.ys ? A.ys + (int64_t)A.group[rc % A.period] * A.ld_s + P.s_off + n0 : nullptr;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            const int c = min(32 * nb + j, ns - 1);
            float o = v[nb][i];
            if (XF && P.sum_row) o *= sr;
            if (P.bias) o = fmaf(f, P.bias[n0 + c], o);
            if (A.ys) o *= t[c];
            if (32 * nb + j < ns && r < M && !(redo >> (i + 16 * hf) & 1)) P.y[r * ld_y + n0 + c] = o;
        }
    }
}

// Splits the weights of a launch once: one wave per 16 k x 32 columns writes the three limbs in the
// order of the LDS image, [16-k step][column block][limb][64 lanes] of 16 bytes, zeros past the last
// column and step (an even number of steps). Launched before rows_gemm_kernel where many row tiles would each split them again.
__global__ __launch_bounds__(kWave) inline void split_weights_kernel(GemmArgs A, char* work) {
    int pi = 0;
    const int64_t it = blockIdx.x;
#pragma unroll 1
    for (int k = 1; k < A.n_probs; ++k)
        if (it >= A.p[k].first_block) pi = k;
    const GemmProb& P = A.p[pi];
    const int lane = threadIdx.x, ncb = (P.n + 31) >> 5;
    const int64_t local = it - P.first_block;
    const int step = (int)(local / ncb), cb = (int)(local - (int64_t)step * ncb);
    const int col = 32 * cb + (lane & 31), k = 16 * step + 8 * (lane >> 5);
    v4f a = {0.f, 0.f, 0.f, 0.f}, b = a;
    if (col < P.n && k < P.k) {
        const bool second = k >= P.k1;
        const float* w = second ? P.w2 : P.w;
        const int64_t ld = second ? P.ld_w2 : P.ld_w, kk = second ? k - P.k1 : k;
        if (A.w_kn) {
            const float* p = w + kk * ld + col;
#pragma unroll
            for (int r = 0; r < 4; ++r) a[r] = p[r * ld], b[r] = p[(r + 4) * ld];
        } else {
            const float* p = w + col * ld + kk;
            a = ld4(p);
            b = ld4(p + 4);
        }
    }
    const uint32_t sg = (step >> 1) >= P.turn0 && (step >> 1) < P.turn1 ? 0x80000000u : 0u;
    const Split8 w = split8(flip_sign(a, sg), flip_sign(b, sg));
    v8bf* d = reinterpret_cast<v8bf*>(work + P.w_off + local * 3072) + lane;
    d[0] = w.h;
    d[64] = w.m;
    d[128] = w.l;
}

// Launch shape: NB column blocks of 32 per wave, NW waves per workgroup; direct: the direct kernel (four waves).
struct RowsShape {
    int NW, NB, xcd;
    bool direct;
};

// Everything a launch needs but its shape.
struct RowsCtx {
    GemmArgs A;                                  // problems filled, tiling not yet
    const face_lin_problem* probs;
    int n_probs, K, n_widest, max_lds, n_cu, n_groups;
    bool x_scale, y_scale, any_ext, any_op;
    bool far;                                    // a row stride past kGemmMaxLd
    char* work;                                  // workspace for split weights, or null
    hipStream_t st;
};

// One launch of a shape; FACE_ERR_UNSUPPORTED, before anything is launched, if there is no such kernel.
template <int XM>
static int launch_rows_xm(const RowsCtx& c, RowsShape S) {
    if (S.NB < 1 || S.NB > 16 || (S.direct && c.work) || (!S.direct && c.far)) return FACE_ERR_UNSUPPORTED;
    GemmArgs A = c.A;
    A.xcd_order = S.xcd;
    A.work = c.work;
    const int waves = S.direct ? kDirectWaves : S.NW, rows = S.direct ? kGemmRows : kGemmRows * S.NW;
    int64_t blocks = 0;
    for (int i = 0; i < c.n_probs; ++i) {
        const face_lin_problem& s = c.probs[i];
        GemmProb& p = A.p[i];
        p.slices = (s.n + 32 * S.NB - 1) / (32 * S.NB);
        p.first_block = blocks;
        blocks += (s.m + rows - 1) / rows * p.slices;
    }
    if (blocks == 0) return 0;
    if (blocks > INT32_MAX) return FACE_ERR_UNSUPPORTED;
    size_t lds = 0;
    if (!S.direct) {
        const int64_t side = (c.y_scale ? (int64_t)c.n_groups * 32 * S.NB : 0) + (c.x_scale ? (int64_t)c.n_groups * c.K : 0);
        A.side_lds = gemm_lds(S.NB, S.NW, side) <= (size_t)c.max_lds;
        lds = gemm_lds(S.NB, S.NW, A.side_lds ? side : 0);
    }
    auto go = [&](auto kern) -> int {
        if (lds > 65536 &&
            hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
            return FACE_ERR_UNSUPPORTED;
        hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(waves * kWave), lds, c.st, A);
        FACE_LAUNCH_CHECK();
        return 0;
    };
    if (S.direct) {
        if (S.NB > 2) return FACE_ERR_UNSUPPORTED;
        return S.NB == 1 ? go(rows_gemm_direct_kernel<1, XM>) : go(rows_gemm_direct_kernel<2, XM>);
    }
    const int NW = S.NW;
    if (c.work) {
        switch (S.NB) {
            case 2: return NW == 4 ? go(rows_gemm_kernel<2, 4, XM, true>) : FACE_ERR_UNSUPPORTED;
            case 3: return NW == 4 ? go(rows_gemm_kernel<3, 4, XM, true>) : FACE_ERR_UNSUPPORTED;
            case 4: return NW == 4 ? go(rows_gemm_kernel<4, 4, XM, true>) : FACE_ERR_UNSUPPORTED;
            case 5: return NW == 4 ? go(rows_gemm_kernel<5, 4, XM, true>) : FACE_ERR_UNSUPPORTED;
            case 6: return NW == 4 ? go(rows_gemm_kernel<6, 4, XM, true>) : FACE_ERR_UNSUPPORTED;
            case 8: return NW == 8 ? go(rows_gemm_kernel<8, 8, XM, true>) : FACE_ERR_UNSUPPORTED;
            default: return FACE_ERR_UNSUPPORTED;
        }
    }
    switch (NW == 4 || NW == 8 ? 16 * NW + S.NB : 0) {
        case 65: return go(rows_gemm_kernel<1, 4, XM, false>);
        case 66: return go(rows_gemm_kernel<2, 4, XM, false>);
        case 67: return go(rows_gemm_kernel<3, 4, XM, false>);
        case 68: return go(rows_gemm_kernel<4, 4, XM, false>);
        case 69: return go(rows_gemm_kernel<5, 4, XM, false>);
        case 129: return go(rows_gemm_kernel<1, 8, XM, false>);
        case 130: return go(rows_gemm_kernel<2, 8, XM, false>);
        case 131: return go(rows_gemm_kernel<3, 8, XM, false>);
        case 132: return go(rows_gemm_kernel<4, 8, XM, false>);
        case 133: return go(rows_gemm_kernel<5, 8, XM, false>);
        default: return FACE_ERR_UNSUPPORTED;
    }
}

// The input modes' launches, one translation unit each (gemm.hip, gemm_xs.hip, gemm_split.hip, gemm_op.hip).
int launch_rows_plain(const RowsCtx& c, RowsShape S);
int launch_rows_xs(const RowsCtx& c, RowsShape S);
int launch_rows_split(const RowsCtx& c, RowsShape S);
int launch_rows_op(const RowsCtx& c, RowsShape S);

}  // namespace face
