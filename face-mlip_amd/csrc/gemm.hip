// face_rows_linear: argument checks, launch shapes and the plain input mode of the row-block linear
// layers (rows_gemm.h).
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>

#include "rows_gemm.h"

namespace face {

int launch_rows_plain(const RowsCtx& c, RowsShape S) { return launch_rows_xm<0>(c, S); }

static bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace face

using namespace face;

// The chunks of negated weights of a sum over K (rows_gemm.h): of the starts in the first half, the one that
// comes nearest to half of the drift between the turns.
static void turn_chunks(GemmProb& p, bool onto_y) {
    constexpr int kMax = 128;
    const int nk = p.k / 16, nc = (nk + 1) / 2;
    p.turn0 = p.turn1 = nc;
    if (nc < 2) return;
    if (nc > kMax) {
        p.turn0 = nc / 5, p.turn1 = p.turn0 + nc / 2;
        return;
    }
    float sum[kMax + 1];                                       // drift of the first c chunks
    sum[0] = 0.f;
    for (int c = 0, st = 0; c < nc; ++c) {
        float d = 0.f;
        for (; st < nk && st < 2 * c + 2; ++st) d += onto_y ? 1.f : (st == 0 ? 6.5f : std::sqrt((float)(st + 1)));
        sum[c + 1] = sum[c] + d;
    }
    float best = 1e30f;
    for (int a = 1, b = 1; a <= (nc + 1) / 2; ++a) {
        auto off = [&](int e) { return std::fabs(2.f * (sum[e] - sum[a]) - sum[nc]); };
        b = std::max(a, b);
        while (b < nc && off(b + 1) <= off(b)) ++b;
        if (off(b) < 0.999f * best) best = off(b), p.turn0 = a, p.turn1 = b;
    }
}

// Validate problem s and fill p (everything but the tiling); 0 or a FACE_ERR_* status.
static int fill_prob(const face_lin_problem& s, int w_kn, bool scaled, const float* x_scale, const float* y_scale,
                     int ld_scale, GemmProb& p) {
    if (s.m < 0 || s.n < 16 || s.n % 16 || s.k < 16 || s.k % 16 || s.ld_y < s.n || s.ld_w < (w_kn ? s.n : (s.w2 ? s.k1 : s.k)))
        return FACE_ERR_ARG;
    const int k1 = s.x2 ? s.k1 : s.k;
    if (k1 < 0 || k1 > s.k || k1 % 16 || (s.ld_x < k1 && s.ld_x != 0) || (s.x2 && s.ld_x2 < s.k - k1)) return FACE_ERR_ARG;
    if (s.x_op < 0 || s.x_op > 2 || (s.x_op == 2 && (!s.xz || s.ld_xz < k1)) || (s.x_op && x_scale)) return FACE_ERR_ARG;
    if (s.w2 && (!s.x2 || s.ld_w2 < (w_kn ? s.n : s.k - k1))) return FACE_ERR_ARG;
    if (s.bias_row && !s.bias) return FACE_ERR_ARG;
    if (s.y0 && (s.n_y0 < 0 || s.n_y0 > s.n || s.n_y0 % 4 || s.ld_y0 < s.n_y0)) return FACE_ERR_ARG;
    if (scaled && (s.s_off < 0 || s.s_off % 4 || s.s_off + (x_scale ? s.k : 0) > ld_scale ||
                   s.s_off + (y_scale ? s.n : 0) > ld_scale))
        return FACE_ERR_ARG;
    if (s.m > 0 && (!s.x || !s.w || !s.y)) return FACE_ERR_ARG;
    // the contract's bound on operand sizes
    const int64_t lim = (int64_t)1 << 31;
    if (s.m * s.ld_x >= lim || s.m * s.ld_y >= lim || (s.x2 && s.m * s.ld_x2 >= lim) ||
        (s.x_op == 2 && s.m * s.ld_xz >= lim) || (s.y0 && s.m * s.ld_y0 >= lim))
        return FACE_ERR_UNSUPPORTED;
    if (s.ld_x % 4 || s.ld_y % 4 || !al16(s.x) || !al16(s.y) || (!w_kn && (!al16(s.w) || s.ld_w % 4)) ||
        (s.w2 && !w_kn && (!al16(s.w2) || s.ld_w2 % 4)) ||
        (s.x2 && (!al16(s.x2) || s.ld_x2 % 4)) || (s.x_op == 2 && (!al16(s.xz) || s.ld_xz % 4)) ||
        (s.y0 && (!al16(s.y0) || s.ld_y0 % 4)))
        return FACE_ERR_UNSUPPORTED;
    p.x = s.x, p.ld_x = s.ld_x, p.m = s.m, p.w = s.w, p.ld_w = s.ld_w, p.y = s.y, p.ld_y = s.ld_y, p.n = s.n;
    p.k = s.k, p.s_off = s.s_off, p.beta = s.beta;
    p.x2 = s.x2 ? s.x2 : s.x, p.ld_x2 = s.x2 ? s.ld_x2 : s.ld_x, p.k1 = k1;
    p.x_op = s.x_op, p.xz = s.x_op == 2 ? s.xz : s.x, p.ld_xz = s.x_op == 2 ? s.ld_xz : s.ld_x;
    p.w2 = s.w2 ? s.w2 : (w_kn ? s.w + (int64_t)k1 * s.ld_w : s.w + k1), p.ld_w2 = s.w2 ? s.ld_w2 : s.ld_w;
    p.bias = s.bias, p.bias_row = s.bias_row, p.sum_row = s.sum_row;
    p.y0 = s.y0, p.ld_y0 = s.y0 ? s.ld_y0 : 0, p.n_y0 = s.y0 ? s.n_y0 : s.n;
    return 0;
}

static int launch_rows(const RowsCtx& c, RowsShape S) {
    if (c.x_scale) return launch_rows_xs(c, S);
    if (c.any_op) return launch_rows_op(c, S);
    return c.any_ext ? launch_rows_split(c, S) : launch_rows_plain(c, S);
}

// Launch shape by size: the block count NB with the least estimated time. A workgroup's time is taken
// as (NB + 0.6) K -- its products, and the split of its rows worth 0.6 of a block (480,000 rows of
// 160 -> 160: 200 us with five blocks, 245 with three and 288 with two, both of which cover 192 columns)
// -- plus a prologue and epilogue worth 64 k; two workgroups on one CU run 1.5 times as much as one.
// Long launches fill the chip with any NB, so the widest slices without padding win (24,000 atoms,
// proj: 668 us with NB = 5, 765 with 4; C = 256: 1498 us with 8, 1624 with 6, 1634 with 4); short
// ones need a workgroup for every CU (864 atoms, 512 -> 96: 27 us with NB = 1, 35 with 3).
// Eight waves share a weight slice where it comes split ahead and 256 columns wide, or is split in the
// kernel from a (k, n) weight by a launch that has a workgroup for every CU anyway (216,000 rows of
// 160 -> 512: 267 against 276 us); else four (the same launch of 160 columns: 212 against 218 us).
// The XCD order pays only where several slices share rows (proj 668 against 680 us; K = 480 -> 160 of
// one slice 419 against 364 us: the plain order spreads neighbouring rows over the XCDs' channels).
// The direct kernel (K in four parts) takes launches of at most one workgroup per CU: 21 atoms, 512 -> 96
// 8.9 against 16.4 us staged, 192 -> 192 5.2 against 7.5; 1,344 rows of 864 -> 192 (252 workgroups) 11.5
// against 22, but 3,000 rows (564) 27 against 22. Two column blocks per wave where that brings a launch
// of long K under the limit (4,000 rows of 512 -> 96: 13.3 against 16.6).
// Row strides past kGemmMaxLd (at most 63 rows of them: an operand has fewer than 2^31 elements) take the
// direct kernel at any number of problems; its addresses are 64 bits wide.
static RowsShape rows_shape(const RowsCtx& c) {
    if (c.far) return {kDirectWaves, 1, 0, true};
    int NW = 4, NB = 2;
    for (int nb = 1; nb <= (c.K >= 384 ? 2 : 1) && !c.work; ++nb) {
        int64_t w = 0;
        for (int k = 0; k < c.n_probs; ++k)
            w += (c.probs[k].m + kGemmRows - 1) / kGemmRows * ((c.probs[k].n + 32 * nb - 1) / (32 * nb));
        if (w <= c.n_cu) return {kDirectWaves, nb, 0, true};
    }
    static constexpr int kSplitAhead[] = {8, 6, 5, 4, 3, 2}, kInKernel[] = {5, 4, 3, 2, 1};
    double best = 1e300;
    for (int i = 0; i < (c.work ? 6 : 5); ++i) {
        const int nb = c.work ? kSplitAhead[i] : kInKernel[i], nw = nb == 8 ? 8 : 4;
        double wgs = 0, cost = 0;
        for (int k = 0; k < c.n_probs; ++k) {
            const face_lin_problem& s = c.probs[k];
            const double w = (double)((s.m + kGemmRows * nw - 1) / (kGemmRows * nw)) * ((s.n + 32 * nb - 1) / (32 * nb));
            wgs += w * (nw / 4);                               // in four-wave workgroups
            cost += w * (nw / 4) * (nb + 0.6) * (s.k + 64);
        }
        if (wgs == 0) continue;
        const double one = cost / wgs, rounds = wgs / (2 * c.n_cu);
        const double t = wgs <= c.n_cu ? one : 1.3 * one * (rounds < 4 ? ceil(rounds) : rounds + 0.5);
        if (t < 0.999 * best) best = t, NB = nb, NW = nw;
    }
    if (!c.work && c.A.w_kn) {
        int64_t w8 = 0;
        for (int k = 0; k < c.n_probs; ++k)
            w8 += (c.probs[k].m + kGemmRows * 8 - 1) / (kGemmRows * 8) * ((c.probs[k].n + 32 * NB - 1) / (32 * NB));
        if (w8 >= 2 * c.n_cu) NW = 8;
    }
    return {NW, NB, c.n_widest > 32 * NB, false};
}

// Workspace: the limbs of every problem, 3 KB per 16 k x 32 columns, for an even number of 16-k steps. A
// problem of no rows has none (its pointers may be NULL).
static int64_t work_blocks(const face_lin_problem& s) {
    return s.m > 0 ? (int64_t)((s.k + 31) / 32 * 2) * ((s.n + 31) / 32) : 0;
}
static int64_t work_layout(const face_lin_problem* probs, int n_probs, GemmProb* p) {
    int64_t bytes = 0;
    for (int i = 0; i < n_probs; ++i) {
        if (p) p[i].w_off = bytes;
        bytes += work_blocks(probs[i]) * 3072;
    }
    return bytes;
}

extern "C" int64_t face_rows_linear_work(const face_lin_problem* probs, int32_t n_probs) {
    if (!probs || n_probs < 1 || n_probs > kGemmMaxProbs) return 0;
    for (int i = 0; i < n_probs; ++i)
        if (probs[i].n < 16 || probs[i].k < 16 || probs[i].m < 0) return 0;
    // Splitting ahead is a launch of its own (4 us) that takes 5-10 % off the products of long ones
    // (24,000 atoms: mix 212 -> 200 us, proj 745 -> 668, 160 -> 512 267 -> 239; 4,000 atoms: proj
    // 120 -> 112 us at 20 GFLOP, mix 44 -> 44 at 4 GFLOP): from 12 GFLOP on.
    double flops = 0;
    for (int i = 0; i < n_probs; ++i) flops += 2.0 * probs[i].m * probs[i].n * probs[i].k;
    const int64_t bytes = work_layout(probs, n_probs, nullptr);
    return flops >= 1.2e10 && bytes < ((int64_t)1 << 30) ? bytes : 0;
}

extern "C" int face_rows_linear(const face_lin_problem* probs, int32_t n_probs, int32_t w_kn, const float* x_scale,
                                const float* y_scale, int32_t ld_scale, int32_t n_groups, const int32_t* group,
                                int64_t period, void* stream) {
    return face_rows_linear_ws(probs, n_probs, w_kn, x_scale, y_scale, ld_scale, n_groups, group, period, nullptr, 0,
                               stream);
}

extern "C" int face_rows_linear_ws(const face_lin_problem* probs, int32_t n_probs, int32_t w_kn, const float* x_scale,
                                const float* y_scale, int32_t ld_scale, int32_t n_groups, const int32_t* group,
                                int64_t period, void* work, int64_t work_bytes, void* stream) {
    if (!probs || n_probs < 1 || n_probs > kGemmMaxProbs) return FACE_ERR_ARG;
    int K = 16, n_widest = 16;
    bool any_ext = false, any_op = false;
    for (int i = 0; i < n_probs; ++i) {
        if (probs[i].k < 16 || probs[i].k % 16) return FACE_ERR_ARG;
        if (probs[i].k > K) K = probs[i].k;
        if (probs[i].n > n_widest) n_widest = probs[i].n;
        if (probs[i].x_op || probs[i].sum_row) any_op = true;
        if (probs[i].x_op || probs[i].sum_row || probs[i].x2 || probs[i].y0) any_ext = true;
    }
    const bool scaled = x_scale || y_scale;
    if (scaled && (!group || period < 1 || ld_scale < 1 || n_groups < 1 || n_groups > kGemmMaxGroups))
        return FACE_ERR_ARG;
    if (!scaled) n_groups = 1;
    if ((x_scale && !al16(x_scale)) || (y_scale && !al16(y_scale)) || (scaled && ld_scale % 4))
        return FACE_ERR_UNSUPPORTED;
    RowsCtx c{};
    GemmArgs& A = c.A;
    A.n_probs = n_probs, A.w_kn = w_kn ? 1 : 0, A.xs = x_scale, A.ys = y_scale;
    A.ld_s = ld_scale, A.n_groups = n_groups, A.group = scaled ? group : nullptr, A.period = period, A.kmax = K;
    for (int i = 0; i < n_probs; ++i) {
        const int st = fill_prob(probs[i], A.w_kn, scaled, x_scale, y_scale, ld_scale, A.p[i]);
        if (st) return st;
    }
    if (x_scale && any_ext) return FACE_ERR_UNSUPPORTED;                 // x scale with split / op / y0
    for (int i = 0; i < n_probs; ++i) turn_chunks(A.p[i], A.p[i].beta != 0.f && !any_ext);
    c.probs = probs, c.n_probs = n_probs, c.K = K, c.n_widest = n_widest, c.max_lds = device_max_lds();
    c.n_cu = device_cu_count(), c.x_scale = x_scale != nullptr, c.y_scale = y_scale != nullptr, c.any_ext = any_ext;
    c.any_op = any_op;
    for (int i = 0; i < n_probs; ++i)
        for (const int64_t ld : {A.p[i].ld_x, A.p[i].ld_x2, A.p[i].ld_xz, A.p[i].ld_y, A.p[i].ld_y0})
            c.far = c.far || ld > kGemmMaxLd;
    c.n_groups = n_groups, c.st = (hipStream_t)stream;
    if (work && (((uintptr_t)work & 255) || work_layout(probs, n_probs, A.p) > work_bytes)) return FACE_ERR_ARG;
    if (work && !c.far) {
        int64_t blocks = 0;
        for (int i = 0; i < n_probs; ++i) {
            A.p[i].first_block = blocks;
            blocks += work_blocks(probs[i]);
        }
        c.work = (char*)work;
        if (blocks == 0) return 0;                               // no rows at all
        hipLaunchKernelGGL(split_weights_kernel, dim3((unsigned)blocks), dim3(kWave), 0, c.st, A, c.work);
        FACE_LAUNCH_CHECK();
    }
    // FACE_GEMM_SHAPE="nw,n_sl,xcd" forces one launch shape (nw = -4: the direct kernel), for tests that compare every
    // shape's results (split ahead where there is such a kernel); FACE_ERR_UNSUPPORTED if there is none
    if (const char* fs = getenv("FACE_GEMM_SHAPE")) {
        int nw = 0, ns = 0, xcd = 0;
        if (sscanf(fs, "%d,%d,%d", &nw, &ns, &xcd) == 3 && ns > 0) {
            const int nb = ((n_widest + ns - 1) / ns + 31) / 32;
            const RowsShape S{nw < 0 ? kDirectWaves : nw, nb, xcd ? 1 : 0, nw < 0};
            const int rc = launch_rows(c, S);
            if (rc != FACE_ERR_UNSUPPORTED || !c.work) return rc;
            c.work = nullptr;                    // no such kernel for weights split ahead
            return launch_rows(c, S);
        }
    }
    return launch_rows(c, rows_shape(c));
}

// y[r] = b + sum_k silu(x[r, k]) w[k]: the energy row of the readout's last layer (face/model.py:336). One
// column is far below the matrix cores' 32, and the layer's other columns need it neither as padding nor
// as a second pass: one wave per row reads the activations once, whole lines of 16 bytes per lane.
__global__ __launch_bounds__(256) void silu_dot_kernel(const float* __restrict__ x, int64_t ld_x, int64_t m, int k,
                                                       const float* __restrict__ w, const float* __restrict__ b,
                                                       float* __restrict__ y) {
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t r = (int64_t)blockIdx.x * 4 + threadIdx.x / kWave;
    if (r >= m) return;
    float s = 0.f;
    for (int c = 4 * lane; c < k; c += 4 * kWave) {
        const v4f a = ld4(x + r * ld_x + c), f = ld4(w + c);
#pragma unroll
        for (int i = 0; i < 4; ++i) s = fmaf(gemm_op(a[i], 0.f, 1), f[i], s);
    }
    s = group_sum(s, kWave);
    if (lane == 0) y[r] = s + (b ? *b : 0.f);
}

extern "C" int face_silu_dot(const float* x, int64_t ld_x, int64_t m, int32_t k, const float* w, const float* b, float* y,
                             void* stream) {
    if (m < 0 || k < 4 || k % 4 || ld_x < k || (m > 0 && (!x || !w || !y))) return FACE_ERR_ARG;
    if (ld_x % 4 || !al16(x) || !al16(w) || m > (int64_t)INT32_MAX) return FACE_ERR_UNSUPPORTED;
    if (m == 0) return 0;
    hipLaunchKernelGGL(silu_dot_kernel, dim3((unsigned)((m + 3) / 4)), dim3(256), 0, (hipStream_t)stream, x, ld_x, m, k, w,
                       b, y);
    FACE_LAUNCH_CHECK();
    return 0;
}
