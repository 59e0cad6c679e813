// CP pooling fed by the last radial layer, forward, in one launch (face/model.py:469-472, 496-502):
// R = h2 W^T + b (the layer's CP columns) and A[i, x, c] = sum_{e in row i} Y[e, x] env[e] R[e, l(x), c] m[e, c].
#include "edges.h"

#include <algorithm>

namespace face {

// Workgroup = (32-channel part, group of kCrfWaves edge shares): the limbs of the part's W rows (4 ranks
// x 32 channels, 48 KB at H = 64) sit in LDS for the whole launch; wave w walks the atom rows whose first
// edge lies in its equal share of the edges, in tiles of 32 consecutive edges that may span atom rows.
// D = h2 . W^T with edges as rows: lane c holds R of 16 edges for one channel, per rank, so R goes out
// in whole 128-byte lines and the pooling is 20 multiply-adds per (edge, channel) on the vector unit
// into 20 sums per lane, Y read as broadcasts from the tile's rows in LDS. The two halves of the wave
// hold the sums of different edges of an atom: they meet when the atom's last edge is pooled and its
// row is stored. Atoms with no edges get zero rows. A differs from the edge-serial cp_density_fwd
// kernels in rounding only; R is bitwise the edge_linear_fwd product.
// R goes out through non-temporal stores (read next by the backward, milliseconds later).
// Bound by two waves per SIMD (256 registers) and the stores: 24,000 atoms, 1.25 M edges, C = 160, H = 64:
// 1.29 ms with per-edge messages and 1.26 with table messages (fp32 instructions with the pooling on them:
// 1.87, and 1.14 + 0.82 ms for head and pooling), 0.90 without R; in timing-only variants the products
// and the pooling take 0.34 ms each, the message loads 0.07. What moved it: no spilled address and no branch
// around an optional operand's load (each wait includes the stores of R in flight). Measured and not
// kept: waiting for the next tile's loads before the stores of R (spills; 1.73 ms).
constexpr int kCrfWaves = 4;
constexpr int kCrfRow = 24;      // floats per edge of the Y tile: x 0-9, envelope, message row, x 10-19, 2 unused

template <int HB>
__global__ __launch_bounds__(kCrfWaves * kWave) __attribute__((amdgpu_waves_per_eu(2))) void cp_radial_fwd_kernel(
    const float* __restrict__ h2, int ld_h2, const float* __restrict__ w, const float* __restrict__ b,
    const float* __restrict__ env, const float* __restrict__ msg, int ld_msg, const int32_t* __restrict__ msg_row,
    const float* __restrict__ Y, int ld_Y, const int32_t* __restrict__ row_ptr, int64_t N, int C, int nparts,
    RankOut A, float* __restrict__ R, int ld_R) {
    constexpr int H = 16 * HB;
    extern __shared__ v8bf lds[];                     // 4 limb images (one per rank), the biases, the waves' Y tiles
    const int tid = threadIdx.x, lane = tid & (kWave - 1), half = lane >> 5;
    const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
    // blocks b and b + 8 run on the same XCD: all parts of an edge share read its rows through one L2
    const int bid = blockIdx.x;
    const int part = (bid / 8) % nparts;
    const int64_t grp = (int64_t)(bid / (8 * nparts)) * 8 + (bid & 7);
    const int64_t ngrp = gridDim.x / nparts;
    const int c = 32 * part + (lane & 31);
    const bool in_c = c < C;
    const int cc = in_c ? c : C - 1;
    const int64_t E = row_ptr[N];
    // W and h2 may be NULL when there are no edges (then only zero rows are written)
    if (E > 0 && (w == nullptr || h2 == nullptr)) return;
    bool big = false;
    if (E > 0)
        big = stage_limbs<HB>(lds, 4, [&](int l, int f) {
            const int ch = 32 * part + f;
            return ch < C ? w + (int64_t)(l * C + ch) * H : nullptr;
        });
    float* const sb = reinterpret_cast<float*>(lds + 4 * kLimbImage<HB>);      // the part's 4 x 32 biases
    for (int v = tid; v < 128; v += kCrfWaves * kWave)
        sb[v] = b ? b[(v >> 5) * C + min(32 * part + (v & 31), C - 1)] : 0.f;
    big = __syncthreads_or(big);
    float* const yt = sb + 128 + wv * 32 * kCrfRow;
    const int64_t W = ngrp * kCrfWaves, gw = grp * kCrfWaves + wv;
    int64_t at = uniform64(wave_lower_bound(row_ptr, N, E * gw / W, lane));
    const int64_t a_end = gw + 1 == W ? N : uniform64(wave_lower_bound(row_ptr, N, E * (gw + 1) / W, lane));
    if (at >= a_end) return;
    const int64_t e_beg = row_ptr[at], e_end = row_ptr[a_end];
    // row_ptr[i] with i wave-uniform: a scalar load, which waits for no store in flight
    auto rp = [&](int64_t i) __attribute__((always_inline)) { return (int64_t)row_ptr[uniform64(i)]; };
    // Two monomials of an atom's row, x and x + 1 of one rank (the second in the upper half of the wave),
    // or x = 0 and 3, at a wave-uniform base and a 32-bit lane offset. The stride passes through an empty
    // asm so that the bases are formed where they are used, not held for the whole launch.
    const uint32_t pair_off = (uint32_t)((half ? A.sx : 0) + c) * 4u;
    auto put_pair = [&](int64_t atom, int x, float v) __attribute__((always_inline)) {
        int64_t sx = A.sx;
        asm volatile("" : "+s"(sx));
        if (!in_c) return;
        if (x == 0) {
            float* p = half ? A.p[1] + 2 * sx : A.p[0];
            p[atom * A.sa + c] = v;
        } else {
            const int l = rank_of(x);
            char* p = reinterpret_cast<char*>(A.p[l] + atom * A.sa + (x - rank_start(l)) * sx);
            *reinterpret_cast<float*>(p + pair_off) = v;
        }
    };
    // leading rows with no edges (and the whole share when it has none)
    while (at < a_end && rp(at + 1) == rp(at)) {
        put_pair(at, 0, 0.f), put_pair(at, 1, 0.f);
#pragma unroll
        for (int x = 4; x < 20; x += 2) put_pair(at, x, 0.f);
        ++at;
    }
    if (e_beg >= e_end) return;
    const uint32_t r_off = (uint32_t)(4 * half * ld_R + c) * 4u;
    float sum[20];
#pragma unroll
    for (int x = 0; x < 20; ++x) sum[x] = 0.f;
    // a tile's h2 rows (A operand: lane = edge, 8 inputs per 16) and Y rows (lane = edge, 10 monomials
    // per half), loaded while the tile before it computes; edges past the share repeat its last one
    v4f hn[2 * HB];
    float yn[10], xn;
    const float* const x_lo = env ? env : Y;          // always a valid row: no branch around the load
    const float* const x_hi = msg_row ? reinterpret_cast<const float*>(msg_row) : Y;
    auto load_tile = [&](int64_t t0) __attribute__((always_inline)) {
        int ln = lane;                                // through an empty asm: addresses are formed here, not
        asm volatile("" : "+v"(ln));                  // held for the whole launch
        const int half = ln >> 5;
        const int64_t e = min(t0 + (ln & 31), e_end - 1);
#pragma unroll
        for (int s = 0; s < HB; ++s) {
            hn[2 * s] = ld4(h2 + e * ld_h2 + 16 * s + 8 * half);
            hn[2 * s + 1] = ld4(h2 + e * ld_h2 + 16 * s + 8 * half + 4);
        }
        const float* ye = Y + e * ld_Y + 10 * half;
        __builtin_memcpy(yn, ye, sizeof(yn));         // rows of any alignment
        xn = (half ? x_hi : x_lo)[e];
    };
    load_tile(e_beg);
    // A tile whose Y rows hold a NaN or an infinity is walked once per atom segment, the rows of the other
    // atoms' edges zero: zero times such a value is NaN, and only the products of other atoms' edges are
    // zeroed below. first() is the first row of the current atom in the tile.
    auto first = [&](int64_t t0) __attribute__((always_inline)) { return (int)max(rp(at) - t0, (int64_t)0); };
    for (int64_t t0 = e_beg; t0 < e_end;) {
        float yc = 0.f;
#pragma unroll
        for (int k = 0; k < 10; ++k) yc = fmaf(yn[k], 0.f, yc);
        int n = (int)min((int64_t)32, e_end - t0);
        if (__any(yc != yc)) n = (int)min(rp(at + 1) - t0, (int64_t)n);
        Split8 x[HB];
        float mx = 0.f;
#pragma unroll
        for (int s = 0; s < HB; ++s) {
            x[s] = split8(hn[2 * s], hn[2 * s + 1]);
            mx = max_abs8(hn[2 * s], hn[2 * s + 1], mx);
        }
        const bool plain = big || __any(mx > kLimbMax);
        {
            float* d = yt + (lane & 31) * kCrfRow + 12 * half;
            const int w0 = first(t0);
#pragma unroll
            for (int k = 0; k < 10; ++k) d[k] = (lane & 31) >= w0 && (lane & 31) < n ? yn[k] : 0.f;
            yt[(lane & 31) * kCrfRow + 10 + half] = half || env ? xn : 1.f;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const float* const yl = yt + 4 * half * kCrfRow;
        // message times envelope of the lane's 16 edges
        float me[16];
        if (msg_row) {
#pragma unroll
            for (int r = 0; r < 16; ++r)
                me[r] = msg[(int64_t)__builtin_bit_cast(int32_t, yl[d_row(r) * kCrfRow + 11]) * ld_msg + cc];
        } else {
            const float* mt = msg + t0 * ld_msg;
#pragma unroll
            for (int r = 0; r < 16; ++r) me[r] = mt[(int64_t)min(d_row(r) + 4 * half, n - 1) * ld_msg + cc];
        }
        const int64_t t1 = n == 32 || t0 + n == e_end ? t0 + 32 : t0;
        if (t1 < e_end) load_tile(t1);
        int64_t nxt = at;
        // ranks L0 .. L0 + NL - 1 (monomials X0 .. X1 - 1): R, its rows out, the pooling
        auto ranks = [&](auto L0_, auto NL_) __attribute__((always_inline)) {
            constexpr int L0 = decltype(L0_)::value, NL = decltype(NL_)::value;
            __builtin_amdgcn_sched_barrier(0);        // one group's operands live at a time
            constexpr int X0 = rank_start(L0), X1 = L0 + NL < 4 ? rank_start(L0 + NL) : 20;
            v16f acc[NL];
#pragma unroll
            for (int l = 0; l < NL; ++l)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[l][r] = 0.f;
            limb_products<HB, NL, true>(
                x, [&](int l) __attribute__((always_inline)) { return lds + (L0 + l) * kLimbImage<HB>; }, lane, acc);
            if (L0 == 0) {                            // here, where the products have covered the loads
#pragma unroll
                for (int r = 0; r < 16; ++r) me[r] *= yl[d_row(r) * kCrfRow + 10];
            }
            if (plain) {                              // a row at a time: this branch holds few registers
                int64_t row0 = t0 * ld_h2;            // (and its addresses stay in it)
                int last = n - 1;
                asm volatile("" : "+s"(row0), "+s"(last));
#pragma unroll
                for (int l = 0; l < NL; ++l)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const float* he = h2 + row0 + (int64_t)min(d_row(r) + 4 * half, last) * ld_h2;
                        const float* we = w + (int64_t)((L0 + l) * C + cc) * H;
                        float s = 0.f;
#pragma unroll 1
                        for (int k = 0; k < H; ++k) s = fmaf(he[k], we[k], s);
                        acc[l][r] = s;
                    }
            }
#pragma unroll
            for (int l = 0; l < NL; ++l) {
                const float bias = sb[32 * (L0 + l) + (lane & 31)];
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[l][r] += bias;
                if (R && in_c) {
                    int64_t ld = ld_R;                // wave-uniform row addresses, formed here
                    asm volatile("" : "+s"(ld));
                    float* const Rt = R + t0 * ld + (L0 + l) * C;
                    auto put = [&](int r) __attribute__((always_inline)) {
                        char* p = reinterpret_cast<char*>(Rt + d_row(r) * ld);
                        __builtin_nontemporal_store(acc[l][r], reinterpret_cast<float*>(p + r_off));
                    };
                    if (n == 32) {
#pragma unroll
                        for (int r = 0; r < 16; ++r) put(r);
                    } else {
#pragma unroll
                        for (int r = 0; r < 16; ++r)
                            if (d_row(r) + 4 * half < n) put(r);
                    }
                }
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[l][r] *= me[r];
            }
            // the tile's atom segments [lo, hi)
            int64_t a = at;
            int lo = first(t0);
            while (true) {
                const int64_t a_hi = rp(a + 1) - t0;
                const int hi = (int)min(a_hi, (int64_t)n);
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    if (lo < 8 * g + 8 && hi > 8 * g) {
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const int r = 4 * g + q, row = 8 * g + q + 4 * half;
                            const bool in = row >= lo && row < hi;
                            const float* ye = yl + d_row(r) * kCrfRow;
#pragma unroll
                            for (int l = 0; l < NL; ++l) {
                                const float v = in ? acc[l][r] : 0.f;
                                constexpr int nl[4] = {1, 3, 6, 10};
#pragma unroll
                                for (int k = 0; k < nl[L0 + l]; ++k) {
                                    const int m = rank_start(L0 + l) + k;
                                    sum[m] = fmaf(ye[m + (m >= 10 ? 2 : 0)], v, sum[m]);
                                }
                            }
                        }
                    }
                }
                if (a_hi > n) break;                  // the atom goes on into the next tile
#pragma unroll
                for (int p = X0; p < X1; p += 2) {
                    const int m0 = X0 == 0 && p == 2 ? 1 : p, m1 = X0 > 0 ? p + 1 : (p == 0 ? 3 : 2);
                    // the lower half keeps m0 and is given the upper half's, which keeps m1
                    const float got = __shfl_xor(half ? sum[m0] : sum[m1], 32, kWave);
                    put_pair(a, m0, (half ? sum[m1] : sum[m0]) + got);
                    sum[m0] = 0.f, sum[m1] = 0.f;
                }
                ++a;
                while (a < a_end && rp(a + 1) - t0 == a_hi) {
#pragma unroll
                    for (int p = X0; p < X1; p += 2) put_pair(a, X0 == 0 && p == 2 ? 1 : p, 0.f);
                    ++a;
                }
                if (a >= a_end || a_hi >= n) break;
                lo = (int)a_hi;
            }
            nxt = a;
        };
        ranks(std::integral_constant<int, 0>{}, std::integral_constant<int, 2>{});
        ranks(std::integral_constant<int, 2>{}, std::integral_constant<int, 1>{});
        ranks(std::integral_constant<int, 3>{}, std::integral_constant<int, 1>{});
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();              // the Y tile is overwritten next
        at = nxt;
        t0 = n == 32 || t0 + n == e_end ? t0 + 32 : t0;
    }
}

}  // namespace face

using namespace face;

extern "C" int face_cp_radial_fwd(const float* h2, int32_t ld_h2, int32_t H, const float* w, const float* b,
                                  const float* env, const float* msg, int32_t ld_msg, const int32_t* msg_row,
                                  const float* Y, int32_t ld_Y, const int32_t* row_ptr, int64_t N, int64_t E,
                                  int32_t C, float* const* A_ranks, int64_t atom_stride, int64_t x_stride, float* R,
                                  int32_t ld_R, void* stream) {
    if (N < 0 || E < 0 || C <= 0 || H < 16 || H > 64 || H % 16 || ld_h2 < H || ld_msg < C || ld_Y < 20 ||
        (R && ld_R < 4 * C))
        return FACE_ERR_ARG;
    if (N == 0) return 0;
    RankOut A;
    if ((E > 0 && (!h2 || !w)) || !msg || !Y || !row_ptr || !rank_out(A_ranks, atom_stride, x_stride, 20, A))
        return FACE_ERR_ARG;
    if (C % 16 || ld_h2 % 4 || !aligned16(h2) || !aligned16(w) || A.sx * 19 + C >= ((int64_t)1 << 31) ||
        (int64_t)ld_R * 16 >= ((int64_t)1 << 31))
        return FACE_ERR_UNSUPPORTED;
    const int nparts = (C + 31) / 32;
    const size_t lds = (size_t)(4 * (H / 16) * 3 * kWave) * 16 + (size_t)(128 + kCrfWaves * 32 * kCrfRow) * sizeof(float);
    if ((int64_t)lds > device_max_lds()) return FACE_ERR_UNSUPPORTED;
    // two workgroups per CU (LDS); edge shares of at least 2 tiles per wave; a multiple of 8 groups, so
    // that blocks b and b + 8 (one XCD) hold the parts of one group
    const int64_t most = std::max<int64_t>(1, 2 * (int64_t)device_cu_count() / (8 * nparts)) * 8;
    const int64_t ngrp = std::min(most, ((E + 32 * 2 * kCrfWaves - 1) / (32 * 2 * kCrfWaves) + 7) / 8 * 8);
    const dim3 grid((unsigned)(std::max<int64_t>(ngrp, 8) * nparts)), block(kCrfWaves * kWave);
    const hipStream_t st = (hipStream_t)stream;
#define FACE_CRF(HB_)                                                                                             \
    do {                                                                                                          \
        auto kern = cp_radial_fwd_kernel<HB_>;                                                                    \
        if (lds > 65536 &&                                                                                        \
            hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) \
            return FACE_ERR_UNSUPPORTED;                                                                          \
        hipLaunchKernelGGL(kern, grid, block, lds, st, h2, ld_h2, w, b, env, msg, ld_msg, msg_row, Y, ld_Y,         \
                           row_ptr, N, C, nparts, A, R, ld_R);                                                    \
    } while (0)
    switch (H / 16) {
        case 1: FACE_CRF(1); break;
        case 2: FACE_CRF(2); break;
        case 3: FACE_CRF(3); break;
        default: FACE_CRF(4); break;
    }
#undef FACE_CRF
    FACE_LAUNCH_CHECK();
    return 0;
}
