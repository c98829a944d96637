// FP64 tridiagonalisation in two stages, K = Q1 B Q1^T (dense to a band of kBW
// subdiagonals) and B = Q2 T Q2^T (bulge chasing), batched over submatrices.
//
// The one-stage reduction (tridiag.hip) reads the trailing matrix once per
// column: sum 4 m^3 / 3 bytes, which HBM bounds.  Here the trailing matrix is
// read and rewritten once per kBW columns by matrix-core products, and the band
// (17 m doubles) is reduced inside one CU.
//
// Stage 1, per panel p of kBW columns k0 .. k0 + 15 (rows from r0 = k0 + 16 on):
//   k_band_qr    Householder QR of the panel below the band in registers;
//                V into the matrix and the panel buffers, R into the band,
//                the WY factor T;
//   k_band_step  the previous panel's update A22 -= V W^T + W V^T (lower
//                triangle) and X = A22 V with the updated tiles, in one pass
//                over the matrix;
//   k_band_x     X summed from the tiles' parts;
//   k_band_w     W = X T - V (T^T (V^T X) T) / 2, and this panel's update on the
//                16 columns that the next panel factors.
// The reflector of column c has its unit at row c + kBW.
//
// Stage 2 (k_chase): sweep s removes column s outside the tridiagonal with a
// reflector over rows s+1 .. s+16 and chases the bulge down in windows of 16
// rows, window k of sweep s being rows s + 1 + 16 k + (0 .. 15).  Reflector
// (s, k) acts on that window.
//
// Application of Q2: the reflectors of 16 consecutive sweeps at one window k
// form a block I - V T V^T of 31 rows.  Q2 is the product over the sweep
// groups G ascending, and inside a group over k descending (blocks of a group
// overlap only their neighbours, and this order keeps every overlapping pair).
#include <algorithm>
#include <type_traits>
#include <utility>

#include "reflector.hpp"
#include "sm_internal.hpp"

namespace {

typedef double d4_t __attribute__((ext_vector_type(4)));
typedef double d2_t __attribute__((ext_vector_type(2)));

constexpr int kBW = kBandWidth;  // 16
constexpr int kABL = kBW + 1;    // doubles per column of the band buffer

// One submatrix of the band route (largest first).
struct BandSub {
    int64_t off;   // matrix block in the arena
    int64_t pw;    // panel buffers by rows (ld x 16 each): V of even and odd panels, W, X; T (256)
    int64_t px;    // parts of X: a 64 x 16 block per tile, then one per unit of k_band_step;
                   // parts of V^T X: 1024 per strip
    int64_t ab;    // band: column c at ab + 17 c, element d below the diagonal at + d
    int64_t blk;   // first block of its Q2 reflectors
    int m, ld, mapoff, ng;  // ng sweep groups
};

// blocks of Q2 per submatrix: group G has ng - G of them (windows that hold at
// least two rows), group after group
__host__ __device__ inline int q2_groups(int m) { return m >= 3 ? (m - 3) / kBW + 1 : 0; }
__device__ inline int64_t q2_block(int ng, int G, int k) {
    return (int64_t)G * ng - (int64_t)G * (G - 1) / 2 + k;
}

// ---- cross-lane sums --------------------------------------------------------
template <int CTRL>
__device__ __forceinline__ double dpp_add(double v) {
    return v + dpp_mov<CTRL>(v);
}
// sum over the 16 lanes of a row, in every lane: quad_perm 1032, 2301, then
// the mirrors within 8 and within 16
__device__ __forceinline__ double row_sum(double v) {
    v = dpp_add<0xB1>(v);
    v = dpp_add<0x4E>(v);
    v = dpp_add<0x141>(v);
    return dpp_add<0x140>(v);
}
// sums over the 16 lanes of a row of four values, times a, in every lane: two
// halving exchanges (quad_perm 1032, 2301) leave one value per lane, summed over
// the quads by rotations of 8 and 4 lanes and broadcast within each quad
__device__ __forceinline__ void row_sum4(const double (&p)[4], double a, int i, double (&z)[4]) {
    const bool b0 = i & 1, b1 = i & 2;
    const double h0 = (b0 ? p[2] : p[0]) + dpp_mov<0xB1>(b0 ? p[0] : p[2]);
    const double h1 = (b0 ? p[3] : p[1]) + dpp_mov<0xB1>(b0 ? p[1] : p[3]);
    double v = (b1 ? h1 : h0) + dpp_mov<0x4E>(b1 ? h0 : h1);
    v = dpp_add<0x128>(v);
    v = dpp_add<0x124>(v) * a;
    z[0] = dpp_mov<0x00>(v);
    z[1] = dpp_mov<0xAA>(v);
    z[2] = dpp_mov<0x55>(v);
    z[3] = dpp_mov<0xFF>(v);
}
// sum over the four 16-lane rows, in every lane
__device__ __forceinline__ double rows_sum(double v) {
    {
        const long long b = __double_as_longlong(v);
        const auto l = __builtin_amdgcn_permlane16_swap((unsigned)b, (unsigned)b, false, false);
        const auto h = __builtin_amdgcn_permlane16_swap((unsigned)(b >> 32), (unsigned)(b >> 32), false, false);
        v = __longlong_as_double(((long long)h[0] << 32) | l[0]) +
            __longlong_as_double(((long long)h[1] << 32) | l[1]);
    }
    const long long b = __double_as_longlong(v);
    const auto l = __builtin_amdgcn_permlane32_swap((unsigned)b, (unsigned)b, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap((unsigned)(b >> 32), (unsigned)(b >> 32), false, false);
    return __longlong_as_double(((long long)h[0] << 32) | l[0]) +
           __longlong_as_double(((long long)h[1] << 32) | l[1]);
}
// Sum over the wavefront of 16 values per lane; value q ends in the lanes with
// (lane >> 2) & 15 == q.
__device__ __forceinline__ double sum16(const double (&p)[16], int lane) {
    double h8[8], h4[4], h2[2];
    const bool b5 = lane & 32, b4 = lane & 16, b3 = lane & 8, b2 = lane & 4;
#pragma unroll
    for (int j = 0; j < 8; ++j) h8[j] = (b5 ? p[j + 8] : p[j]) + __shfl_xor(b5 ? p[j] : p[j + 8], 32);
#pragma unroll
    for (int j = 0; j < 4; ++j) h4[j] = (b4 ? h8[j + 4] : h8[j]) + __shfl_xor(b4 ? h8[j] : h8[j + 4], 16);
#pragma unroll
    for (int j = 0; j < 2; ++j) h2[j] = (b3 ? h4[j + 2] : h4[j]) + __shfl_xor(b3 ? h4[j] : h4[j + 2], 8);
    const double v = (b2 ? h2[1] : h2[0]) + __shfl_xor(b2 ? h2[0] : h2[1], 4);
    return dpp_add<0x4E>(dpp_add<0xB1>(v));
}

// reflector() for the chase, where it is on the serial chain of every step: the norm
// and its reciprocal from one hardware estimate of 1 / sqrt (coupled Newton
// steps), the scale from one of 1 / x, each refined to rounding level.  The chase
// works on a matrix whose largest element is near 1, so elements that the test drops
// (3e-145 of it) count for nothing, and the squares of the others are normal.
__device__ __forceinline__ Reflector reflector_fast(double alpha, double sigma) {
    if (sigma < kSquareMin) return {alpha, 0.0, 0.0};
    const double n2 = alpha * alpha + sigma, y = __builtin_amdgcn_rsq(n2);
    double g = n2 * y, h = 0.5 * y;
    double e = fma(-h, g, 0.5);
    g = fma(g, e, g), h = fma(h, e, h);
    e = fma(-h, g, 0.5);
    g = fma(g, e, g), h = fma(h, e, h);
    g = fma(fma(-g, g, n2), h, g);  // sqrt(n2), 2 h its reciprocal
    h = fma(h, fma(-2.0 * h, g, 1.0), h);
    const double q = fabs(alpha) + g;
    double r = __builtin_amdgcn_rcp(q);
    r = fma(r, fma(-q, r, 1.0), r);
    r = fma(r, fma(-q, r, 1.0), r);
    return {-copysign(g, alpha), fma(2.0 * h, fabs(alpha), 1.0), copysign(r, alpha)};
}

// ---- stage 1 ------------------------------------------------------------------

// QR of one 16-column panel, rows r0 .. m - 1 in registers (thread t holds rows
// t + NT q): per column one pass of 16 dot products x^T A(:, l) over the rows
// below the pivot (l = j: sigma; l > j: the update; l < j: V^T v for T), one
// barrier, one update.  A workgroup's time is the serial chain of its 16 columns
// (about 1 us each), so the panel stays in registers and the workgroups of
// other submatrices fill the CU.  The row-to-thread map and the order of every sum
// depend on the panel's own height only.
template <int NT, int R>
__global__ __launch_bounds__(NT, R == 4 ? 2 : 4) void k_band_qr(const BandSub *__restrict__ subs,
                                                 double *__restrict__ Aa, double *__restrict__ PW,
                                                 double *__restrict__ ABa,
                                                 double *__restrict__ tau_all, int first, int panel) {
    constexpr int NW = NT / PTB_WAVE;
    const BandSub d = subs[first + blockIdx.x];
    const int k0 = panel * kBW, r0 = k0 + kBW;
    const int n = d.m - r0;
    if (n < 2) return;
    const int nref = min(kBW, n - 1);
    __shared__ double red[2][NW][kBW], prow[2][kBW], zt[kBW][kBW], ts[kBW];
    const int lane = threadIdx.x % PTB_WAVE, wave = threadIdx.x / PTB_WAVE;
    double *a = Aa + d.off + (int64_t)k0 * d.ld + r0;
    double x[R][kBW];
#pragma unroll
    for (int q = 0; q < R; ++q) {
        const int i = threadIdx.x + NT * q;
        const unsigned ic = (unsigned)min(i, n - 1);
#pragma unroll
        for (int l = 0; l < kBW; ++l) x[q][l] = a[(unsigned)(l * d.ld) + ic];
    }
#pragma unroll
    for (int q = 0; q < R; ++q)
#pragma unroll
        for (int l = 0; l < kBW; ++l) x[q][l] = (int)threadIdx.x + NT * q < n ? x[q][l] : 0.0;
    auto column = [&](auto J) {
        constexpr int j = decltype(J)::value;
        if (j >= nref) return;
        const int bf = j & 1;
        const int l = lane & 15;
        double pl, dot, alpha, sigma, down = 1.0;
        for (;;) {
            double p[kBW];
#pragma unroll
            for (int l = 0; l < kBW; ++l) p[l] = 0.0;
#pragma unroll
            for (int q = 0; q < R; ++q) {
                const double xi = (int)threadIdx.x + NT * q > j ? x[q][j] : 0.0;
#pragma unroll
                for (int l = 0; l < kBW; ++l) p[l] += xi * x[q][l];
            }
            const double s = sum16(p, lane);
            if ((lane & 3) == 0) red[bf][wave][lane >> 2] = s;
            if ((int)threadIdx.x == j)
#pragma unroll
                for (int l = 0; l < kBW; ++l) prow[bf][l] = x[0][l];
            __syncthreads();
            // every wavefront forms the scalars, lane l (mod 16) those of column l
            dot = 0.0;
#pragma unroll
            for (int w = 0; w < NW; ++w) dot += red[bf][w][l];
            pl = prow[bf][l];
            alpha = read_lane(pl, j), sigma = read_lane(dot, j);
            if (!(alpha * alpha + sigma < kSquareMin) || down != 1.0) break;
            down = 1.0 / kRescale;
#pragma unroll
            for (int q = 0; q < R; ++q)
                x[q][j] *= (int)threadIdx.x + NT * q >= j ? kRescale : 1.0;
            __syncthreads();  // (the sums are written again)
        }
        Reflector h = reflector(alpha, sigma);
        h.beta *= down;
        const double zl = pl + h.scale * dot;  // A(:, l)^T v
        const double wl = l > j ? h.tau * zl : 0.0;
        if (threadIdx.x < kBW) zt[j][l] = zl;
        if (threadIdx.x == 0) ts[j] = h.tau;
        double ws_[kBW];
#pragma unroll
        for (int c = j + 1; c < kBW; ++c) ws_[c] = read_lane(wl, c);
#pragma unroll
        for (int q = 0; q < R; ++q) {
            const int i = threadIdx.x + NT * q;
            const double vi = i > j ? x[q][j] * h.scale : i == j ? 1.0 : 0.0;
#pragma unroll
            for (int c = j + 1; c < kBW; ++c) x[q][c] -= ws_[c] * vi;
            x[q][j] = i > j ? vi : i == j ? h.beta : x[q][j];
        }
    };
    column(std::integral_constant<int, 0>{}), column(std::integral_constant<int, 1>{});
    column(std::integral_constant<int, 2>{}), column(std::integral_constant<int, 3>{});
    column(std::integral_constant<int, 4>{}), column(std::integral_constant<int, 5>{});
    column(std::integral_constant<int, 6>{}), column(std::integral_constant<int, 7>{});
    column(std::integral_constant<int, 8>{}), column(std::integral_constant<int, 9>{});
    column(std::integral_constant<int, 10>{}), column(std::integral_constant<int, 11>{});
    column(std::integral_constant<int, 12>{}), column(std::integral_constant<int, 13>{});
    column(std::integral_constant<int, 14>{}), column(std::integral_constant<int, 15>{});
    __syncthreads();
    double *vr = PW + d.pw + (int64_t)(panel & 1) * 16 * d.ld;
    double *T = PW + d.pw + (int64_t)64 * d.ld;
    // R into the band, T (wavefront 0; lane i holds row i)
    if (threadIdx.x < kBW) {
        const int i = threadIdx.x;
        double *ab = ABa + d.ab;
        if (i < n)
#pragma unroll
            for (int l = 0; l < kBW; ++l)
                if (l >= i) ab[(int64_t)(k0 + l) * kABL + kBW + i - l] = x[0][l];
        double t[kBW];
#pragma unroll
        for (int j = 0; j < kBW; ++j) {
            double s = 0.0;
            if (j < nref) {
#pragma unroll
                for (int c = 0; c < j; ++c) s += t[c] * zt[j][c];
                const double tj = ts[j];
                t[j] = i == j ? tj : i < j ? -tj * s : 0.0;
                if (i == j) tau_all[d.mapoff + k0 + j] = tj;
            } else {
                t[j] = 0.0;
            }
            T[j * kBW + i] = t[j];
        }
    }
    // V: unit lower trapezoidal, zero columns past the last reflector
#pragma unroll
    for (int q = 0; q < R; ++q) {
        const int i = threadIdx.x + NT * q;
#pragma unroll
        for (int l = 0; l < kBW; ++l) {
            const double v = l >= nref ? 0.0 : i > l ? x[q][l] : i == l ? 1.0 : 0.0;
            x[q][l] = v;
            if (i < n && l < nref) a[(unsigned)(l * d.ld) + (unsigned)i] = v;
        }
        // by rows, zero up to the next multiple of 16 rows
        if (i < ((n + 15) & ~15)) {
            d2_t *row = reinterpret_cast<d2_t *>(vr + (int64_t)(r0 + i) * kBW);
#pragma unroll
            for (int l = 0; l < kBW / 2; ++l) {
                const bool in = i < n;
                row[l] = d2_t{in ? x[q][2 * l] : 0.0, in ? x[q][2 * l + 1] : 0.0};
            }
        }
    }
}

// Units of k_band_step: strip i (64 rows) in chunks of kChunk 64-column tiles.
// Strips 4 a .. 4 a + 3 have a + 1 chunks each.
constexpr int kChunk = 4;
__host__ __device__ inline int band_units(int ns) {  // of ns strips
    const int a = ns / kChunk;
    return 2 * a * (a + 1) + (ns - kChunk * a) * (a + 1);
}
// where a submatrix's parts of V^T X (1024 per strip) begin in its part buffer
__host__ __device__ inline int64_t gram_at(int m) {
    const int64_t ns = m > kBW ? (m - kBW + 63) / 64 : 0;
    return 1024 * (ns * (ns + 1) / 2 + band_units((int)ns));
}
__device__ inline int band_unit(int i, int q) { return band_units(i) + q; }

// One pass over the lower triangle of the trailing matrix (rows and columns from
// r0 = 16 (panel + 1) on): the previous panel's update (not for the first
// panel) and the parts of X = A22 V of this panel.  A 256-thread workgroup takes
// a strip of 64 rows and up to four 64 x 64 tiles of it, each wavefront 16 columns
// of a tile.  A tile is loaded with a lane per row (coalesced), which is both the
// result layout of v_mfma_f64_16x16x4 for A^T and its operand layout for A V, so
// it is updated, stored and multiplied from the same registers; A^T V takes it
// transposed through the wavefront's own LDS (no barrier).  Tile (i, j) gives rows
// of strip i (summed over the unit's tiles) and of strip j, both to the part
// buffers, summed by k_band_x in a fixed order.  Bound by HBM: the triangle is read
// and written once, and parts of a quarter of it written and read (1.3e11 bytes at
// 4.0 TB/s on the 512-water box), instead of three reads and a write: 38.8 ms per
// build with k_band_x, against 47.0 for separate product and update kernels (39.7
// against 42.6 on 256 molecules), and no host tables.  134 VGPRs and 42 KB of LDS
// hold three workgroups per CU; with the next tile's loads in flight the kernel
// spills (72 ms).  grid: 8 XCDs x (submatrices of an XCD x units); a submatrix's
// units run on one XCD.
template <bool UPD>
__global__ __launch_bounds__(256, 3) void k_band_step(const BandSub *__restrict__ subs, int nsub,
                                                      double *__restrict__ Aa,
                                                      const double *__restrict__ PW,
                                                      double *__restrict__ PXa, int panel, int nunit) {
    const unsigned lin = blockIdx.x, slot = lin >> 3;
    const int si = (int)((slot / (unsigned)nunit) * 8 + (lin & 7));
    if (si >= nsub) return;
    const BandSub d = subs[si];
    const int r0 = panel * kBW + kBW;
    const int n = d.m - r0;
    if (n < 2) return;
    const int ns = (n + 63) / 64;
    const int unit = (int)(slot % (unsigned)nunit);
    if (unit >= band_units(ns)) return;
    int i = 0, q = 0;
    {
        int a = 0;
        while (2 * (a + 1) * (a + 2) <= unit) ++a;
        const int rem = unit - 2 * a * (a + 1);
        i = kChunk * a + rem / (a + 1);
        q = rem % (a + 1);
    }
    constexpr int LR = 66, LT = 34;
    __shared__ double vs[16][LR], ws_[16][LR], vn[64][16];
    __shared__ double tbuf[4][16][LT];
    const int lane = threadIdx.x % PTB_WAVE, lr = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PTB_WAVE);
    const unsigned ld = (unsigned)d.ld;
    double *a = Aa + d.off + (int64_t)r0 * d.ld + r0;
    const double *pw = PW + d.pw + (int64_t)r0 * kBW;
    const double *vprev = pw + (int64_t)((panel + 1) & 1) * 16 * d.ld;
    const double *vcur = pw + (int64_t)(panel & 1) * 16 * d.ld;
    const double *wprev = pw + (int64_t)32 * d.ld;
    double *px = PXa + d.px;
    const int rb = 64 * i;
    {
        // the strip's rows of V and W (previous panel, by columns) and of this V
        const int row = threadIdx.x >> 2, c = (threadIdx.x & 3) * 4;
        const bool in = rb + row < n;
        const unsigned at = (unsigned)min(rb + row, n - 1) * kBW + c;
        const d4_t z = *reinterpret_cast<const d4_t *>(vcur + at);
#pragma unroll
        for (int u = 0; u < 4; ++u) vn[row][c + u] = in ? z[u] : 0.0;
        if (UPD) {
            const d4_t x = *reinterpret_cast<const d4_t *>(vprev + at);
            const d4_t y = *reinterpret_cast<const d4_t *>(wprev + at);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                vs[c + u][row] = in ? x[u] : 0.0;
                ws_[c + u][row] = in ? y[u] : 0.0;
            }
        }
    }
    __syncthreads();
    d4_t xi[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) xi[b] = d4_t{0.0, 0.0, 0.0, 0.0};
    // one tile's 16 columns: A^T by row blocks, and the operands of its columns
    struct Tile {
        d4_t t[4];
        double wc[4], vc[4], vb[4];
    };
    const int j0 = kChunk * q;
    // 32-bit byte offsets from uniform bases: one register per address
    auto at = [](auto *base, unsigned bytes) {
        return reinterpret_cast<decltype(base)>(reinterpret_cast<uintptr_t>(base) + bytes);
    };
    unsigned ro[4];  // the lane's rows, clamped
#pragma unroll
    for (int b = 0; b < 4; ++b) ro[b] = 8u * (unsigned)min(rb + 16 * b + lr, n - 1);
    auto load = [&](int j, Tile &x) {
        const int cb = 64 * j + 16 * wave;
        const unsigned cl = 8u * ((unsigned)min(cb + lr, n - 1) * kBW + g);
        const unsigned cv = 8u * ((unsigned)(cb + g) * kBW + lr);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const unsigned co = 8u * (unsigned)min(cb + 4 * r + g, n - 1) * ld;
#pragma unroll
            for (int b = 0; b < 4; ++b) x.t[b][r] = *at(a, co + ro[b]);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (UPD) {
                x.wc[u] = *at(wprev, cl + 32 * u);
                x.vc[u] = *at(vprev, cl + 32 * u);
            }
            x.vb[u] = *at(vcur, cv + 512 * u);  // zero past n
        }
    };
    int zero = 0;
    const int jl = min(j0 + kChunk - 1, i);
    for (int j = j0; j <= jl && 64 * j + 16 * wave < n; ++j) {
        asm volatile("" : "+v"(zero));  // (keeps the strip's operands in LDS)
        Tile x;
        load(j, x);
        const int cb = 64 * j + 16 * wave;
        const bool diag = j == i, edge = diag || rb + 64 > n;  // cut by the diagonal or the last row
        if (UPD) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const double w = -x.wc[u], v = -x.vc[u];
#pragma unroll
                for (int b = 0; b < 4; ++b)
                    x.t[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(w, vs[4 * u + g][16 * b + lr + zero], x.t[b], 0, 0, 0);
#pragma unroll
                for (int b = 0; b < 4; ++b)
                    x.t[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(v, ws_[4 * u + g][16 * b + lr + zero], x.t[b], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);  // (else every operand is read ahead, and registers spill)
            }
        }
        const unsigned so = 8u * ((unsigned)(cb + g) * ld + (unsigned)(rb + lr)), ld32 = 32u * ld;
        d4_t xj = d4_t{0.0, 0.0, 0.0, 0.0}, xk = xj;
#pragma unroll
        for (int h = 0; h < 2; ++h) {  // 32 rows at a time through LDS
            double e[2][4];
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    e[b][r] = x.t[2 * h + b][r];
                    tbuf[wave][4 * r + g][16 * b + lr] = e[b][r];
                }
            if (edge) {
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int row = rb + 16 * (2 * h + b) + lr + zero, col = cb + 4 * r + g;
                        const bool on = row < n && col < n && (!diag || row >= col);
                        if (UPD && on) *at(a, so + r * ld32 + 128u * (2 * h + b)) = e[b][r];
                        e[b][r] = on ? e[b][r] : 0.0;
                        tbuf[wave][4 * r + g][16 * b + lr] = diag && row == col ? 0.0 : e[b][r];
                    }
            } else if (UPD) {
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int r = 0; r < 4; ++r) *at(a, so + r * ld32 + 128u * (2 * h + b)) = e[b][r];
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int b = 0; b < 2; ++b)
                    xi[2 * h + b] = __builtin_amdgcn_mfma_f64_16x16x4f64(e[b][r], x.vb[r], xi[2 * h + b], 0, 0, 0);
#pragma unroll
            for (int u = 0; u < 8; u += 2) {
                xj = __builtin_amdgcn_mfma_f64_16x16x4f64(tbuf[wave][lr][4 * u + g], vn[32 * h + 4 * u + g][lr + zero],
                                                          xj, 0, 0, 0);
                xk = __builtin_amdgcn_mfma_f64_16x16x4f64(tbuf[wave][lr][4 * u + 4 + g],
                                                          vn[32 * h + 4 * u + 4 + g][lr + zero], xk, 0, 0, 0);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_sched_barrier(0);
        }
        double *p = px + (int64_t)(i * (i + 1) / 2 + j) * 1024 + (16 * wave + g) * 16 + lr;
#pragma unroll
        for (int r = 0; r < 4; ++r) p[64 * r] = xj[r] + xk[r];
    }
    // the strip's own rows: the wavefronts' parts in fixed order, 32 rows at a time
    double *xs = &tbuf[0][0][0];  // [wave][32 x 16]
    const int ns0 = (d.m - kBW + 63) / 64;
    double *o = px + (int64_t)(ns0 * (ns0 + 1) / 2 + unit) * 1024;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        __syncthreads();
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) xs[wave * 512 + (16 * b + 4 * r + g) * 16 + lr] = xi[2 * h + b][r];
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int l = threadIdx.x + 256 * e;
            o[512 * h + l] = ((xs[l] + xs[512 + l]) + xs[1024 + l]) + xs[1536 + l];
        }
    }
}

// X (by rows) of one 64-row strip from its parts: the strip's own chunks, then
// the tiles below it in its columns, in order; SPLIT: and the strip's parts of
// V^T X, one of 16 rows per wavefront, behind the parts of X.
// grid: (submatrix, strip)
template <bool SPLIT>
__global__ __launch_bounds__(256) void k_band_x(const BandSub *__restrict__ subs,
                                                double *__restrict__ PXa, double *__restrict__ PW,
                                                int panel) {
    const BandSub d = subs[blockIdx.x];
    const int r0 = panel * kBW + kBW;
    const int n = d.m - r0, i = blockIdx.y;
    if (n < 2 || 64 * i >= n) return;
    const int ns = (n + 63) / 64, ns0 = (d.m - kBW + 63) / 64;
    double *px = PXa + d.px;
    const double *own = px + (int64_t)(ns0 * (ns0 + 1) / 2 + band_unit(i, 0)) * 1024;
    const int nq = i / kChunk + 1;
    double *x = PW + d.pw + (int64_t)48 * d.ld + (int64_t)(r0 + 64 * i) * kBW;
    const int rows = min(64, ((n + 15) & ~15) - 64 * i);
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    for (int q = 0; q < nq; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] += own[(int64_t)q * 1024 + threadIdx.x + 256 * e];
#pragma unroll 4
    for (int j = i; j < ns; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e)
            s[e] += px[(int64_t)(j * (j + 1) / 2 + i) * 1024 + threadIdx.x + 256 * e];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int l = threadIdx.x + 256 * e;
        s[e] = 64 * i + (l >> 4) < n ? s[e] : 0.0;
        if (l < 16 * rows) x[l] = s[e];
    }
    if constexpr (!SPLIT) return;
    __shared__ double xs[1024];
#pragma unroll
    for (int e = 0; e < 4; ++e) xs[threadIdx.x + 256 * e] = s[e];
    __syncthreads();
    const int lane = threadIdx.x % PTB_WAVE, wave = threadIdx.x / PTB_WAVE;
    const int lr = lane & 15, g = lane >> 4, k = 64 * i + 16 * wave;
    d4_t acc = d4_t{0.0, 0.0, 0.0, 0.0};
    if (k < n) {  // (V is zero up to the next multiple of 16 rows)
        const double *vr = PW + d.pw + (int64_t)(panel & 1) * 16 * d.ld + (int64_t)(r0 + k) * kBW;
#pragma unroll
        for (int u = 0; u < 4; ++u)
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(vr[(4 * u + g) * kBW + lr],
                                                       xs[(16 * wave + 4 * u + g) * kBW + lr], acc, 0, 0, 0);
    }
    double *gp = px + gram_at(d.m) + 1024 * i + 256 * wave;
#pragma unroll
    for (int r = 0; r < 4; ++r) gp[(4 * r + g) * kBW + lr] = acc[r];
}

// W = X T - V S, S = T^T (V^T X) T / 2, by rows, and the panel's update
// A -= V W^T + W V^T on the next 16 columns (rows and columns from r0 on), which
// the next panel's QR reads: V^T X on the matrix cores (wavefronts on alternate
// 16-row tiles, a sum of tile products each), the 16 x 16 products in LDS, then W^T
// and the columns tile by tile (lane = row; W^T's result layout is the operand
// layout of the update).  One workgroup per submatrix, or (SPLIT) one per strip of
// 64 rows, each adding up the parts of V^T X that k_band_x left, in the same order:
// the same bits.  SPLIT serves panels of no more submatrices than CUs (one of
// 1472 rows 27 us with k_band_x -> 14, 192 of 64 waters 24 -> 20); beyond that the
// parts cost more than the second workgroup gains (256 molecules: 328 us -> 393).
template <bool SPLIT>
__global__ __launch_bounds__(256) void k_band_w(const BandSub *__restrict__ subs,
                                                double *__restrict__ Aa, double *__restrict__ PW,
                                                const double *__restrict__ PXa, int panel) {
    const BandSub d = subs[blockIdx.x];
    const int r0 = panel * kBW + kBW;
    const int n = d.m - r0;
    if (n < 2 || 64 * (int)blockIdx.y >= n) return;
    double *pw = PW + d.pw;
    const double *vr = pw + (int64_t)(panel & 1) * 16 * d.ld + (int64_t)r0 * kBW;
    double *wr = pw + (int64_t)32 * d.ld + (int64_t)r0 * kBW;
    const double *xr = pw + (int64_t)48 * d.ld + (int64_t)r0 * kBW;
    const double *T = pw + (int64_t)64 * d.ld;
    double *a = Aa + d.off + (int64_t)r0 * d.ld + r0;
    __shared__ double gs[SPLIT ? 1 : 4][16][17], ts[16][17], ms[16][17], ss[16][17];
    const int lane = threadIdx.x % PTB_WAVE, wave = threadIdx.x / PTB_WAVE;
    const int lr = lane & 15, g = lane >> 4;
    const int ti = threadIdx.x & 15, tj = threadIdx.x >> 4;
    ts[ti][tj] = T[tj * kBW + ti];
    if constexpr (SPLIT) {
        const double *gp = PXa + d.px + gram_at(d.m) + threadIdx.x;
        double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
        for (int i = 0; i < (n + 63) / 64; ++i)
#pragma unroll
            for (int w = 0; w < 4; ++w) s[w] += gp[1024 * i + 256 * w];
        ss[tj][ti] = ((s[0] + s[1]) + s[2]) + s[3];
    } else {
        d4_t sum = d4_t{0.0, 0.0, 0.0, 0.0};
        for (int k = 16 * wave; k < n; k += 64) {
            double av[4], bv[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                av[u] = vr[(unsigned)(k + 4 * u + g) * kBW + lr];
                bv[u] = xr[(unsigned)(k + 4 * u + g) * kBW + lr];
            }
            d4_t acc = d4_t{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int u = 0; u < 4; ++u) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(av[u], bv[u], acc, 0, 0, 0);
            sum += acc;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) gs[wave][4 * r + g][lr] = sum[r];
        __syncthreads();
        ss[ti][tj] = ((gs[0][ti][tj] + gs[1][ti][tj]) + gs[2][ti][tj]) + gs[3][ti][tj];
    }
    __syncthreads();
    {
        double s = 0.0;  // M = G T
#pragma unroll
        for (int c = 0; c < 16; ++c) s += ss[ti][c] * ts[c][tj];
        ms[ti][tj] = s;
    }
    __syncthreads();
    {
        double s = 0.0;  // S = T^T M / 2
#pragma unroll
        for (int c = 0; c < 16; ++c) s += ts[c][ti] * ms[c][tj];
        ss[ti][tj] = 0.5 * s;
    }
    __syncthreads();
    // W^T(col, row) = sum_c T(c, col) X(row, c) - S(c, col) V(row, c)
    double ta[4], sa[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        ta[u] = ts[4 * u + g][lr];
        sa[u] = -ss[4 * u + g][lr];
    }
    auto make_w = [&](int k, double (&vb)[4]) {
        double xb[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            xb[u] = xr[(unsigned)(k + lr) * kBW + 4 * u + g];
            vb[u] = vr[(unsigned)(k + lr) * kBW + 4 * u + g];
        }
        d4_t w = d4_t{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            w = __builtin_amdgcn_mfma_f64_16x16x4f64(ta[u], xb[u], w, 0, 0, 0);
            w = __builtin_amdgcn_mfma_f64_16x16x4f64(sa[u], vb[u], w, 0, 0, 0);
        }
        return w;
    };
    // rows r0 .. r0 + 15 of V and W, the update's column operands
    double v0[4];
    const d4_t w0 = make_w(0, v0);
    for (int k = 64 * blockIdx.y + 16 * wave; k < n; k += 64 * gridDim.y) {
        const int row = k + lr;
        d4_t t;
#pragma unroll
        for (int r = 0; r < 4; ++r)
            t[r] = a[(unsigned)min(4 * r + g, n - 1) * (unsigned)d.ld + (unsigned)min(row, n - 1)];
        double vb[4];
        const d4_t w = make_w(k, vb);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            t = __builtin_amdgcn_mfma_f64_16x16x4f64(-w0[u], vb[u], t, 0, 0, 0);
            t = __builtin_amdgcn_mfma_f64_16x16x4f64(-v0[u], w[u], t, 0, 0, 0);
        }
        if (row < n)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                wr[(unsigned)row * kBW + 4 * r + g] = w[r];
                if (4 * r + g <= row) a[(unsigned)(4 * r + g) * (unsigned)d.ld + (unsigned)row] = t[r];
            }
        if (n == kBW + 1 && k == kBW) {  // no next panel: the last diagonal element
            double s = 0.0;
#pragma unroll
            for (int u = 0; u < 4; ++u) s += vb[u] * w[u];
            s = rows_sum(s);
            if (lane == 0) a[(unsigned)kBW * (unsigned)d.ld + kBW] -= 2.0 * s;
        }
    }
}

// The band's diagonal blocks (lower) and the rows below them that no panel
// reduced; then zeros in the reflector columns above the panel's own rows, as far
// as the block readers see (from 16 rows below the column's block of `qblk`
// reflectors).  grid: (submatrix, 16-column block)
__global__ __launch_bounds__(256) void k_band_extract(const BandSub *__restrict__ subs,
                                                      double *__restrict__ Aa,
                                                      double *__restrict__ ABa, int qblk) {
    const BandSub d = subs[blockIdx.x];
    const int k0 = blockIdx.y * kBW;
    if (k0 >= d.m) return;
    const bool qr = d.m - (k0 + kBW) >= 2;  // the panel was factored: R is in the band
    double *a = Aa + d.off;
    double *ab = ABa + d.ab;
    for (int l = threadIdx.x; l < kBW * kABL; l += 256) {
        const int c = k0 + l / kABL, dd = l % kABL, r = c + dd;
        if (c >= d.m) continue;
        if (r < k0 + kBW || !qr) ab[(int64_t)c * kABL + dd] = r < d.m ? a[(int64_t)c * d.ld + r] : 0.0;
    }
    __syncthreads();
    if (!qr) return;
    const int b0 = k0 & ~(qblk - 1);
    const int rows = k0 - b0;  // rows b0 + 16 .. k0 + 15
    for (int l = threadIdx.x; l < kBW * rows; l += 256) {
        const int c = k0 + l / rows, r = b0 + kBW + l % rows;
        if (c < d.m - kBW - 1) a[(int64_t)c * d.ld + r] = 0.0;
    }
}

// ---- stage 2 ------------------------------------------------------------------

// Message area of a chase, per window k: the reflector that acts on it (vm, by
// slot; tm), its diagonal block's first column and the element below it (cm,
// bm), and its off-diagonal block's first row (rm).  Before vm: what takes the
// scaled matrix back (vm[-2]).
struct ChaseLds {
    double *vm, *tm, *cm, *bm, *rm, *wsc;
};

// element c (the same in every lane) of a lane's four, by scalar branches (the empty
// statements keep them from becoming selects)
__device__ __forceinline__ void set_slot(double (&A)[4], int c, double v) {
    if (c == 0) {
        asm volatile("");
        A[0] = v;
    } else if (c == 1) {
        asm volatile("");
        A[1] = v;
    } else if (c == 2) {
        asm volatile("");
        A[2] = v;
    } else {
        asm volatile("");
        A[3] = v;
    }
}
__device__ __forceinline__ double get_slot(const double (&A)[4], int c) {
    double v;
    if (c == 0) {
        asm volatile("");
        v = A[0];
    } else if (c == 1) {
        asm volatile("");
        v = A[1];
    } else if (c == 2) {
        asm volatile("");
        v = A[2];
    } else {
        asm volatile("");
        v = A[3];
    }
    return v;
}

// One step of the chase: window k of sweep s.  A wavefront holds the window's
// diagonal block D and the block B below it (rows of window k + 1), 16 x 16, in
// cyclic slots: row or column r sits in slot r mod 16, so moving from sweep s - 1
// to sweep s replaces one slot and shifts nothing.  Lane l holds row slot l % 16
// and column slots 4 (l / 16) + c.  f = (s + 1) mod 16 is the slot of every
// window's first row.  BRANCH: slots are replaced under scalar and lane branches, 35
// vector instructions fewer than selects, where several windows per wavefront keep
// the CU's issue busy (512-water box 15.2 -> 14.3 ms, 1472 rows 11.6 -> 10.2); a
// wavefront with one window of each parity waits for the branches instead (4-9 %).
template <bool BRANCH>
__device__ __forceinline__ void chase_step(double (&D)[4], double (&B)[4], int k, int s, int m, int ng,
                                           const ChaseLds &L, double *__restrict__ raw,
                                           double *__restrict__ rtau, double *__restrict__ dv,
                                           double *__restrict__ ev, int lane) {
    const int i = lane & 15, g = lane >> 4;
    const int fo = s & 15, f = (s + 1) & 15;
    if (s > 0) {
        // the slot of the row that left takes the row that enters: D's from B's
        // first row, B's column from the next window's first column
        const double cmv = L.cm[(k + 1) * 16 + i], bmv = L.bm[k + 1], rmv = L.rm[k * 16 + i];
        const bool rf = i == fo;
        const double dcol = rf ? cmv : rmv, bcol = rf ? bmv : cmv;
        if constexpr (BRANCH) {
            if (rf) {
                asm volatile("");
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    D[c] = B[c];
                    B[c] = 0.0;
                }
            }
            if (g == fo >> 2) {
                set_slot(D, fo & 3, dcol);
                set_slot(B, fo & 3, bcol);
            }
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const bool cc = 4 * g + c == fo;
                D[c] = cc ? dcol : rf ? B[c] : D[c];
                B[c] = cc ? bcol : rf ? 0.0 : B[c];
            }
        }
    }
    const bool pivot = i == f;
    // where the reflectors of this step go (those the sweep has)
    const bool last = s >= m - 2;
    const unsigned ro = (unsigned)((i - f) & 15);
    const int64_t blk = q2_block(ng, s >> 4, k);
    if (k == 0) {
        // the sweep's first reflector: column s below its diagonal
        const double dia = L.cm[fo];
        const double x = i == fo ? L.bm[0] : L.cm[i];
        const Reflector h = reflector_fast(read_lane(x, f), row_sum(pivot ? 0.0 : x * x));
        const double u = pivot ? 1.0 : x * h.scale;
        if (g == 0) {
            L.vm[i] = u;
            if (!last) (raw + blk * 256 + (s & 15) * 16)[ro] = u;
        }
        if (lane == 0) {
            L.tm[0] = h.tau;
            dv[s] = dia * L.vm[-2];
            ev[s] = s < m - 1 ? h.beta * L.vm[-2] : 0.0;
            if (!last) rtau[blk * 16 + (s & 15)] = h.tau;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    const double vr = L.vm[k * 16 + i], tau = L.tm[k];
    double vc[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) vc[c] = L.vm[k * 16 + 4 * g + c];
    const int gf = f >> 2, cf = f & 3;
    double bf = 0.0;
    if constexpr (BRANCH) {
        if (g == gf) bf = get_slot(B, cf);
    } else {
        const double b0 = cf & 1 ? B[1] : B[0], b1 = cf & 1 ? B[3] : B[2];
        bf = g == gf ? (cf & 2 ? b1 : b0) : 0.0;
    }
    // p = D v, y = B v and B's first column, by rows
    double p = D[0] * vc[0], y = B[0] * vc[0];
#pragma unroll
    for (int c = 1; c < 4; ++c) {
        p += D[c] * vc[c];
        y += B[c] * vc[c];
    }
    p = tau * rows_sum(p);
    y = tau * rows_sum(y);
    // (v is 1 at the pivot, so the column after B <- B H is x = B(:, f) - y)
    const double x = rows_sum(bf) - y;
    const double pv = row_sum(p * vr), sig = row_sum(pivot ? 0.0 : x * x);
    const double w = p - (0.5 * tau * pv) * vr;
    if (g == 0) L.wsc[i] = w;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const Reflector h = reflector_fast(read_lane(x, f), sig);
    const double u = pivot ? 1.0 : x * h.scale;
    // B <- H' B H, its first column beta e
    double q[4], z[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        B[c] -= y * vc[c];
        q[c] = u * B[c];
    }
    row_sum4(q, h.tau, i, z);
    const double xf = pivot ? h.beta : 0.0;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const double t = B[c] - u * z[c];
        B[c] = !BRANCH && 4 * g + c == f ? xf : t;
    }
    if constexpr (BRANCH)
        if (g == gf) set_slot(B, cf, xf);
    // D <- H D H
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const double wc = L.wsc[4 * g + c];
        D[c] -= vr * wc;
        D[c] -= w * vc[c];
    }
    const bool next = !last && s + 1 + 16 * (k + 1) <= m - 2;
    if (g == 0) {
        L.vm[(k + 1) * 16 + i] = u;
        if (next) (raw + (blk + 1) * 256 + (s & 15) * 16)[ro] = u;
    }
    if (lane == 0) {
        L.tm[k + 1] = h.tau;
        L.bm[k] = h.beta;
        if (next) rtau[(blk + 1) * 16 + (s & 15)] = h.tau;
    }
    // the first rows of D (its first column, D being symmetric) and of B
    if (pivot)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            L.cm[k * 16 + 4 * g + c] = D[c];
            L.rm[k * 16 + 4 * g + c] = B[c];
        }
}

// Bulge chasing of one submatrix by nw wavefronts (this one its `wave`-th).  Step (s, k)
// needs (s, k - 1) and (s - 1, k + 1), so at time t = 2 s + k all windows of one
// parity step at once; a barrier ends each time step.  Wavefront w owns the
// windows 2 w and 2 w + 1 (mod 2 nw), so the work stays even as the band
// shortens, and ends when they have left it.  P windows per wavefront live in
// registers (16 VGPRs each), up to 16 nw P rows; MEM: those above that in device
// memory (state), which they need for the first sweeps only.
// Bound by instruction issue of the CU (about 390 vector instructions a step; with
// IEEE square root and divisions, and one row sum per column of B, it was 430).
// One window of each parity per wavefront where 16 hold them: a step's chain is the
// time step.  512-water box 21.6 -> 17.3 ms, 256 molecules 46.4 -> 32.0, one
// 1472-row matrix (every window in memory before) 14.0 -> 11.7.
template <int P, bool MEM>
__device__ __forceinline__ void chase(const BandSub &b, double *sm, int nw, int wave, const double *__restrict__ ABa,
                                      double *__restrict__ raw_all, double *__restrict__ rtau_all,
                                      double *__restrict__ d_all, double *__restrict__ e_all,
                                      double *__restrict__ state) {
    const int m = b.m;
    const int K = max((m - 1 + kBW - 1) / kBW, 1);  // windows
    const int lane = threadIdx.x % PTB_WAVE, tid = PTB_WAVE * wave + lane, NW = nw;
    ChaseLds L;
    L.vm = sm + 2;
    L.cm = L.vm + 16 * (K + 2);
    L.rm = L.cm + 16 * (K + 2);
    L.wsc = L.rm + 16 * (K + 2) + 16 * wave;
    L.tm = L.rm + 16 * (K + 2) + 16 * NW;
    L.bm = L.tm + (K + 2);
    const double *ab = ABa + b.ab;
    // the power of two that brings the largest element near 1 (see reflector_fast)
    double up = 1.0;
    {
        double big = 0.0;
        for (int l = tid; l < kABL * m; l += NW * 64)
            big = fmax(big, l / kABL + l % kABL < m ? fabs(ab[l]) : 0.0);
        big = wave_max(big);
        if (lane == 0) L.wsc[0] = big;
        __syncthreads();
        for (int w = 0; w < NW; ++w) big = fmax(big, L.wsc[16 * (w - wave)]);
        if (big > 0.0 && big < HUGE_VAL) up = ldexp(1.0, -min(max(ilogb(big), -1000), 1000));
        if (tid == 0) L.vm[-2] = 1.0 / up;
    }
    for (int l = tid; l < 16 * (K + 2); l += NW * 64) {
        L.vm[l] = 0.0;
        L.rm[l] = 0.0;
        L.cm[l] = l < 16 && l < m ? up * ab[l] : 0.0;
    }
    for (int l = tid; l < K + 2; l += NW * 64) {
        L.tm[l] = 0.0;
        L.bm[l] = l == 0 && m > kBW ? up * ab[kBW] : 0.0;
    }
    double *raw = raw_all + b.blk * 256, *rtau = rtau_all + b.blk * 16;
    double *dv = d_all + b.mapoff, *ev = e_all + b.mapoff;
    const int i = lane & 15, g = lane >> 4;
    auto load_window = [&](int k, double (&D)[4], double (&B)[4]) {
        const int r = 1 + 16 * k + ((i - 1) & 15);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int cl = 1 + 16 * k + ((4 * g + c - 1) & 15);
            const int lo = min(r, cl), hi = max(r, cl);
            D[c] = hi < m ? up * ab[(int64_t)lo * kABL + hi - lo] : 0.0;
            B[c] = r + 16 < m && r <= cl ? up * ab[(int64_t)cl * kABL + r + 16 - cl] : 0.0;
        }
    };
    auto active = [&](int k, int s) { return s >= 0 && s < m && (k == 0 || s + 1 + 16 * k < m); };
    // (the panel buffers are free by now)
    auto stored = [&](int k) {
        return reinterpret_cast<d4_t *>(state + b.pw) + ((int64_t)k * 64 + lane) * 2;
    };
    double D[P][4], B[P][4];
#pragma unroll
    for (int q = 0; q < P; ++q) load_window(2 * wave + 2 * NW * (q / 2) + (q & 1), D[q], B[q]);
    if constexpr (MEM)
        for (int k = 2 * wave + P * NW; k < K; k = k & 1 ? k + 2 * NW - 1 : k + 1) {
            double Dk[4], Bk[4];
            load_window(k, Dk, Bk);
            stored(k)[0] = d4_t{Dk[0], Dk[1], Dk[2], Dk[3]};
            stored(k)[1] = d4_t{Bk[0], Bk[1], Bk[2], Bk[3]};
        }
    __syncthreads();
    if (2 * wave >= K) return;
    // the last step of window 2 w: sweep m - 1 of window 0, else s + 1 + 32 w = m - 1
    const int T2 = wave == 0 ? m - 1 : m - 2 - 31 * wave;
    for (int t = 0; t <= T2; ++t) {
#pragma unroll
        for (int par = 0; par < 2; ++par) {
#pragma unroll
            for (int q = par; q < P; q += 2) {
                const int k = 2 * wave + 2 * NW * (q / 2) + par, s = t - wave - NW * (q / 2);
                if (active(k, s)) chase_step<P == 4 || MEM>(D[q], B[q], k, s, m, b.ng, L, raw, rtau, dv, ev, lane);
            }
            if constexpr (MEM)
                for (int j = P / 2; 2 * wave + par + 2 * NW * j < K; ++j) {
                    const int k = 2 * wave + par + 2 * NW * j, s = t - wave - NW * j;
                    if (!active(k, s)) break;  // (nor are the windows above)
                    const d4_t p0 = stored(k)[0], p1 = stored(k)[1];
                    double Dk[4] = {p0[0], p0[1], p0[2], p0[3]}, Bk[4] = {p1[0], p1[1], p1[2], p1[3]};
                    chase_step<true>(Dk, Bk, k, s, m, b.ng, L, raw, rtau, dv, ev, lane);
                    stored(k)[0] = d4_t{Dk[0], Dk[1], Dk[2], Dk[3]};
                    stored(k)[1] = d4_t{Bk[0], Bk[1], Bk[2], Bk[3]};
                }
            __syncthreads();
        }
    }
}

// One workgroup of the chase: the submatrices [first, first + n), 16 / n wavefronts
// each (P = 2 windows per wavefront, 4 for the ones that need them).
struct ChaseJob {
    int first, n, p;
};
// doubles of LDS of a submatrix of m rows and nw wavefronts
__host__ __device__ inline int chase_lds(int m, int nw) {
    const int K = m > kBW ? (m - 1 + kBW - 1) / kBW : 1;
    return 50 * (K + 2) + 16 * nw + 2;
}

// A small batch (submatrices of up to 1025 rows) in one launch of 16-wavefront
// workgroups, a CU each, the largest first: 1025 to 514 rows take 16 wavefronts with
// two windows of each parity, 513 to 258 16 with one, and below that 2, 4 or 8
// submatrices share a workgroup and its barriers where there are more of them than
// CUs.  The small ones run beside the large: 64 waters (192 submatrices) 5.3 ms one
// class after the other, 3.4 so; 621 single columns of 27 waters 2.3 and 1.4.
__global__ __launch_bounds__(1024) void k_chase(const BandSub *__restrict__ subs,
                                                const ChaseJob *__restrict__ jobs,
                                                const double *__restrict__ ABa,
                                                double *__restrict__ raw_all,
                                                double *__restrict__ rtau_all,
                                                double *__restrict__ d_all,
                                                double *__restrict__ e_all) {
    extern __shared__ double sm[];
    const ChaseJob jb = jobs[blockIdx.x];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PTB_WAVE);
    const int nw = jb.n == 1 ? 16 : jb.n == 2 ? 8 : jb.n <= 4 ? 4 : 2;
    const int x = wave / nw;
    if (x >= jb.n) return;
    const BandSub b = subs[jb.first + x];
    double *lds = sm + x * chase_lds(subs[jb.first].m, nw);
    if (jb.p == 4) chase<4, false>(b, lds, 16, wave, ABa, raw_all, rtau_all, d_all, e_all, nullptr);
    else chase<2, false>(b, lds, nw, wave % nw, ABa, raw_all, rtau_all, d_all, e_all, nullptr);
}

// One size class of a large batch, a workgroup of NW wavefronts per submatrix: the
// smaller workgroups start as wavefronts before them end, which a chip full of each
// class gains more from than from the overlap of classes (256 molecules 32 ms, 40 in
// k_chase; C400H802 2.5 and 2.8).
template <int NW, int P>
__global__ __launch_bounds__(NW * 64) void k_chase_class(const BandSub *__restrict__ subs,
                                                         const double *__restrict__ ABa,
                                                         double *__restrict__ raw_all,
                                                         double *__restrict__ rtau_all,
                                                         double *__restrict__ d_all,
                                                         double *__restrict__ e_all) {
    extern __shared__ double sm[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PTB_WAVE);
    chase<P, false>(subs[blockIdx.x], sm, NW, wave, ABa, raw_all, rtau_all, d_all, e_all, nullptr);
}

// Submatrices of 1026 to 2048 rows, a workgroup of 16 wavefronts each.
__global__ __launch_bounds__(1024) void k_chase_mem(const BandSub *__restrict__ subs,
                                                    const double *__restrict__ ABa,
                                                    double *__restrict__ raw_all,
                                                    double *__restrict__ rtau_all,
                                                    double *__restrict__ d_all,
                                                    double *__restrict__ e_all,
                                                    double *__restrict__ state) {
    extern __shared__ double sm[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PTB_WAVE);
    chase<2, true>(subs[blockIdx.x], sm, 16, wave, ABa, raw_all, rtau_all, d_all, e_all, state);
}

// ---- application of Q2 ---------------------------------------------------------

// Factors of every block of 16 reflectors: V, the block's 31 x 16 parallelogram
// (reflector j at rows j .. j + 15), and -(V T), T its WY factor, both 32 x 16 by
// rows (V at fac, -(V T) at fac + 512).  Reflectors that the chase never made
// (past the last sweep or window) are zero.  One wavefront per block, kPrepBlk
// blocks each.  grid: (submatrix, ceil(blocks / (4 kPrepBlk)))
constexpr int kPrepBlk = 4;
__global__ __launch_bounds__(256, 4) void k_q2_prep(const BandSub *__restrict__ subs,
                                                 const double *__restrict__ raw_all,
                                                 const double *__restrict__ rtau_all,
                                                 double *__restrict__ fac_all) {
    const BandSub d = subs[blockIdx.x];
    const int lane = threadIdx.x % PTB_WAVE, wave = threadIdx.x / PTB_WAVE;
    const int lr = lane & 15, g = lane >> 4;
    __shared__ double gsh[4][16][18], vsh[4][16][17], ths[4][16][17];
    double (*gs)[18] = gsh[wave], (*vs)[17] = vsh[wave];
    const int nblk = d.ng * (d.ng + 1) / 2;
    for (int u = 0; u < kPrepBlk; ++u) {
        const int bi = (blockIdx.y * 4 + wave) * kPrepBlk + u;
        if (bi >= nblk) return;
        // group G of block bi: the last with base(G) <= bi
        int G = 0;
        {
            const double t = 2.0 * d.ng + 1.0;
            G = (int)((t - sqrt(fmax(t * t - 8.0 * bi, 0.0))) * 0.5);
            while (G > 0 && q2_block(d.ng, G, 0) > bi) --G;
            while (G + 1 < d.ng && q2_block(d.ng, G + 1, 0) <= bi) ++G;
        }
        const int k = bi - (int)q2_block(d.ng, G, 0);
        const int64_t blk = d.blk + bi;
        const double *raw = raw_all + blk * 256;
        double *fac = fac_all + blk * 1024;
        // reflector 16 G + j exists for j < nv
        const int nv = min(16, min(d.m - 2 - 16 * G, d.m - 2 - 16 * (G + k)));
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int j = 4 * q + g;
            const double v = raw[j * 16 + lr];
            vs[j][lr] = j < nv ? v : 0.0;
        }
        double tj = lr < nv ? rtau_all[blk * 16 + lr] : 0.0;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        // Gram matrix: V(row, refl) = vs[refl][row - refl]
        d4_t acc = d4_t{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            const int rel = 4 * ks + g - lr;
            const double x = vs[lr][rel & 15];
            const double v = (rel >= 0 && rel < 16) ? x : 0.0;
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(v, v, acc, 0, 0, 0);
            fac[(4 * ks + g) * 16 + lr] = v;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) gs[4 * r + g][lr] = acc[r];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        // T(i, j) = -tau_j sum_{i <= c < j} T(i, c) G(c, j), T(j, j) = tau_j:
        // lane i + 16 g holds row i, columns 4 g .. 4 g + 3 (G is symmetric:
        // row j of it supplies column j)
        double t[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
        for (int jg = 0; jg < 4; ++jg)
#pragma unroll
            for (int jq = 0; jq < 4; ++jq) {
                const int j = 4 * jg + jq;
                const double tauj = read_lane(tj, j);
                double s = 0.0;
#pragma unroll
                for (int q = 0; q < 4; ++q) s += t[q] * gs[j][4 * g + q];  // t is zero past column j
                s = rows_sum(s);
                const double v = lr == j ? tauj : lr < j ? -tauj * s : 0.0;
                t[jq] = g == jg ? v : t[jq];
            }
#pragma unroll
        for (int q = 0; q < 4; ++q) ths[wave][lr][4 * g + q] = t[q];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        // V T(row, refl) = sum_c V(row, c) T(c, refl)
        d4_t o0 = d4_t{0.0, 0.0, 0.0, 0.0}, o1 = o0;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const int c = 4 * ks + g;
            const double tc = -ths[wave][c][lr];
            const int e0 = lr - c, e1 = 16 + lr - c;
            const double x0 = vs[c][e0 & 15], x1 = vs[c][e1 & 15];
            o0 = __builtin_amdgcn_mfma_f64_16x16x4f64(e0 >= 0 ? x0 : 0.0, tc, o0, 0, 0, 0);
            o1 = __builtin_amdgcn_mfma_f64_16x16x4f64(e1 < 16 ? x1 : 0.0, tc, o1, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            fac[512 + (4 * r + g) * 16 + lr] = o0[r];
            fac[768 + (4 * r + g) * 16 + lr] = o1[r];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
}

constexpr int kQ2Groups = 4;  // sweep groups per pass of k_q2_apply, a wavefront each

constexpr int64_t kQ2Wide = 2;  // 32-column jobs per CU from which they are taken (what a CU holds)

// A chunk of columns of one submatrix's right-hand sides (m = 0: none).
struct Q2Job {
    int64_t y;    // first element (row 0 of the first column)
    int64_t blk;  // the submatrix's first block
    int m, ld, ng, nc;
};

// Y <- Q2 Y (TRANS false: groups descending, windows ascending) or Q2^T Y (the
// reverse) for up to 16 CT columns per workgroup.  The 32 rows a block touches sit
// in registers as two 16 x 16 tiles per 16 columns, in the layout in which
// v_mfma_f64_16x16x4 takes its B operand and leaves its result, so nothing moves
// between the two products of a block; the next block shares one tile.  The
// matrix instruction's row 4 r + g (register r, lane group g) stands for row
// 4 g + r of the tile, so a lane's four values are four consecutive rows (two
// 16-byte accesses), and for reflector 4 g + r between the products, so the
// second factor is read 32 bytes per lane.
//
// kQ2Groups groups run in one pass over the rows, a wavefront each: a wavefront
// keeps the tile that its next block shares, hands the finished one to the next
// wavefront through LDS (the last one stores it) and takes a new one from the
// wavefront before (the first one loads it), one barrier per step.  So a job's
// chain is a quarter of its blocks long and every SIMD of a CU has one of its
// wavefronts.  Against one wavefront per job that takes the four groups in turn:
// one 1472-row matrix, all columns, 3.57 -> 1.27 ms; both applications of 64 waters
// 2.67 -> 1.21, C400H802 2.9 -> 0.9, 8 waters 0.23 -> 0.08, the 512-water box (whose
// products alone fill the matrix cores for 5.5 ms) 15.0 -> 13.1.
// Factors and the first wavefront's tiles are fetched three steps ahead.
template <bool TRANS, int CT>
__global__ __launch_bounds__(256, 2) void k_q2_apply(const Q2Job *__restrict__ jobs,
                                                     const double *__restrict__ fac_all,
                                                     double *__restrict__ Ya) {
    typedef double d2u_t __attribute__((ext_vector_type(2), aligned(8)));
    constexpr int Q = kQ2Groups, S = 3;
    __shared__ d2_t hand[2][Q - 1][CT][2][PTB_WAVE];
    const int h = __builtin_amdgcn_readfirstlane(threadIdx.x / PTB_WAVE);
    const Q2Job jb = jobs[blockIdx.x];
    if (jb.m == 0) return;
    const int lane = threadIdx.x % PTB_WAVE, lr = lane & 15, g = lane >> 4;
    const int m = jb.m, ng = jb.ng;
    double *y[CT];
    bool cok[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) {
        cok[c] = 16 * c + lr < jb.nc;
        y[c] = Ya + jb.y + (int64_t)min(16 * c + lr, jb.nc - 1) * jb.ld + 1 + 4 * g;
    }
    // tile t: rows 16 t + 1 .. 16 t + 16, cut at m
    auto load = [&](int t, d4_t (&x)[CT]) {
        if (16 * t + 17 <= m) {
#pragma unroll
            for (int c = 0; c < CT; ++c) {
                const d2u_t *p = reinterpret_cast<const d2u_t *>(y[c] + 16 * t);
                const d2u_t u = p[0], v = p[1];
                x[c] = d4_t{u[0], u[1], v[0], v[1]};
            }
        } else {
#pragma unroll
            for (int c = 0; c < CT; ++c)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int row = 16 * t + 1 + 4 * g + r;
                    const double v = y[c][min(row, m - 1) - 1 - 4 * g];
                    x[c][r] = row < m ? v : 0.0;
                }
        }
    };
    auto store = [&](int t, const d4_t (&x)[CT]) {
        if (16 * t + 17 <= m) {
#pragma unroll
            for (int c = 0; c < CT; ++c)
                if (cok[c]) {
                    d2u_t *p = reinterpret_cast<d2u_t *>(y[c] + 16 * t);
                    p[0] = d2u_t{x[c][0], x[c][1]};
                    p[1] = d2u_t{x[c][2], x[c][3]};
                }
        } else {
#pragma unroll
            for (int c = 0; c < CT; ++c)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (16 * t + 1 + 4 * g + r < m && cok[c]) y[c][16 * t + r] = x[c][r];
        }
    };
    // block (G, k)'s operands: f1 (reflectors x rows, slice s: row 4 g + s of the
    // low and the high tile), f2 (rows x reflectors, slice s: reflector 4 g + s)
    const int pr = 4 * (lr & 3) + (lr >> 2);
    const double *f1a = fac_all + jb.blk * 1024 + (TRANS ? 512 : 0) + 64 * g + pr;
    const double *f2a = fac_all + jb.blk * 1024 + (TRANS ? 0 : 512) + 16 * pr + 4 * g;
    struct Fac {
        double f1[8], f2[8];
    };
    auto fetch = [&](int64_t b, Fac &f) {
        const double *p1 = f1a + b * 1024;
        const d2_t *p2 = reinterpret_cast<const d2_t *>(f2a + b * 1024);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            f.f1[s] = p1[16 * s];
            f.f1[4 + s] = p1[256 + 16 * s];
        }
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const d2_t v = p2[128 * q + s];
                f.f2[4 * q + 2 * s] = v[0];
                f.f2[4 * q + 2 * s + 1] = v[1];
            }
    };
    Fac F[S];
    d4_t X[S][CT];  // the first wavefront's tiles
    d4_t keep[CT];
    const int npass = (ng + Q - 1) / Q;
    for (int pass = 0; pass < npass; ++pass) {
        // the pass' first group; wavefront h takes the h-th one after it
        const int A = TRANS ? Q * pass : ng - 1 - Q * pass;
        const int nq = min(Q, TRANS ? ng - A : A + 1);
        const bool on = h < nq;
        const int G = !on ? 0 : TRANS ? A + h : A - h;
        const int nb = ng - G;  // its blocks
        // Block j of group G (window j, TRANS: from the top) is step j + lag.  It
        // needs the tile that the wavefront before finished one step earlier: in
        // its block j, TRANS: j + 1
        const int lag = TRANS ? 2 * h : h;
        const int steps = TRANS ? ng - A + nq - 1 : ng - A + 2 * nq - 1;
        auto tile_in = [&](int j) { return TRANS ? ng - 1 - j : G + j + 1; };
        auto get = [&](int j, Fac &f) {
            const int jc = min(max(j, 0), nb - 1);
            fetch(q2_block(ng, G, TRANS ? nb - 1 - jc : jc), f);
        };
        if (on) {
            if (h == 0)
                [&]<int... U>(std::integer_sequence<int, U...>) {
                    ((U < nb ? load(tile_in(U), X[U]) : (void)0), ...);
                }(std::make_integer_sequence<int, S>{});
            if (!TRANS) load(G, keep);
            else if (h == 0) load(ng, keep);
            get(-lag, F[0]);
            get(1 - lag, F[1]);
            get(2 - lag, F[2]);
        }
        auto step = [&](auto U, int t) {
            constexpr int u = decltype(U)::value;
            const int j = t - lag;
            auto take = [&](d4_t (&x)[CT]) {
#pragma unroll
                for (int c = 0; c < CT; ++c) {
                    const d2_t a = hand[(t - 1) & 1][h - 1][c][0][lane], b = hand[(t - 1) & 1][h - 1][c][1][lane];
                    x[c] = d4_t{a[0], a[1], b[0], b[1]};
                }
            };
            auto pass_on = [&](int tile, const d4_t (&x)[CT]) {
                if (h == nq - 1) {
                    store(tile, x);
                    return;
                }
#pragma unroll
                for (int c = 0; c < CT; ++c) {
                    hand[t & 1][h][c][0][lane] = d2_t{x[c][0], x[c][1]};
                    hand[t & 1][h][c][1][lane] = d2_t{x[c][2], x[c][3]};
                }
            };
            if (on) {
                if (j >= 0 && j < nb) {
                    if (h > 0) take(X[u]);
                    Fac &f = F[u];
                    d4_t done[CT];
#pragma unroll
                    for (int c = 0; c < CT; ++c) {
                        d4_t &lo = TRANS ? X[u][c] : keep[c], &hi = TRANS ? keep[c] : X[u][c];
                        d4_t w = d4_t{0.0, 0.0, 0.0, 0.0};
#pragma unroll
                        for (int r = 0; r < 4; ++r) w = __builtin_amdgcn_mfma_f64_16x16x4f64(f.f1[r], lo[r], w, 0, 0, 0);
#pragma unroll
                        for (int r = 0; r < 4; ++r) w = __builtin_amdgcn_mfma_f64_16x16x4f64(f.f1[4 + r], hi[r], w, 0, 0, 0);
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            lo = __builtin_amdgcn_mfma_f64_16x16x4f64(f.f2[r], w[r], lo, 0, 0, 0);
                            hi = __builtin_amdgcn_mfma_f64_16x16x4f64(f.f2[4 + r], w[r], hi, 0, 0, 0);
                        }
                        done[c] = keep[c];
                        keep[c] = X[u][c];
                    }
                    pass_on(TRANS ? ng - j : G + j, done);
                    if (h == 0 && j + S < nb) load(tile_in(j + S), X[u]);
                    if (TRANS && j == nb - 1) store(G, keep);
                } else if (TRANS && j == -1) {
                    take(keep);  // (h > 0: the top tile)
                } else if (!TRANS && j == nb) {
                    pass_on(ng, keep);
                }
                get(j + S, F[u]);
            }
            __syncthreads();
        };
        for (int t = 0; t < steps; t += S)
            [&]<int... U>(std::integer_sequence<int, U...>) {
                ((t + U < steps ? step(std::integral_constant<int, U>{}, t + U) : (void)0), ...);
            }(std::make_integer_sequence<int, S>{});
    }
}

}  // namespace

namespace ptb {

int64_t band_blocks(int m) {
    const int64_t ng = q2_groups(m);
    return ng * (ng + 1) / 2;
}

int64_t band_parts(int m) {
    const int64_t ns = m > kBW ? (m - kBW + 63) / 64 : 0;
    return gram_at(m) + 1024 * ns;
}

int sytrd_band(ptbgpu_ctx *ctx, const std::vector<SubDesc> &desc, double *A, double *d, double *e,
               double *tau, QFactor &qf) {
    const int nsm = (int)desc.size();
    qf.q2blk.assign(nsm, -1);
    qf.q2fac = nullptr;
    std::vector<int> order;
    for (int s = 0; s < nsm; ++s)
        if (desc[s].flags & kSubBand) order.push_back(s);
    const int nb = (int)order.size();
    if (nb == 0) return PTBGPU_OK;
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return desc[a].m > desc[b].m; });
    std::vector<BandSub> subs(nb);
    int64_t pw = 0, px = 0, ab = 0, blk = 0;
    for (int i = 0; i < nb; ++i) {
        const SubDesc &x = desc[order[i]];
        subs[i] = {x.off, pw, px, ab, blk, x.m, x.ld, x.mapoff, q2_groups(x.m)};
        qf.q2blk[order[i]] = blk;
        pw += (int64_t)x.ld * 64 + 256;
        px += band_parts(x.m);
        ab += ((int64_t)x.m * kABL + 15) & ~15;
        blk += band_blocks(x.m);
    }
    auto *PW = static_cast<double *>(ws(ctx, "band_pw", sizeof(double) * pw));
    auto *PX = static_cast<double *>(ws(ctx, "band_px", sizeof(double) * std::max<int64_t>(px, 1)));
    auto *AB = static_cast<double *>(ws(ctx, "band_ab", sizeof(double) * ab));
    auto *raw = static_cast<double *>(ws(ctx, "band_q2raw", sizeof(double) * 256 * std::max<int64_t>(blk, 1)));
    auto *rtau = static_cast<double *>(ws(ctx, "band_q2tau", sizeof(double) * 16 * std::max<int64_t>(blk, 1)));
    auto *fac = static_cast<double *>(ws(ctx, "band_q2fac", sizeof(double) * 1024 * std::max<int64_t>(blk, 1)));
    if (!PW || !PX || !AB || !raw || !rtau || !fac) return PTBGPU_E_NOMEM;
    if (ctx->poison_arenas && !ctx->capturing) {  // all bytes 0xff: NaN
        const std::pair<void *, int64_t> bufs[] = {{PW, pw}, {PX, px}, {AB, ab}, {raw, 256 * blk}, {rtau, 16 * blk},
                                                   {fac, 1024 * blk}};
        for (const auto &[p, n] : bufs) PTB_HIP(ctx, hipMemsetAsync(p, 0xff, sizeof(double) * n, ctx->stream));
    }
    auto *ds = static_cast<BandSub *>(upload_table(ctx, "band_subs", subs.data(), sizeof(BandSub) * nb));
    if (!ds) return PTBGPU_E_NOMEM;
    qf.q2fac = fac;
    hipStream_t st = ctx->stream;
    const int max_m = subs[0].m;
    // submatrices (largest first) of at least `rows` rows
    auto count = [&](int rows) {
        return (int)(std::partition_point(subs.begin(), subs.end(), [&](const BandSub &x) { return x.m >= rows; }) -
                     subs.begin());
    };
    // panels: at least two rows below the band
    const int npanel = max_m >= kBW + 2 ? (max_m - kBW - 2) / kBW + 1 : 0;
    {
        ProfScope prof_(ctx, "band_reduce");
        for (int p = 0; p < npanel; ++p) {
            const int r0 = (p + 1) * kBW, na = count(r0 + 2);
            const int n = max_m - r0;  // the tallest panel
            {
                ProfScope kprof_(ctx, "band_qr");
                const int big = count(r0 + 1025);  // panels of more than 1024 rows
                if (big > 0)
                    hipLaunchKernelGGL((k_band_qr<512, 4>), dim3(big), dim3(512), 0, st, ds, A, PW, AB, tau, 0, p);
                const int nl = big < na ? subs[big].m - r0 : 0;
                if (nl > 512)
                    hipLaunchKernelGGL((k_band_qr<256, 4>), dim3(na - big), dim3(256), 0, st, ds, A, PW, AB, tau, big, p);
                else if (nl > 256)
                    hipLaunchKernelGGL((k_band_qr<256, 2>), dim3(na - big), dim3(256), 0, st, ds, A, PW, AB, tau, big, p);
                else if (nl > 0)
                    hipLaunchKernelGGL((k_band_qr<256, 1>), dim3(na - big), dim3(256), 0, st, ds, A, PW, AB, tau, big, p);
                PTB_CHECK_LAUNCH(ctx);
            }
            const int ns = (n + 63) / 64;
            const bool split = na <= ctx->num_cus;
            {
                ProfScope kprof_(ctx, "band_step");
                const int nunit = band_units(ns);
                // (a grid holds fewer than 2^32 threads: 116 504 submatrices, if one of
                // them has 2048 rows)
                const int most = (int)(((int64_t)1 << 32) / 256 - 1) / nunit / 8 * 8;
                for (int f = 0; f < na; f += most) {
                    const int nf = std::min(na - f, most);
                    const dim3 grid((unsigned)((nf + 7) / 8 * 8 * nunit));
                    if (p == 0)
                        hipLaunchKernelGGL(k_band_step<false>, grid, dim3(256), 0, st, ds + f, nf, A, PW, PX, p, nunit);
                    else
                        hipLaunchKernelGGL(k_band_step<true>, grid, dim3(256), 0, st, ds + f, nf, A, PW, PX, p, nunit);
                    PTB_CHECK_LAUNCH(ctx);
                }
            }
            {
                ProfScope kprof_(ctx, "band_x");
                hipLaunchKernelGGL(split ? k_band_x<true> : k_band_x<false>, dim3(na, ns), dim3(256), 0, st, ds, PX, PW, p);
                PTB_CHECK_LAUNCH(ctx);
            }
            {
                ProfScope kprof_(ctx, "band_w");
                hipLaunchKernelGGL(split ? k_band_w<true> : k_band_w<false>, dim3(na, split ? ns : 1), dim3(256), 0, st, ds,
                                   A, PW, PX, p);
                PTB_CHECK_LAUNCH(ctx);
            }
        }
        hipLaunchKernelGGL(k_band_extract, dim3(nb, (max_m + kBW - 1) / kBW), dim3(256), 0, st, ds, A, AB,
                           kQBlk);
        PTB_CHECK_LAUNCH(ctx);
    }
    {
        ProfScope prof_(ctx, "band_chase");
        const int big = count(1026);
        if (big > 0) {
            hipLaunchKernelGGL(k_chase_mem, dim3(big), dim3(1024), sizeof(double) * (size_t)chase_lds(max_m, 16),
                               st, ds, AB, raw, rtau, d, e, PW);
            PTB_CHECK_LAUNCH(ctx);
        }
        std::vector<ChaseJob> jobs;
        int words = 0;
        for (int i = big; i < nb;) {
            const int m = subs[i].m;
            const int most = nb - big <= ctx->num_cus || m > 257 ? 1 : m > 129 ? 2 : m > 65 ? 4 : 8;
            const int n = std::min(most, nb - i), nw = n == 1 ? 16 : n == 2 ? 8 : n <= 4 ? 4 : 2;
            jobs.push_back({i, n, m > 513 ? 4 : 2});
            words = std::max(words, n * chase_lds(m, nw));
            i += n;
        }
        if (jobs.size() <= 2 * (size_t)ctx->num_cus) {
            if (!jobs.empty()) {
                auto *dj = static_cast<ChaseJob *>(
                    upload_table(ctx, "band_chase", jobs.data(), sizeof(ChaseJob) * jobs.size()));
                if (!dj) return PTBGPU_E_NOMEM;
                hipLaunchKernelGGL(k_chase, dim3((unsigned)jobs.size()), dim3(1024), sizeof(double) * (size_t)words,
                                   st, ds, dj, AB, raw, rtau, d, e);
                PTB_CHECK_LAUNCH(ctx);
            }
        } else {
            int done = big;
            auto run = [&](int nw, int low, auto kern) {
                const int to = count(low);
                if (to > done)
                    hipLaunchKernelGGL(kern, dim3(to - done), dim3(nw * 64),
                                       sizeof(double) * (size_t)chase_lds(subs[done].m, nw), st, ds + done, AB, raw,
                                       rtau, d, e);
                done = std::max(done, to);
            };
            run(16, 514, k_chase_class<16, 4>);
            run(16, 258, k_chase_class<16, 2>);
            run(8, 130, k_chase_class<8, 2>);
            run(4, 66, k_chase_class<4, 2>);
            run(2, 0, k_chase_class<2, 2>);
            PTB_CHECK_LAUNCH(ctx);
        }
    }
    if (blk > 0) {
        ProfScope prof_(ctx, "q2_prep");
        const int nblk = (int)band_blocks(max_m);
        hipLaunchKernelGGL(k_q2_prep, dim3(nb, (nblk + 4 * kPrepBlk - 1) / (4 * kPrepBlk)), dim3(256), 0, st,
                           ds, raw, rtau, fac);
        PTB_CHECK_LAUNCH(ctx);
    }
    return PTBGPU_OK;
}

int apply_q2(ptbgpu_ctx *ctx, const std::vector<SubDesc> &desc, const QFactor &qf, double *Y,
             const std::vector<int64_t> &yoff, const std::vector<int> &ncols, bool trans,
             const char *tag) {
    if (!qf.q2fac) return PTBGPU_OK;
    ProfScope prof_(ctx, "apply_q2");
    // two 16-column tiles per workgroup (each factor feeds both) where that leaves
    // kQ2Wide workgroups per CU, else one; one for a last piece of at most 16
    int64_t pairs = 0;
    for (int s = 0; s < (int)desc.size(); ++s)
        if (qf.q2blk[s] >= 0) pairs += (ncols[s] + 31) / 32;
    const int step = pairs >= kQ2Wide * (int64_t)ctx->num_cus ? 32 : 16;
    std::vector<int> order;
    for (int s = 0; s < (int)desc.size(); ++s)
        if (qf.q2blk[s] >= 0 && desc[s].m >= 3 && ncols[s] > 0) order.push_back(s);
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return desc[a].m > desc[b].m; });
    // largest submatrices first, each one's jobs on one XCD (whose L2 holds its
    // factors): entry 8 k + x is XCD x's k-th job
    auto run = [&](const char *nm, bool two) -> int {
        std::vector<Q2Job> q[8];
        for (int s : order) {
            const SubDesc &x = desc[s];
            int to = 0;
            for (int i = 1; i < 8; ++i)
                if (q[i].size() < q[to].size()) to = i;
            for (int c = 0; c < ncols[s]; c += step) {
                const int nc = std::min(step, ncols[s] - c);
                if ((nc > 16) != two) continue;
                q[order.size() < 8 ? (c / step) & 7 : to].push_back(
                    {yoff[s] + (int64_t)c * x.ld, qf.q2blk[s], x.m, x.ld, q2_groups(x.m), nc});
            }
        }
        size_t len = 0;
        for (const auto &l : q) len = std::max(len, l.size());
        if (len == 0) return PTBGPU_OK;
        std::vector<Q2Job> jobs(8 * len, Q2Job{});
        for (int x = 0; x < 8; ++x)
            for (size_t k = 0; k < q[x].size(); ++k) jobs[8 * k + x] = q[x][k];
        auto *dj = static_cast<Q2Job *>(
            upload_table(ctx, (std::string(nm) + tag).c_str(), jobs.data(), sizeof(Q2Job) * jobs.size()));
        if (!dj) return PTBGPU_E_NOMEM;
        auto kern = two ? (trans ? k_q2_apply<true, 2> : k_q2_apply<false, 2>)
                        : (trans ? k_q2_apply<true, 1> : k_q2_apply<false, 1>);
        hipLaunchKernelGGL(kern, dim3((unsigned)jobs.size()), dim3(256), 0, ctx->stream, dj, qf.q2fac, Y);
        PTB_CHECK_LAUNCH(ctx);
        return PTBGPU_OK;
    };
    PTB_TRY(run("q2_jw_", true));
    return run("q2_jn_", false);
}

}  // namespace ptb
