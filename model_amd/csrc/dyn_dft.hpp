// Transforms as products with the matrices of their cosines and sines on the FP64 matrix units: lengths with
// a prime factor above 5 up to kDftMax, and smooth lengths up to dft_x_smooth() (along i) and kDftYSmooth (along j),
// on the grids that pressure_init gives them to (all of these in FP64, fewer in FP32).
//
// A length-n transform needs only rows 0 .. n/2 of the cosine matrix C and the sine matrix S once its input
// is folded into sums and differences of mirrored elements, E(i) = x(i) + x(n-i), D(i) = x(i) - x(n-i):
//   real x:     Re X(m) = (C E)(m), Im X(m) = -(S D)(m), m = 0 .. n/2;
//   complex x:  X(m) = (C E)(m) -+ i (S D)(m), X(n-m) = (C E)(m) +- i (S D)(m)
// and the real inverse is the same two products of the half spectrum's real and imaginary parts.  C and S
// are (n/2+1) x (n/2+1) and symmetric.  The levels (and rows, and real and imaginary parts) of the other
// dimensions are the columns of the right operand, so the work is a contraction: n^2/2 multiply-adds per
// real line in 16x16x4 FP64 tiles whatever the factors of n, in one pass over LDS instead of one per radix.
// Sums run in FP64 in both forms.
//
// Measured, us of the i transforms (forward with the divergence, then inverse): against direct sums over the
// prime factors, 194x100x40 FP32 moist 194 + 185 -> 14.5 + 12.6, 251x251x94 FP64 2214 + 2166 -> 73 + 51; against
// the radix passes of smooth lengths, FP64 64x64x40 20.6 + 18.7 -> 7.3 + 8.3, 192x192x40 42.2 + 33.4 -> 19.4 +
// 17.1, 384x384x80 238 + 171 -> 211 + 141; FP32 64x64x40 14.9 + 14.2 -> 7.5 + 7.9.  The work grows with n where the
// passes' grows with log n, and FP32 passes move half the bytes, so FP32 changes over between 192 points (27.3 + 23.7
// against 22.5 + 18.1 by products, 40 levels) and 256 (33.1 + 28.3 against 52.7 + 38.2, 64 levels).
#pragma once

#include <cmath>
#include <vector>

#include "dyn_internal.hpp"

namespace dyn {
namespace {

// smooth lengths that may take the matrix products: measured faster up to these
template <typename T>
constexpr int dft_x_smooth() { return sizeof(T) == 4 ? 192 : 384; }
constexpr int kDftYSmooth = 192, kDftYThree = 112;

constexpr int kDftMax = 511;  // 256 matrix rows: 16 tiles, one per wavefront of the largest block
typedef double dvec4 __attribute__((ext_vector_type(4)));

// rows of the matrices, padded to whole tiles
__host__ __device__ __forceinline__ int dft_rows(int n) { return n / 2 + 1; }
__host__ __device__ __forceinline__ int dft_pad(int n) { return (dft_rows(n) + 15) & ~15; }
// columns per row of the LDS operands: rows 128 bytes apart modulo 256, so that the two rows a
// half-wavefront reads fall into different banks
__host__ __device__ __forceinline__ int dft_pitch(int nc) { return nc | 16; }
inline size_t dft_lds(int n, int nc) { return 2 * (size_t)((dft_rows(n) + 3) & ~3) * dft_pitch(nc) * sizeof(double); }

// threads of the largest block with NT column tiles: 80 KiB of operands hold 64 matrix rows with 4 tiles and
// 104 with 2 (dft_tiles)
constexpr int dft_bound(int nt) { return nt == 4 ? 256 : nt == 2 ? 512 : 1024; }

// C and S of length n on the host: dft_pad x dft_pad each, zero outside dft_rows
inline std::vector<double> dft_matrices(int n) {
    const int h = dft_rows(n), p = dft_pad(n);
    std::vector<double> t(2 * (size_t)p * p, 0.0);
    std::vector<double> cs(n), sn(n);
    for (int e = 0; e < n; e++) {  // the angles at which a cosine or sine vanishes are kept exact
        const double x = 2.0 * kTrigPi * (double)e / (double)n;
        cs[e] = 4 * e == n || 4 * e == 3 * n ? 0.0 : std::cos(x);
        sn[e] = e == 0 || 2 * e == n ? 0.0 : std::sin(x);
    }
    for (int a = 0; a < h; a++)
        for (int b = 0; b < h; b++) {
            const int e = (int)((long long)a * b % n);
            t[(size_t)a * p + b] = cs[e];
            t[(size_t)p * p + (size_t)a * p + b] = sn[e];
        }
    return t;
}

// The two products for one tile of 16 rows (m0 ..) and NT tiles of 16 columns: C E into c, S D into s.
// Matrix fragments come from L2 (each wavefront reads its tile's rows once), kDftU steps ahead of their use;
// the folded operands from LDS.  Of a 16x16x4 tile a lane holds A(lane % 16, lane / 16), B(lane / 16,
// lane % 16) and results (lane / 16 + 4 v, lane % 16), v = 0 .. 3.
constexpr int kDftU = 2;
template <int NT>
__device__ __forceinline__ void dft_products(const double *__restrict__ tab, int n, int m0, const double *E, const double *D, int pitch,
                                             dvec4 (&c)[NT], dvec4 (&s)[NT]) {
    const int p = dft_pad(n), steps = (dft_rows(n) + 3) / 4;
    const int lane = threadIdx.x & 63, row = lane >> 4, col = lane & 15;
    const double *ca = tab + (size_t)row * p + m0 + col, *sa = ca + (size_t)p * p;  // C(k, m) = C(m, k)
    const double *e = E + row * pitch + col, *d = D + row * pitch + col;
#pragma unroll
    for (int t = 0; t < NT; t++) {
        c[t] = dvec4{0.0, 0.0, 0.0, 0.0};
        s[t] = dvec4{0.0, 0.0, 0.0, 0.0};
    }
    double ac[2][kDftU], as[2][kDftU];
    auto fetch = [&](int k, double (&fc)[kDftU], double (&fs)[kDftU]) {
#pragma unroll
        for (int u = 0; u < kDftU; u++) {
            const size_t o = (size_t)min(k + u, steps - 1) * 4 * p;
            fc[u] = ca[o];
            fs[u] = sa[o];
        }
    };
    auto use = [&](int k, const double (&fc)[kDftU], const double (&fs)[kDftU]) {
#pragma unroll
        for (int u = 0; u < kDftU; u++) {
            if (k + u >= steps) break;
            const int o = (k + u) * 4 * pitch;
#pragma unroll
            for (int t = 0; t < NT; t++) {
                c[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(fc[u], e[o + 16 * t], c[t], 0, 0, 0);
                s[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(fs[u], d[o + 16 * t], s[t], 0, 0, 0);
            }
        }
    };
    fetch(0, ac[0], as[0]);
    for (int k = 0; k < steps; k += 2 * kDftU) {
        fetch(k + kDftU, ac[1], as[1]);
        use(k, ac[0], as[0]);
        fetch(k + 2 * kDftU, ac[0], as[0]);
        use(k + kDftU, ac[1], as[1]);
    }
}

// The mass divergence over step * dt of one cell from the winds on its six faces (pressure.cpp:1390-1406), in T.
// The fluxes through a face cancel between its two cells only if they are rounded alike, and what FP32 leaves over,
// the solve amplifies most in the longest waves: with a matrix product in either horizontal pass the arithmetic is
// therefore in 64 bits (T = double) for FP32 fields too (pi of 194x100x40 moist after 4 steps, against a 64-bit run:
// 2e-6 to 1e-5 off by the seed with FP32 arithmetic here).  Factored FP32 transforms of both sides round
// by more of their own and keep FP32.
template <typename T>
struct DivStep {
    T odx, ody, odz, sdt;
    __device__ __forceinline__ DivStep(const Geo &g, double step)
        : odx(T(g.one_d_dx)), ody(T(g.one_d_dy)), odz(T(g.one_d_dz)), sdt(T(step * g.dt)) {}
    __device__ __forceinline__ T operator()(double rhou, double rw1, double rw0, double mu, T ue, T uw, T vn, T vs, T wt, T wb) const {
        T d = T(rhou) * (ue - uw) * odx + T(rhou) * (vn - vs) * ody + (T(rw1) * wt - T(rw0) * wb) * (odz * T(mu));
        return d / sdt;
    }
};

// Forward along i: the divergence (as div_rfft_x_block forms it), or with SRC the ready field src(i+3, j, k)
// (the transposed solve of the adjoint), of NC = 16 NT columns (j, level), folded, and its half spectrum.
// Threads keep their column, so its coefficients and row offsets are read once.
template <typename T, int NT, bool SRC>
__device__ __forceinline__ void div_dft_x_block(const Geo &g, const Cols &c, const T *__restrict__ UP, const T *__restrict__ VP,
                                                const T *__restrict__ WP, T *__restrict__ spec, int n, const double *__restrict__ tab,
                                                int nk2, double step, const T *__restrict__ src, int block, unsigned char *smem) {
    constexpr int NC = 16 * NT;
    const int pitch = dft_pitch(NC), h = dft_rows(n), hk = (h + 3) & ~3, ncol = g.NY * nk2;
    double *E = (double *)smem, *D = E + hk * pitch;
    const int c0 = block * NC, b = threadIdx.x % NC, q = min(c0 + b, ncol - 1), j = q / nk2, k = q - j * nk2 + 1;
    const int jj = j == 0 ? 1 : (j == g.NY - 1 ? g.NY - 2 : j);  // mirrored rows, pressure.cpp:1408-1415
    const double rhou = c.rhou[k], rw1 = c.rhow[k + 1], rw0 = c.rhow[k], mu = c.mu[k];
    const DivStep<double> ds(g, step);
    const T *u = UP + (long long)jj * g.NZ + k, *v = VP + (long long)jj * g.NZ + k, *w = WP + (long long)jj * g.NZ + k;
    auto load = [&](int i, T (&f)[6]) {
        if (SRC) {
            f[0] = src[(long long)(i + 3) * g.NYNZ + (long long)j * g.NZ + k];
            return;
        }
        const int ia = i + 3, ie = ia + 1 == g.NX - 3 ? 3 : ia + 1;  // the periodic column UP(NX-3) is read as UP(3)
        f[0] = u[(long long)ie * g.NYNZ];
        f[1] = u[(long long)ia * g.NYNZ];
        f[2] = v[(long long)ia * g.NYNZ + g.NZ];
        f[3] = v[(long long)ia * g.NYNZ];
        f[4] = w[(long long)ia * g.NYNZ + 1];
        f[5] = w[(long long)ia * g.NYNZ];
    };
    auto value = [&](const T (&f)[6]) -> double {
        if (SRC) return double(f[0]);
        return ds(rhou, rw1, rw0, mu, f[0], f[1], f[2], f[3], f[4], f[5]);
    };
    const int rows = blockDim.x / NC;
    for (int i = threadIdx.x / NC; i < hk; i += 2 * rows) {
        // two rows at a time, their loads issued together (clamped rows, so none sits behind a branch)
        T x[2][6], y[2][6];
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const int ir = min(i + r * rows, h - 1);
            load(ir, x[r]);
            load(ir == 0 ? 0 : n - ir, y[r]);
        }
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const int ir = i + r * rows;
            if (ir >= hk) break;
            const double a = value(x[r]), m = value(y[r]);
            const bool self = ir == 0 || 2 * ir == n;
            E[ir * pitch + b] = ir < h ? (self ? a : a + m) : 0.0;
            D[ir * pitch + b] = ir < h && !self ? a - m : 0.0;
        }
    }
    __syncthreads();
    dvec4 pc[NT], ps[NT];
    const int lane = threadIdx.x & 63;
    for (int m0 = (threadIdx.x >> 6) * 16; m0 < h; m0 += (blockDim.x >> 6) * 16) {
        dft_products<NT>(tab, n, m0, E, D, pitch, pc, ps);
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const int qc = c0 + 16 * t + (lane & 15);
#pragma unroll
            for (int v4 = 0; v4 < 4; v4++) {
                const int m = m0 + (lane >> 4) + 4 * v4;
                if (m < h && qc < ncol) st2(spec + ((long long)m * ncol + qc) * 2, T(pc[t][v4]), T(-ps[t][v4]));
            }
        }
    }
}
template <typename T, int NT, bool SRC>
__global__ void __launch_bounds__(dft_bound(NT)) k_div_dft_x(Geo g, Cols c, const T *__restrict__ UP, const T *__restrict__ VP,
                                                             const T *__restrict__ WP, T *__restrict__ spec, int n,
                                                             const double *__restrict__ tab, int nk2, double step,
                                                             const T *__restrict__ src) {
    extern __shared__ __align__(16) unsigned char smem[];
    div_dft_x_block<T, NT, SRC>(g, c, UP, VP, WP, spec, n, tab, nk2, step, src, xcd_tile(blockIdx.x, gridDim.x), smem);
}

// Backward along i: the half spectrum's rows, weighted for their mirror images (2, and 1 for the
// self-conjugate wavenumbers, whose imaginary part is dropped), to PI with its ghost levels and periodic
// halos (pressure.cpp:878-892, boundaries.cpp:533-540).  With jhalf the half-slab j pass left row j of the full
// inverse as v0(j') + s v1(j'), j' = j mod jhalf (see irfft_x_out_block).
template <typename T, int NT>
__device__ __forceinline__ void idft_x_out_block(const Geo &g, const T *__restrict__ spec, T *__restrict__ PI, int n,
                                                 const double *__restrict__ tab, int nk2, int block, unsigned char *smem, int jhalf = 0) {
    constexpr int NC = 16 * NT;
    const int pitch = dft_pitch(NC), h = dft_rows(n), hk = (h + 3) & ~3, ncol = g.NY * nk2;
    double *E = (double *)smem, *D = E + hk * pitch;
    const int c0 = block * NC, b = threadIdx.x % NC, q = min(c0 + b, ncol - 1);
    const bool second = jhalf && q >= jhalf * nk2;
    const int q0 = second ? q - jhalf * nk2 : q;
    const T sg = second ? T(-1) : T(1);
    const int rows = blockDim.x / NC;
    for (int i = threadIdx.x / NC; i < hk; i += 4 * rows) {
        T a[4], m[4];
        if (jhalf) {
            T a1[4], m1[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const T *o = spec + ((long long)min(i + r * rows, h - 1) * ncol + q0) * 2;
                ld2(o, a[r], m[r]);
                ld2(o + 2LL * jhalf * nk2, a1[r], m1[r]);
            }
#pragma unroll
            for (int r = 0; r < 4; r++) {
                a[r] = a[r] + sg * a1[r];
                m[r] = m[r] + sg * m1[r];
            }
        } else {
#pragma unroll
            for (int r = 0; r < 4; r++) ld2(spec + ((long long)min(i + r * rows, h - 1) * ncol + q) * 2, a[r], m[r]);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int ir = i + r * rows;
            if (ir >= hk) break;
            const bool self = ir == 0 || 2 * ir == n;
            E[ir * pitch + b] = ir < h ? (self ? 1.0 : 2.0) * double(a[r]) : 0.0;
            D[ir * pitch + b] = ir < h && !self ? 2.0 * double(m[r]) : 0.0;
        }
    }
    __syncthreads();
    const int shift = g.NX - 6, lane = threadIdx.x & 63;
    auto put = [&](int ia, int j, int kk, T v) {
        const long long o = (long long)ia * g.NYNZ + (long long)j * g.NZ;
        const int ks[3] = {kk + 1, kk == 0 ? 0 : -1, kk == nk2 - 1 ? g.NZ - 1 : -1};
        for (int t = 0; t < 3; t++) {
            if (ks[t] < 0) continue;
            PI[o + ks[t]] = v;
            if (ia >= shift && ia < shift + 3) PI[o - shift * g.NYNZ + ks[t]] = v;
            if (ia >= 3 && ia < 6) PI[o + shift * g.NYNZ + ks[t]] = v;
        }
    };
    dvec4 pc[NT], ps[NT];
    for (int m0 = (threadIdx.x >> 6) * 16; m0 < h; m0 += (blockDim.x >> 6) * 16) {
        dft_products<NT>(tab, n, m0, E, D, pitch, pc, ps);
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const int qc = c0 + 16 * t + (lane & 15);
            if (qc >= ncol) continue;
            const int j = qc / nk2, kk = qc - j * nk2;
#pragma unroll
            for (int v4 = 0; v4 < 4; v4++) {
                const int i = m0 + (lane >> 4) + 4 * v4;
                if (i >= h) continue;
                put(i + 3, j, kk, T(pc[t][v4] - ps[t][v4]));
                if (i > 0 && 2 * i != n) put(n - i + 3, j, kk, T(pc[t][v4] + ps[t][v4]));
            }
        }
    }
}

template <typename T, int NT>
__global__ void __launch_bounds__(dft_bound(NT)) k_idft_x_out(Geo g, const T *__restrict__ spec, T *__restrict__ PI, int n,
                                                              const double *__restrict__ tab, int nk2, int jhalf) {
    extern __shared__ __align__(16) unsigned char smem[];
    idft_x_out_block<T, NT>(g, spec, PI, n, tab, nk2, xcd_tile(blockIdx.x, gridDim.x), smem, jhalf);
}

// value of the neighbouring lane (lane ^ 1) by a DPP quad permutation
__device__ __forceinline__ double lane_pair(double x) {
    const long long v = __double_as_longlong(x);
    const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0xb1, 0xf, 0xf, true);
    const unsigned hi = (unsigned)__builtin_amdgcn_mov_dpp((int)(v >> 32), 0xb1, 0xf, 0xf, true);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Along j, complex, for one kx and NC real columns (level, part): real and imaginary parts sit in
// neighbouring columns, so the products' cross terms come from the neighbouring lane.  In place (in == out) every
// element a block reads is in LDS before it writes any, and no other block touches its columns.  FP32 spectra are
// handed to the vertical sweeps in 64 bits (TO = double): rounded there, the longest waves' columns, whose systems
// are nearly singular, lose most of what a single-precision solve loses in its transforms.
template <typename TI, typename TO, int NT>
__global__ void __launch_bounds__(dft_bound(NT)) k_dft_y(const TI *in, TO *out, int n, const double *__restrict__ tab, int nk2, int sign) {
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int NC = 16 * NT;
    const int pitch = dft_pitch(NC), h = dft_rows(n), hk = (h + 3) & ~3, ncol = 2 * nk2;
    double *E = (double *)smem, *D = E + hk * pitch;
    const TileXY tile = xcd_tile_xy();
    const TI *x = in + (long long)tile.x * n * ncol;
    TO *o = out + (long long)tile.x * n * ncol;
    const int c0 = tile.y * NC, b = threadIdx.x % NC, q = min(c0 + b, ncol - 1);
    const int rows = blockDim.x / NC;
    for (int i = threadIdx.x / NC; i < hk; i += 4 * rows) {
        TI a[4], m[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int ir = min(i + r * rows, h - 1);
            a[r] = x[(long long)ir * ncol + q];
            m[r] = x[(long long)(ir == 0 ? 0 : n - ir) * ncol + q];
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int ir = i + r * rows;
            if (ir >= hk) break;
            const bool self = ir == 0 || 2 * ir == n;
            E[ir * pitch + b] = ir < h ? (self ? double(a[r]) : double(a[r]) + double(m[r])) : 0.0;
            D[ir * pitch + b] = ir < h && !self ? double(a[r]) - double(m[r]) : 0.0;
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
    // X(m) = P + s i Q and X(n-m) = P - s i Q with s = sign: +-Q(im) on the real part's lane, -+Q(re) on the other's
    const double sg = (lane & 1) != (sign < 0) ? 1.0 : -1.0;
    dvec4 pc[NT], ps[NT];
    for (int m0 = (threadIdx.x >> 6) * 16; m0 < h; m0 += (blockDim.x >> 6) * 16) {
        dft_products<NT>(tab, n, m0, E, D, pitch, pc, ps);
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const int qc = c0 + 16 * t + (lane & 15);
#pragma unroll
            for (int v4 = 0; v4 < 4; v4++) {
                const int m = m0 + (lane >> 4) + 4 * v4;
                const double d = sg * lane_pair(ps[t][v4]);
                if (m < h && qc < ncol) {
                    o[(long long)m * ncol + qc] = TO(pc[t][v4] + d);
                    if (m > 0 && 2 * m != n) o[(long long)(n - m) * ncol + qc] = TO(pc[t][v4] - d);
                }
            }
        }
    }
}

// Column tiles per block (4, 2 or 1) for `lines` groups of `ncol` columns: the most whose operands leave room
// for two blocks on a CU and whose blocks number one per CU, down to one tile
inline int dft_tiles(int n, long long lines, int ncol, int cus) {
    for (int nt = 4; nt > 1; nt /= 2)
        if (dft_lds(n, 16 * nt) <= 80 * 1024 && lines * ((ncol + 16 * nt - 1) / (16 * nt)) >= cus) return nt;
    return 1;
}
// threads of a block: a wavefront per tile of matrix rows, at least four (they share the loading)
inline int dft_threads(int n) { return 64 * std::min(16, std::max(4, dft_pad(n) / 16)); }

}  // namespace
}  // namespace dyn
