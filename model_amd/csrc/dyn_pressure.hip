// Anelastic pressure Poisson solve for gfx950 (serial periodic branch of solve_pressure,
// pressure.cpp:142-224, with poisson_fft3d 805-893 and divergence3d_periodic 1390-1424).
//
// Pipeline over the active levels kk = k-1, k in [1, NZ-1):
//   P1  divergence (fused prologue) + forward DFT along i     fields -> spec[kx][j][kk]
//   P2  forward DFT along j                                  spec -> spec (in place)
//   P3  1/(ni*nj) scaling + tridiagonal solve in k, FP64      spec -> spec (in place)
//   P4  backward DFT along j                                 spec -> spec
//   P5  backward DFT along i + real part -> PI with the k=0/NZ-1 copies and periodic halos fused
// The DFTs are Stockham auto-sort passes over an LDS tile [n][kc] (radix 4/2/3/5, direct sums for larger primes),
// batched over a chunk of kc consecutive levels so every global access is a contiguous kc-run of a k column, or
// products with their matrices (dyn_dft.hpp); pressure_init says which lengths take which.
#include <cmath>
#include <cstdlib>
#include <type_traits>
#include <vector>

#include "dyn_internal.hpp"

namespace dyn {
namespace {


constexpr int kThreads = 256;
constexpr int kThreadsX = 512;  // the real-transform passes along i (more loads in flight per CU)
constexpr size_t kLdsBudget = 64 * 1024;

// exp(sign * 2 pi i * e / n) from the forward table (cos, -sin)
template <typename T>
__device__ __forceinline__ void twiddle(const double *tw, int e, int sign, T &wr, T &wi) {
    wr = T(tw[2 * e]);
    wi = sign < 0 ? T(tw[2 * e + 1]) : -T(tw[2 * e + 1]);
}

template <typename T>
__device__ __forceinline__ void cmul(T &ar, T &ai, T br, T bi) {
    T r = ar * br - ai * bi;
    T i = ar * bi + ai * br;
    ar = r;
    ai = i;
}

// Two or four consecutive elements of a spectrum in one vector access.  A complex value starts at an even
// element, so a pair is aligned to its size; four elements (the two complex values of a level pair
// starting at an even level) are aligned to theirs when the level count is even.
template <typename T>
struct Vec2T;
template <>
struct Vec2T<float> {
    using type = float2;
};
template <>
struct Vec2T<double> {
    using type = double2;
};
template <typename T>
__device__ __forceinline__ void ld2(const T *p, T &a, T &b) {
    typename Vec2T<T>::type v;
    __builtin_memcpy(&v, __builtin_assume_aligned(p, sizeof(v)), sizeof(v));
    a = v.x;
    b = v.y;
}
template <typename T>
__device__ __forceinline__ void st2(T *p, T a, T b) {
    typename Vec2T<T>::type v;
    v.x = a;
    v.y = b;
    __builtin_memcpy(__builtin_assume_aligned(p, sizeof(v)), &v, sizeof(v));
}
template <typename T>
__device__ __forceinline__ void ld4(const T *p, T (&x)[4]) {
    if constexpr (sizeof(T) == 4) {
        float4 v;
        __builtin_memcpy(&v, __builtin_assume_aligned(p, 16), 16);
        x[0] = v.x;
        x[1] = v.y;
        x[2] = v.z;
        x[3] = v.w;
    } else {
        ld2(p, x[0], x[1]);
        ld2(p + 2, x[2], x[3]);
    }
}
template <typename T>
__device__ __forceinline__ void st4(T *p, T a, T b, T c, T d) {
    if constexpr (sizeof(T) == 4) {
        float4 v;
        v.x = a;
        v.y = b;
        v.z = c;
        v.w = d;
        __builtin_memcpy(__builtin_assume_aligned(p, 16), &v, 16);
    } else {
        st2(p, a, b);
        st2(p + 2, c, d);
    }
}

}  // namespace
}  // namespace dyn

#include "dyn_dft.hpp"

namespace dyn {
namespace {

// in-register DFT of length R with exponent sign `sign`
template <typename T>
__device__ __forceinline__ void butterfly(int R, T *xr, T *xi, int sign) {
    const T s = T(sign);
    if (R == 2) {
        T ar = xr[0] + xr[1], ai = xi[0] + xi[1];
        xr[1] = xr[0] - xr[1];
        xi[1] = xi[0] - xi[1];
        xr[0] = ar;
        xi[0] = ai;
    } else if (R == 4) {
        T t0r = xr[0] + xr[2], t0i = xi[0] + xi[2];
        T t1r = xr[0] - xr[2], t1i = xi[0] - xi[2];
        T t2r = xr[1] + xr[3], t2i = xi[1] + xi[3];
        T t3r = xr[1] - xr[3], t3i = xi[1] - xi[3];
        // i*s*(a1 - a3) = (-s*t3i, s*t3r)
        xr[0] = t0r + t2r;
        xi[0] = t0i + t2i;
        xr[2] = t0r - t2r;
        xi[2] = t0i - t2i;
        xr[1] = t1r - s * t3i;
        xi[1] = t1i + s * t3r;
        xr[3] = t1r + s * t3i;
        xi[3] = t1i - s * t3r;
    } else if (R == 3) {
        const T m = s * T(0.86602540378443864676);
        T t1r = xr[1] + xr[2], t1i = xi[1] + xi[2];
        T dr = xr[1] - xr[2], di = xi[1] - xi[2];
        T t2r = xr[0] - T(0.5) * t1r, t2i = xi[0] - T(0.5) * t1i;
        xr[0] = xr[0] + t1r;
        xi[0] = xi[0] + t1i;
        xr[1] = t2r - m * di;
        xi[1] = t2i + m * dr;
        xr[2] = t2r + m * di;
        xi[2] = t2i - m * dr;
    } else {  // R == 5
        const T c1 = T(0.30901699437494742410), c2 = T(-0.80901699437494742410);
        const T s1 = s * T(0.95105651629515357212), s2 = s * T(0.58778525229247312917);
        T b1r = xr[1] + xr[4], b1i = xi[1] + xi[4], b2r = xr[2] + xr[3], b2i = xi[2] + xi[3];
        T d1r = xr[1] - xr[4], d1i = xi[1] - xi[4], d2r = xr[2] - xr[3], d2i = xi[2] - xi[3];
        T a0r = xr[0], a0i = xi[0];
        T p1r = a0r + c1 * b1r + c2 * b2r, p1i = a0i + c1 * b1i + c2 * b2i;
        T p2r = a0r + c2 * b1r + c1 * b2r, p2i = a0i + c2 * b1i + c1 * b2i;
        T q1r = s1 * d1r + s2 * d2r, q1i = s1 * d1i + s2 * d2i;  // multiplied by i below
        T q2r = s2 * d1r - s1 * d2r, q2i = s2 * d1i - s1 * d2i;
        xr[0] = a0r + b1r + b2r;
        xi[0] = a0i + b1i + b2i;
        xr[1] = p1r - q1i;
        xi[1] = p1i + q1r;
        xr[4] = p1r + q1i;
        xi[4] = p1i - q1r;
        xr[2] = p2r - q2i;
        xi[2] = p2i + q2r;
        xr[3] = p2r + q2i;
        xi[3] = p2i - q2r;
    }
}

// in-register DFT of length 8: two length-4 DFTs of the even and odd inputs, combined with
// w^k = exp(sign i pi k / 4)
template <typename T>
__device__ __forceinline__ void butterfly8(T *xr, T *xi, int sign) {
    T er[4] = {xr[0], xr[2], xr[4], xr[6]}, ei[4] = {xi[0], xi[2], xi[4], xi[6]};
    T orr[4] = {xr[1], xr[3], xr[5], xr[7]}, oi[4] = {xi[1], xi[3], xi[5], xi[7]};
    butterfly(4, er, ei, sign);
    butterfly(4, orr, oi, sign);
    const T h = T(0.70710678118654752440), s = T(sign);
    // w^1 = h (1 + s i), w^2 = s i, w^3 = h (-1 + s i)
    T t1r = h * (orr[1] - s * oi[1]), t1i = h * (oi[1] + s * orr[1]);
    T t2r = -s * oi[2], t2i = s * orr[2];
    T t3r = h * (-orr[3] - s * oi[3]), t3i = h * (-oi[3] + s * orr[3]);
    xr[0] = er[0] + orr[0];
    xi[0] = ei[0] + oi[0];
    xr[4] = er[0] - orr[0];
    xi[4] = ei[0] - oi[0];
    xr[1] = er[1] + t1r;
    xi[1] = ei[1] + t1i;
    xr[5] = er[1] - t1r;
    xi[5] = ei[1] - t1i;
    xr[2] = er[2] + t2r;
    xi[2] = ei[2] + t2i;
    xr[6] = er[2] - t2r;
    xi[6] = ei[2] - t2i;
    xr[3] = er[3] + t3r;
    xi[3] = ei[3] + t3i;
    xr[7] = er[3] - t3r;
    xi[7] = ei[3] - t3i;
}

// Output q of butterfly jj of a Stockham pass of prime radix R > 5, summed directly: the butterfly's
// inputs x_r (element jj + r n/R), each twiddled by W^(r jm stride), times omega_R^(r q) = W^(r q n/R),
// i.e. sum_r x_r W^(r E mod n) with E = jm stride + q n/R.  The R-term sum runs in FP64 whatever the
// storage type (its rounding grows with R, where a factored transform's grows with log R).  `at(e)` is
// the twiddle W^e as (cos, -sin) of 2 pi e / n; `in(m)` returns element m of the line.
template <typename In, typename Tw>
__device__ __forceinline__ void dft_radix(int n, int R, int jj, int q, int Ns, int stride, int sign, In in, Tw at, double &yr,
                                          double &yi) {
    const int nbf = n / R, jm = jj % Ns;
    const int E = (int)(((long long)jm * stride + (long long)q * nbf) % n);
    double ar = 0.0, ai = 0.0;
    int e = 0;
    for (int r = 0; r < R; r++) {
        double xr, xi, wr, wi;
        in(jj + r * nbf, xr, xi);
        at(e, wr, wi);
        if (sign > 0) wi = -wi;
        ar += xr * wr - xi * wi;
        ai += xr * wi + xi * wr;
        e += E;
        if (e >= n) e -= n;
    }
    yr = ar;
    yi = ai;
}

// Stockham DFT of kc interleaved batches held in LDS as [n][kc] (re and im planes); ping-pongs
// between buffer 0 and 1 and returns the index of the buffer holding the result.  Radices 2 to 5 take
// the butterflies; a prime radix above 5 takes the direct sums of dft_radix, one output per work item.
template <typename T>
__device__ int lds_fft(T *re[2], T *im[2], const Radix &rad, int kc, const double *tw, int sign) {
    const int n = rad.n;
    int cur = 0, Ns = 1;
    for (int s = 0; s < rad.nr; s++) {
        const int R = rad.r[s];
        const int nb = n / R;
        const int stride = n / (Ns * R);
        T *ir = re[cur], *ii = im[cur], *orr = re[cur ^ 1], *oi = im[cur ^ 1];
        if (R > 5) {
            for (int idx = threadIdx.x; idx < n * kc; idx += blockDim.x) {
                const int b = idx % kc, o = idx / kc, jj = o % nb, q = o / nb;
                double yr, yi;
                dft_radix(
                    n, R, jj, q, Ns, stride, sign, [&](int m, double &xr, double &xi) { xr = double(ir[m * kc + b]); xi = double(ii[m * kc + b]); },
                    [&](int e, double &wr, double &wi) { wr = tw[2 * e]; wi = tw[2 * e + 1]; }, yr, yi);
                const int od = (jj / Ns) * Ns * R + jj % Ns;
                orr[(od + q * Ns) * kc + b] = T(yr);
                oi[(od + q * Ns) * kc + b] = T(yi);
            }
            __syncthreads();
            cur ^= 1;
            Ns *= R;
            continue;
        }
        for (int idx = threadIdx.x; idx < nb * kc; idx += blockDim.x) {
            int b = idx % kc, jj = idx / kc;
            T xr[5], xi[5];
            int jm = jj % Ns;
#pragma unroll
            for (int r = 0; r < 5; r++) {
                if (r < R) {
                    xr[r] = ir[(jj + r * nb) * kc + b];
                    xi[r] = ii[(jj + r * nb) * kc + b];
                }
            }
            if (Ns > 1) {
#pragma unroll
                for (int r = 1; r < 5; r++) {
                    if (r < R) {
                        T wr, wi;
                        twiddle(tw, r * jm * stride, sign, wr, wi);
                        cmul(xr[r], xi[r], wr, wi);
                    }
                }
            }
            butterfly(R, xr, xi, sign);
            int od = (jj / Ns) * Ns * R + jm;
#pragma unroll
            for (int r = 0; r < 5; r++) {
                if (r < R) {
                    orr[(od + r * Ns) * kc + b] = xr[r];
                    oi[(od + r * Ns) * kc + b] = xi[r];
                }
            }
        }
        __syncthreads();
        cur ^= 1;
        Ns *= R;
    }
    return cur;
}

#define IX(i, j, k) ((long long)(i) * g.NYNZ + (long long)(j) * g.NZ + (long long)(k))

// P1: divergence3d_periodic prologue + forward DFT along i; block = (j, level chunk)
template <typename T>
__global__ void __launch_bounds__(kThreads) k_div_fft_x(Geo g, Cols c, const T *__restrict__ UP, const T *__restrict__ VP,
                                                        const T *__restrict__ WP, T *__restrict__ spec, Radix rad, const double *tw,
                                                        int nk2, int kc, double step) {
    extern __shared__ unsigned char smem[];
    const int n = rad.n;
    T *re[2] = {(T *)smem, (T *)smem + 2 * n * kc};
    T *im[2] = {(T *)smem + n * kc, (T *)smem + 3 * n * kc};
    const int j = blockIdx.x;
    const int kk0 = blockIdx.y * kc;
    const int jj = j == 0 ? 1 : (j == g.NY - 1 ? g.NY - 2 : j);  // mirrored rows, pressure.cpp:1408-1415
    const DivStep<T> ds(g, step);
    // element idx = i*kc + b; when kc divides the block size each thread keeps its level b
    const bool fixed_b = (blockDim.x % kc) == 0;
    const int di = blockDim.x / kc;
    for (int idx = threadIdx.x, b = threadIdx.x % kc, i = threadIdx.x / kc - di; idx < n * kc; idx += blockDim.x) {
        i += di;
        if (!fixed_b) {
            b = idx % kc;
            i = idx / kc;
        }
        int kk = kk0 + b;
        T d = T(0);
        if (kk < nk2) {
            // the periodic column UP(NX-3) is read as UP(3), the value periodic_uvw_boundaries puts there
            int k = kk + 1, ia = i + 3;
            int ie = ia + 1 == g.NX - 3 ? 3 : ia + 1;
            d = T(ds(c.rhou[k], c.rhow[k + 1], c.rhow[k], c.mu[k], UP[IX(ie, jj, k)], UP[IX(ia, jj, k)], VP[IX(ia, jj + 1, k)],
                     VP[IX(ia, jj, k)], WP[IX(ia, jj, k + 1)], WP[IX(ia, jj, k)]));
        }
        re[0][idx] = d;
        im[0][idx] = T(0);
    }
    __syncthreads();
    int out = lds_fft(re, im, rad, kc, tw, -1);
    // spec[kx][j][kk] (interleaved complex)
    for (int idx = threadIdx.x; idx < n * kc; idx += blockDim.x) {
        int b = idx % kc, kx = idx / kc, kk = kk0 + b;
        if (kk < nk2) {
            long long o = (((long long)kx * g.NY + j) * nk2 + kk) * 2;
            spec[o] = re[out][idx];
            spec[o + 1] = im[out][idx];
        }
    }
}

// P2/P4: DFT along j for fixed kx; block = (kx, level chunk)
template <typename T>
__global__ void __launch_bounds__(kThreads) k_fft_y(T *__restrict__ spec, int nj, int nk2, Radix rad, const double *tw, int kc, int sign) {
    extern __shared__ unsigned char smem[];
    const int n = rad.n;
    T *re[2] = {(T *)smem, (T *)smem + 2 * n * kc};
    T *im[2] = {(T *)smem + n * kc, (T *)smem + 3 * n * kc};
    const int kx = blockIdx.x, kk0 = blockIdx.y * kc;
    for (int idx = threadIdx.x; idx < n * kc; idx += blockDim.x) {
        int b = idx % kc, ky = idx / kc, kk = kk0 + b;
        T vr = T(0), vi = T(0);
        if (kk < nk2) {
            long long o = (((long long)kx * nj + ky) * nk2 + kk) * 2;
            vr = spec[o];
            vi = spec[o + 1];
        }
        re[0][idx] = vr;
        im[0][idx] = vi;
    }
    __syncthreads();
    int out = lds_fft(re, im, rad, kc, tw, sign);
    for (int idx = threadIdx.x; idx < n * kc; idx += blockDim.x) {
        int b = idx % kc, ky = idx / kc, kk = kk0 + b;
        if (kk < nk2) {
            long long o = (((long long)kx * nj + ky) * nk2 + kk) * 2;
            spec[o] = re[out][idx];
            spec[o + 1] = im[out][idx];
        }
    }
}

// Pivot reciprocals z of pressure.cpp:840-855 for every (kx,ky): a pure function of the coefficients, so they
// are formed once per context instead of once per solve.  The multipliers F2 = ccoef z are one product away
// and are formed where they are used (the same bits).  Layout [kx][kk][ky]: the columns of one kx are
// adjacent for every level.
__global__ void k_thomas_factors(int ni, int nj, int nk, const double *__restrict__ coskx, const double *__restrict__ cosly,
                                 const double *__restrict__ rhou, const double *__restrict__ rhow, const double *__restrict__ mu,
                                 const double *__restrict__ mw, const double *__restrict__ acoef, const double *__restrict__ ccoef,
                                 double dx, double dz, double *__restrict__ zpiv) {
    int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= ni * nj) return;
    int kx = q / nj, ky = q % nj;
    int nk2 = nk - 2;
    double *Z = zpiv + (long long)kx * nk2 * nj + ky;
    const long long fs = nj;
    double ck = coskx[kx], cl = cosly[ky];
    // B2 of pressure.cpp:787-791
    double B = rhou[1] * 2.0 * (ck + cl - 2.0) / (dx * dx) - mu[1] * mw[2] * rhow[2] / (dz * dz);
    double z = 1.0 / B;
    double Fp = ccoef[1] * z;
    Z[0] = z;
    for (int k = 2; k < nk - 1; k++) {
        if (k < nk - 2) B = rhou[k] * 2.0 * (ck + cl - 2.0) / (dx * dx) - mu[k] * (mw[k + 1] * rhow[k + 1] + mw[k] * rhow[k]) / (dz * dz);
        else B = rhou[nk - 2] * 2.0 * (ck + cl - 2.0) / (dx * dx) - (mu[nk - 2] * mw[nk - 2] * rhow[nk - 2]) / (dz * dz);
        z = 1.0 / (B - acoef[k] * Fp);
        Fp = ccoef[k] * z;
        Z[(k - 1) * fs] = z;
    }
}

// P3: normalisation (pressure.cpp:824-827), forward elimination (837-856), mean-mode gauge (858-859)
// and back substitution (864-871), in FP64 whatever the storage precision.
template <typename T>
__global__ void k_thomas(T *__restrict__ spec, int ni, int nj, int nk, const double *__restrict__ acoef, const double *__restrict__ ccoef,
                         const double *__restrict__ zpiv) {
    int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= ni * nj) return;
    int kx = q / nj, ky = q % nj;
    const int nk2 = nk - 2;
    T *x = spec + (long long)q * nk2 * 2;
    const long long fs = nj;
    const double *Z = zpiv + (long long)kx * nk2 * nj + ky;
    const double size2d = (double)(ni * nj);
    double z = Z[0];
    double pr = (double(x[0]) / size2d) * z, pi = (double(x[1]) / size2d) * z;
    x[0] = T(pr);
    x[1] = T(pi);
    for (int k = 2; k < nk - 1; k++) {
        z = Z[(k - 1) * fs];
        double xr = double(x[2 * (k - 1)]) / size2d, xi = double(x[2 * (k - 1) + 1]) / size2d;
        pr = (xr - acoef[k] * pr) * z;
        pi = (xi - acoef[k] * pi) * z;
        x[2 * (k - 1)] = T(pr);
        x[2 * (k - 1) + 1] = T(pi);
    }
    if (kx == 0 && ky == 0) {  // OUT3D(0,0,NZ-2) = 0
        pr = 0.0;
        pi = 0.0;
        x[2 * (nk2 - 1)] = T(0);
        x[2 * (nk2 - 1) + 1] = T(0);
    }
    for (int k = nk - 3; k >= 1; k--) {
        double f = ccoef[k] * Z[(k - 1) * fs];
        pr = double(x[2 * (k - 1)]) - f * pr;
        pi = double(x[2 * (k - 1) + 1]) - f * pi;
        x[2 * (k - 1)] = T(pr);
        x[2 * (k - 1) + 1] = T(pi);
    }
}

// P5: backward DFT along i, real part -> PI (pressure.cpp:878-892) + periodic halos (boundaries.cpp:533-540)
template <typename T>
__global__ void __launch_bounds__(kThreads) k_ifft_x_out(Geo g, const T *__restrict__ spec, T *__restrict__ PI, Radix rad,
                                                         const double *tw, int nk2, int kc) {
    extern __shared__ unsigned char smem[];
    const int n = rad.n;
    T *re[2] = {(T *)smem, (T *)smem + 2 * n * kc};
    T *im[2] = {(T *)smem + n * kc, (T *)smem + 3 * n * kc};
    const int j = blockIdx.x, kk0 = blockIdx.y * kc;
    for (int idx = threadIdx.x; idx < n * kc; idx += blockDim.x) {
        int b = idx % kc, kx = idx / kc, kk = kk0 + b;
        T vr = T(0), vi = T(0);
        if (kk < nk2) {
            long long o = (((long long)kx * g.NY + j) * nk2 + kk) * 2;
            vr = spec[o];
            vi = spec[o + 1];
        }
        re[0][idx] = vr;
        im[0][idx] = vi;
    }
    __syncthreads();
    int out = lds_fft(re, im, rad, kc, tw, +1);
    const int shift = g.NX - 6;
    const bool fixed_b = (blockDim.x % kc) == 0;
    const int di = blockDim.x / kc;
    for (int idx = threadIdx.x, b = threadIdx.x % kc, i = threadIdx.x / kc - di; idx < n * kc; idx += blockDim.x) {
        i += di;
        if (!fixed_b) {
            b = idx % kc;
            i = idx / kc;
        }
        const int kk = kk0 + b;
        if (kk >= nk2) continue;
        T v = re[out][idx];
        int ia = i + 3;
        int k = kk + 1;
        int ks[3] = {k, -1, -1};
        if (kk == 0) ks[1] = 0;
        if (kk == nk2 - 1) ks[2] = g.NZ - 1;
        for (int t = 0; t < 3; t++) {
            if (ks[t] < 0) continue;
            PI[IX(ia, j, ks[t])] = v;
            if (ia >= shift && ia < shift + 3) PI[IX(ia - shift, j, ks[t])] = v;
            if (ia >= 3 && ia < 6) PI[IX(ia + shift, j, ks[t])] = v;
        }
    }
}


// ---- half-spectrum path -----------------------------------------------------------------------------
// The divergence is real, so two levels travel as the real and imaginary parts of one complex DFT along
// i and only kx = 0..ni/2 is kept (the rest is the conjugate mirror).  After the j-transform and the
// tridiagonal solve the real part of the inverse is rebuilt from that half, which is what taking the real
// part of the full inverse (pressure.cpp:881-890) computes.

// in-place Stockham DFT over LDS: element (n, b) at re[n*sn + b*sb], im[...]; every butterfly's inputs are
// read into registers before a barrier, then written to their output slots
// In-place Stockham DFT of nbatch sequences of length n held in LDS (element (jj, b) at jj*sn + b*sb, re
// and im in separate planes); twiddles come from an LDS copy of the table (twl[2e], twl[2e+1] = cos,
// -sin of 2 pi e / n).  Work item idx = tid + t*nthreads is butterfly jj = idx / nbatch of batch
// b = idx % nbatch; that split is done once, and the per-pass index arithmetic uses shifts while the
// running length Ns is a power of two (every pass of the radix-4/2-first plans before a 3 or 5).
// One radix-R pass of the power-of-two plans of lds_fft_ip with R a template parameter: items past the
// end read a valid slot (and are not written back), so the pass is straight-line code and every LDS
// load is issued before the first is waited on.
template <typename T, int R, int MAXB>
__device__ __forceinline__ void fft_pass_pow2(T *re, T *im, int n, int Ns, int lg, int sn, int sb, const int *bq, const int *jq,
                                              const T *twl, int sign) {
    const int nbf = n / R;
    const int stride = n / (Ns * R);
    T xr[MAXB][R], xi[MAXB][R];
    int oidx[MAXB];
#pragma unroll
    for (int t = 0; t < MAXB; t++) {
        const bool ok = jq[t] < nbf;
        const int jj = ok ? jq[t] : 0, b = bq[t];
        const int jm = jj & (Ns - 1), jd = jj >> lg;
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int e = (jj + r * nbf) * sn + b * sb;
            xr[t][r] = re[e];
            xi[t][r] = im[e];
        }
        if (Ns > 1) {
#pragma unroll
            for (int r = 1; r < R; r++) {
                const int e = r * jm * stride;
                const T wr = twl[2 * e], wi = sign < 0 ? twl[2 * e + 1] : -twl[2 * e + 1];
                cmul(xr[t][r], xi[t][r], wr, wi);
            }
        }
        if constexpr (R == 8) butterfly8(xr[t], xi[t], sign);
        else butterfly(R, xr[t], xi[t], sign);
        oidx[t] = ok ? (jd * Ns * R + jm) * sn + b * sb : -1;
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < MAXB; t++) {
        if (oidx[t] >= 0) {
#pragma unroll
            for (int r = 0; r < R; r++) {
                re[oidx[t] + r * Ns * sn] = xr[t][r];
                im[oidx[t] + r * Ns * sn] = xi[t][r];
            }
        }
    }
    __syncthreads();
}

// butterflies a thread holds in a radix-8 pass of a plan whose other passes hold MAXB (the radix-8 pass
// has half the radix-4 count; a third of MAXB keeps its registers within what the radix-4 passes use)
constexpr int pow2_maxb8(int maxb) { return maxb / 3 > 0 ? maxb / 3 : 1; }

// the power-of-two plans of lds_fft_ip alone (radix-4 passes, with one radix-2 or radix-8 pass when
// log2 n is odd)
template <typename T, int MAXB>
__device__ void lds_fft_pow2(T *re, T *im, const Radix &rad, int nbatch, int sn, int sb, const T *twl, int sign) {
    const int n = rad.n;
    int bq[MAXB], jq[MAXB];
#pragma unroll
    for (int t = 0; t < MAXB; t++) {
        const int idx = threadIdx.x + t * (int)blockDim.x;
        bq[t] = idx % nbatch;
        jq[t] = idx / nbatch;
    }
    int Ns = 1, lg = 0;
    for (int s = 0; s < rad.nr; s++) {
        if (rad.r[s] == 4) fft_pass_pow2<T, 4, MAXB>(re, im, n, Ns, lg, sn, sb, bq, jq, twl, sign);
        else if (rad.r[s] == 8) fft_pass_pow2<T, 8, pow2_maxb8(MAXB)>(re, im, n, Ns, lg, sn, sb, bq, jq, twl, sign);
        else fft_pass_pow2<T, 2, MAXB>(re, im, n, Ns, lg, sn, sb, bq, jq, twl, sign);
        Ns *= rad.r[s];
        lg = 31 - __clz(Ns);
    }
}

// power-of-two plan of the half-slab j pass: radix-4 passes, the first one radix 8 when log2 n is odd
// (so no radix-2 pass, whose butterflies would be twice as many per thread)
bool factorize(int n, Radix &rad);

inline bool pow2_plan48(int n, Radix &rad, bool radix8) {
    if (n < 2 || (n & (n - 1)) != 0) return false;
    if (!radix8) return factorize(n, rad);  // 4, ..., 4, 2
    rad.n = n;
    rad.nr = 0;
    int m = n;
    if (__builtin_ctz(n) % 2 == 1) {
        if (n == 2) {
            rad.r[rad.nr++] = 2;
            return true;
        }
        rad.r[rad.nr++] = 8;
        m /= 8;
    }
    while (m > 1 && rad.nr < kMaxRad) {
        rad.r[rad.nr++] = 4;
        m /= 4;
    }
    return m == 1;
}

template <typename T, int MAXB, bool POW2 = false>
__device__ __forceinline__ void lds_fft_ip(T *re, T *im, const Radix &rad, int nbatch, int sn, int sb, const T *twl, int sign) {
    const int n = rad.n;
    const int nthr = blockDim.x;
    int bq[MAXB], jq[MAXB];
#pragma unroll
    for (int t = 0; t < MAXB; t++) {
        const int idx = threadIdx.x + t * nthr;
        bq[t] = idx % nbatch;
        jq[t] = idx / nbatch;
    }
    if (POW2 && (n & (n - 1)) == 0) {  // power of two: radix-4 passes, then one radix-2 pass when log2 n is odd
        int Ns = 1, lg = 0;
        for (int s = 0; s < rad.nr; s++) {
            if (rad.r[s] == 4) fft_pass_pow2<T, 4, MAXB>(re, im, n, Ns, lg, sn, sb, bq, jq, twl, sign);
            else fft_pass_pow2<T, 2, MAXB>(re, im, n, Ns, lg, sn, sb, bq, jq, twl, sign);
            Ns *= rad.r[s];
            lg = 31 - __clz(Ns);
        }
        return;
    }
    int Ns = 1, lg = 0;
    for (int s = 0; s < rad.nr; s++) {
        const int R = rad.r[s];
        const int nbf = n / R;
        const int stride = n / (Ns * R);
        const bool pow2 = (Ns & (Ns - 1)) == 0;
        T xr[MAXB][5], xi[MAXB][5];
        int oidx[MAXB];
#pragma unroll
        for (int t = 0; t < MAXB; t++) {
            const int jj = jq[t], b = bq[t];
            if (jj < nbf) {
                const int jm = pow2 ? (jj & (Ns - 1)) : jj % Ns;
                const int jd = pow2 ? (jj >> lg) : jj / Ns;
#pragma unroll
                for (int r = 0; r < 5; r++) {
                    if (r < R) {
                        const int e = (jj + r * nbf) * sn + b * sb;
                        xr[t][r] = re[e];
                        xi[t][r] = im[e];
                    }
                }
                if (Ns > 1) {
#pragma unroll
                    for (int r = 1; r < 5; r++) {
                        if (r < R) {
                            const int e = r * jm * stride;
                            const T wr = twl[2 * e], wi = sign < 0 ? twl[2 * e + 1] : -twl[2 * e + 1];
                            cmul(xr[t][r], xi[t][r], wr, wi);
                        }
                    }
                }
                butterfly(R, xr[t], xi[t], sign);
                oidx[t] = (jd * Ns * R + jm) * sn + b * sb;
            }
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < MAXB; t++) {
            if (jq[t] < nbf) {
#pragma unroll
                for (int r = 0; r < 5; r++) {
                    if (r < R) {
                        re[oidx[t] + r * Ns * sn] = xr[t][r];
                        im[oidx[t] + r * Ns * sn] = xi[t][r];
                    }
                }
            }
        }
        __syncthreads();
        Ns *= R;
        if ((Ns & (Ns - 1)) == 0) lg = 31 - __clz(Ns);
    }
}

// copy the (cos, -sin) table of length n into LDS in the storage type
template <typename T>
__device__ __forceinline__ void load_twiddles(T *twl, const double *tw, int n) {
    for (int e = threadIdx.x; e < 2 * n; e += blockDim.x) twl[e] = T(tw[e]);
}

// j transforms of the three-kernel j pass for power-of-two nj: kc levels of one kx in LDS as [ky][level]
// (one padding level), transformed in place by the straight-line radix-8/4 passes with the twiddles in
// LDS; the same layout in HBM as k_fft_y
// 512 threads with two butterflies each keep the registers low (two blocks per CU) and still take 8
// FP32 or 8 FP64 levels per block, whole 64- or 128-byte runs of the spectrum per ky
constexpr int kFftYThreads = 512, kFftYMaxB = 2;
constexpr size_t kFftYLds = 96 * 1024;
template <typename T, int MAXB>
__global__ void __launch_bounds__(kFftYThreads) k_fft_y_pow2(T *__restrict__ spec, int nj, int nk2, Radix rad, const double *tw, int kc,
                                                         int sign) {
    extern __shared__ unsigned char smem[];
    const int n = rad.n, P2 = kc + 1;
    T *re = (T *)smem, *im = re + n * P2, *twl = im + n * P2;
    load_twiddles(twl, tw, n);
    const TileXY tile = xcd_tile_xy();
    const int kx = tile.x, kk0 = tile.y * kc;
    for (int idx = threadIdx.x; idx < n * kc; idx += blockDim.x) {
        const int b = idx % kc, ky = idx / kc, kk = kk0 + b;
        T vr = T(0), vi = T(0);
        if (kk < nk2) {
            const long long o = (((long long)kx * nj + ky) * nk2 + kk) * 2;
            vr = spec[o];
            vi = spec[o + 1];
        }
        re[ky * P2 + b] = vr;
        im[ky * P2 + b] = vi;
    }
    __syncthreads();
    lds_fft_pow2<T, MAXB>(re, im, rad, kc, P2, 1, twl, sign);
    for (int idx = threadIdx.x; idx < n * kc; idx += blockDim.x) {
        const int b = idx % kc, ky = idx / kc, kk = kk0 + b;
        if (kk < nk2) {
            const long long o = (((long long)kx * nj + ky) * nk2 + kk) * 2;
            spec[o] = re[ky * P2 + b];
            spec[o + 1] = im[ky * P2 + b];
        }
    }
}
inline size_t fft_y_pow2_lds(int n, int kc, size_t elt) { return 2 * (size_t)n * (kc + 1) * elt + 2 * (size_t)n * elt; }
// levels per block of k_fft_y_pow2 for the plan `rad` (the most that fit the LDS budget and the
// butterflies a thread holds in every pass), 0 when none do
template <typename T>
int fft_y_pow2_chunk(const Radix &rad, int nk2) {
    const int n = rad.n, maxb = kFftYMaxB;
    for (int kc = nk2 < 32 ? nk2 : 32; kc >= 1; kc--) {
        if (fft_y_pow2_lds(n, kc, sizeof(T)) > kFftYLds) continue;
        bool ok = true;
        for (int st = 0; ok && st < rad.nr; st++) {
            const int items = n / rad.r[st] * kc, per = (items + kFftYThreads - 1) / kFftYThreads;
            ok = per <= (rad.r[st] == 8 ? pow2_maxb8(maxb) : maxb);
        }
        if (ok) return kc;
    }
    return 0;
}

constexpr int kMaxBX = 4;   // butterflies per thread in the x passes (register-resident)
constexpr int kMaxBY = 4;   // and in the fused y pass (FP32, 1024 threads)
constexpr int kMaxBY64 = 6; // the fused y pass in FP64 runs 512 threads with up to 6 butterflies each
template <typename T>
constexpr int ypass_threads() { return sizeof(T) == 4 ? 1024 : 512; }
template <typename T>
constexpr int ypass_maxb() { return sizeof(T) == 4 ? kMaxBY : kMaxBY64; }
// the half-slab j pass (power-of-two plans, radix 4 and one radix-8 pass): FP32 1024 threads with up to
// 4 butterflies each, FP64 512 threads with up to 6 (what fits each thread's registers)
template <typename T>
constexpr int half_threads() { return sizeof(T) == 4 ? 1024 : 512; }
template <typename T>
constexpr int half_maxb() { return sizeof(T) == 4 ? 4 : 6; }

// Q1: divergence3d_periodic prologue + forward real DFT along i; block = (j, chunk of kc levels, kc even).
// The periodic column UP(NX-3) is read as UP(3), the value periodic_uvw_boundaries puts there.
// With src != nullptr the transform reads a ready real field src(i+3, j, k) instead of the divergence
// (the transposed solve of the adjoint).
template <typename T, int MAXB = kMaxBX>
__device__ __forceinline__ void div_rfft_x_block(const Geo &g, const Cols &c, const T *__restrict__ UP, const T *__restrict__ VP,
                                                 const T *__restrict__ WP, T *__restrict__ spec, const Radix &rad, const double *tw,
                                                 int nk2, int kc, double step, const T *__restrict__ src, int j, int chunk,
                                                 unsigned char *smem, bool wide) {
    const int n = rad.n, P = kc / 2, nkx = n / 2 + 1;
    T *re = (T *)smem, *im = re + n * P, *twl = im + n * P;
    const int kk0 = chunk * kc;
    load_twiddles(twl, tw, n);
    const int jj = j == 0 ? 1 : (j == g.NY - 1 ? g.NY - 2 : j);  // mirrored rows, pressure.cpp:1408-1415
    // the column coefficients of the block's kc levels (rhou(k), rhow(k+1), rhow(k), mu(k)), read once
    // into LDS instead of once per element
    double *colc = (double *)(twl + 2 * n);
    if (!src) {
        for (int b = (int)threadIdx.x; b < kc; b += (int)blockDim.x) {
            const int k = min(kk0 + b, nk2 - 1) + 1;
            colc[4 * b] = c.rhou[k];
            colc[4 * b + 1] = c.rhow[k + 1];
            colc[4 * b + 2] = c.rhow[k];
            colc[4 * b + 3] = c.mu[k];
        }
        __syncthreads();
    }
    // element idx = i*kc + b.  kU elements per thread per round: every global load of a round is issued
    // (clamped levels, so no load sits behind a branch) before any of them is used; the source-field form
    // and the divergence form are separate loops for the same reason.
    constexpr int kU = 4;
    const int ne = n * kc, nt = (int)blockDim.x;
    auto gather = [&](auto from_src, auto arithmetic) {
        constexpr bool kSrc = decltype(from_src)::value;
        const DivStep<decltype(arithmetic)> ds(g, step);
        for (int idx0 = (int)threadIdx.x; idx0 < ne; idx0 += kU * nt) {
            T f0[kU], f1[kU], f2[kU], f3[kU], f4[kU], f5[kU];
#pragma unroll
            for (int u = 0; u < kU; u++) {
                const int idx = min(idx0 + u * nt, ne - 1), b = idx % kc, i = idx / kc;
                const int k = min(kk0 + b, nk2 - 1) + 1, ia = i + 3;
                if (kSrc) {
                    f0[u] = src[IX(ia, j, k)];
                } else {
                    const int ie = ia + 1 == g.NX - 3 ? 3 : ia + 1;
                    f0[u] = UP[IX(ie, jj, k)];
                    f1[u] = UP[IX(ia, jj, k)];
                    f2[u] = VP[IX(ia, jj + 1, k)];
                    f3[u] = VP[IX(ia, jj, k)];
                    f4[u] = WP[IX(ia, jj, k + 1)];
                    f5[u] = WP[IX(ia, jj, k)];
                }
            }
#pragma unroll
            for (int u = 0; u < kU; u++) {
                const int idx = idx0 + u * nt, b = idx % kc, i = idx / kc;
                const int kk = kk0 + b;
                T d = T(0);
                if (kk < nk2 && kSrc) {
                    d = f0[u];
                } else if (kk < nk2) {
                    const double *cb = colc + 4 * b;
                    d = T(ds(cb[0], cb[1], cb[2], cb[3], f0[u], f1[u], f2[u], f3[u], f4[u], f5[u]));
                }
                if (idx < ne) {
                    if (b & 1) im[i * P + (b >> 1)] = d;
                    else re[i * P + (b >> 1)] = d;
                }
            }
        }
    };
    if (src) gather(std::true_type{}, T(0));
    else if (sizeof(T) == 4 && wide) gather(std::false_type{}, double(0));
    else gather(std::false_type{}, T(0));
    __syncthreads();
    lds_fft_ip<T, MAXB>(re, im, rad, P, P, 1, twl, -1);
    // split the packed pair: A = (Z[m] + conj Z[-m]) / 2, B = (Z[m] - conj Z[-m]) / 2i
    for (int idx = threadIdx.x; idx < nkx * P; idx += blockDim.x) {
        int pp = idx % P, m = idx / P;
        int mm = m == 0 ? 0 : n - m;
        T zr = re[m * P + pp], zi = im[m * P + pp], wr = re[mm * P + pp], wi = im[mm * P + pp];
        int ka = kk0 + 2 * pp, kb = ka + 1;
        long long o = ((long long)m * g.NY + j) * nk2;
        if (kb < nk2 && (nk2 & 1) == 0) {  // the pair's four values in one store
            st4(spec + (o + ka) * 2, T(0.5) * (zr + wr), T(0.5) * (zi - wi), T(0.5) * (zi + wi), T(0.5) * (wr - zr));
        } else {
            if (ka < nk2) {
                spec[(o + ka) * 2] = T(0.5) * (zr + wr);
                spec[(o + ka) * 2 + 1] = T(0.5) * (zi - wi);
            }
            if (kb < nk2) {
                spec[(o + kb) * 2] = T(0.5) * (zi + wi);
                spec[(o + kb) * 2 + 1] = T(0.5) * (wr - zr);
            }
        }
    }
}

// Q3: backward real DFT along i -> PI (pressure.cpp:878-892) with the ghost levels and periodic halos
template <typename T, int MAXB = kMaxBX>
__device__ __forceinline__ void irfft_x_out_block(const Geo &g, const T *__restrict__ spec, T *__restrict__ PI, const Radix &rad,
                                                  const double *tw, int nk2, int kc, int j, int chunk, unsigned char *smem,
                                                  int jhalf = 0) {
    const int n = rad.n, P = kc / 2, half = n / 2;
    T *re = (T *)smem, *im = re + n * P, *twl = im + n * P;
    const int kk0 = chunk * kc;
    load_twiddles(twl, tw, n);
    // rebuild Z = A + iB for m in [0, n) from the half spectra of the two levels of each pair.  kU
    // elements per thread per round: every global load of a round is issued (clamped levels, so no load
    // sits behind a branch) before any of them is used.
    // With jhalf the half-slab j pass left row j of the full inverse as v0(j') + s v1(j'), j' = j mod
    // jhalf, with v0 in row j' and v1 in row jhalf + j' (s = +1 on the first half of the rows, -1 on the
    // second).
    constexpr int kU = 4;
    const int ne = n * P, nt = (int)blockDim.x;
    const int jp = jhalf ? (j < jhalf ? j : j - jhalf) : j;
    const T sg = j < jhalf ? T(1) : T(-1);
    for (int idx0 = (int)threadIdx.x; idx0 < ne; idx0 += kU * nt) {
        T x[kU][4], y[kU][4];  // (re, im) at ka, then at kb: row jp (x) and, with jhalf, row jhalf + jp (y)
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const int idx = min(idx0 + u * nt, ne - 1), pp = idx % P, m = idx / P;
            const int ka = min(kk0 + 2 * pp, nk2 - 1), kb = min(kk0 + 2 * pp + 1, nk2 - 1);
            const int ms = m <= half ? m : n - m;
            const long long o0 = ((long long)ms * g.NY + jp) * nk2;
            x[u][0] = spec[(o0 + ka) * 2];
            x[u][1] = spec[(o0 + ka) * 2 + 1];
            x[u][2] = spec[(o0 + kb) * 2];
            x[u][3] = spec[(o0 + kb) * 2 + 1];
            if (jhalf) {
                const long long o1 = ((long long)ms * g.NY + jhalf + jp) * nk2;
                y[u][0] = spec[(o1 + ka) * 2];
                y[u][1] = spec[(o1 + ka) * 2 + 1];
                y[u][2] = spec[(o1 + kb) * 2];
                y[u][3] = spec[(o1 + kb) * 2 + 1];
            }
        }
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const int idx = idx0 + u * nt, pp = idx % P, m = idx / P;
            const int ka = kk0 + 2 * pp, kb = ka + 1;
            const int ms = m <= half ? m : n - m;
            T ar = T(0), ai = T(0), br = T(0), bi = T(0);
            if (jhalf) {
                if (ka < nk2) {
                    ar = x[u][0] + sg * y[u][0];
                    ai = x[u][1] + sg * y[u][1];
                }
                if (kb < nk2) {
                    br = x[u][2] + sg * y[u][2];
                    bi = x[u][3] + sg * y[u][3];
                }
            } else {
                if (ka < nk2) {
                    ar = x[u][0];
                    ai = x[u][1];
                }
                if (kb < nk2) {
                    br = x[u][2];
                    bi = x[u][3];
                }
            }
            if (ms == 0 || 2 * ms == n) {  // self-conjugate wavenumbers: only the real part is kept
                ai = T(0);
                bi = T(0);
            }
            if (m > half) {  // conjugate mirror
                ai = -ai;
                bi = -bi;
            }
            if (idx < ne) {
                re[m * P + pp] = ar - bi;
                im[m * P + pp] = ai + br;
            }
        }
    }
    __syncthreads();
    lds_fft_ip<T, MAXB>(re, im, rad, P, P, 1, twl, +1);
    const int shift = g.NX - 6;
    const bool fixed_b = (blockDim.x % kc) == 0;
    const int di = blockDim.x / kc;
    for (int idx = threadIdx.x, b = threadIdx.x % kc, i = threadIdx.x / kc - di; idx < n * kc; idx += blockDim.x) {
        i += di;
        if (!fixed_b) {
            b = idx % kc;
            i = idx / kc;
        }
        const int kk = kk0 + b;
        if (kk >= nk2) continue;
        T v = (b & 1) ? im[i * P + (b >> 1)] : re[i * P + (b >> 1)];
        int ia = i + 3, k = kk + 1;
        int ks[3] = {k, -1, -1};
        if (kk == 0) ks[1] = 0;
        if (kk == nk2 - 1) ks[2] = g.NZ - 1;
        for (int t = 0; t < 3; t++) {
            if (ks[t] < 0) continue;
            PI[IX(ia, j, ks[t])] = v;
            if (ia >= shift && ia < shift + 3) PI[IX(ia - shift, j, ks[t])] = v;
            if (ia >= 3 && ia < 6) PI[IX(ia + shift, j, ks[t])] = v;
        }
    }
}

// a_k and c_k of levels k = 1 .. nk2 in LDS (ac[kk], cc[kk], kk = k-1): read from global memory they are scalar
// loads of a cache line per chunk, each waited for in turn
struct ThomasCoef {
    const double *ac, *cc;
};
struct ThomasArgs {
    const double *acoef, *ccoef;  // by level k
    const double *zpiv;           // pivot reciprocals z of every column, [kx][kk][ky]
    int ni, nj, nk;
};
inline ThomasArgs thomas_args(const PressurePlan &pp, int nk) { return ThomasArgs{pp.acoef, pp.ccoef, pp.zpiv, pp.ni, pp.nj, nk}; }

__device__ __forceinline__ ThomasCoef thomas_coef(const ThomasArgs &ta, int nk2, double *lds) {
    for (int q = (int)threadIdx.x; q < 2 * nk2; q += (int)blockDim.x) lds[q] = q < nk2 ? ta.acoef[q + 1] : ta.ccoef[q - nk2 + 1];
    return ThomasCoef{lds, lds + nk2};
}

// x / d for the divisor's correctly rounded reciprocal r: x r is within an ulp of the quotient, its remainder
// is exact in a fused multiply-add, and adding remainder r rounds to the quotient itself (Markstein 1990);
// a dozen FP64 instructions fewer than a division, and the sweeps are bound by what they issue.
__device__ __forceinline__ double div_exact(double x, double d, double r) {
    const double q = x * r;
    return __builtin_fma(__builtin_fma(-q, d, x), r, q);
}

// The sweeps below walk the levels in chunks of kTC and load the next chunk's pivots (one column of the table,
// from global memory or from a copy in LDS) while the current chunk is eliminated, so the dependent
// recurrence does not wait on memory latency level by level.  The multipliers are F_k = c_k z_k.
constexpr int kThomasChunk = 8;  // levels per chunk of the Thomas sweeps

// Forward elimination and back substitution of one real sequence (the real or the imaginary part) of one
// (kx,ky) column whose values sit at x[kk*xs]; FP64 arithmetic with the pivots and multipliers of the
// tables; the (0,0) column (m0) keeps its eliminated values in the FP64 scratch mean[2*kk] instead of the
// storage type (pressure.cpp:837-871).  Level k = kk+1; acoef[1] = 0, so the first level needs no
// special case.
// The sweeps walk kTC levels at a time, and the table entries of the next chunk are loaded while the
// current chunk is eliminated, into the second of two register sets that take turns: a loop that copied
// the prefetched set into the current one at its end had to wait there for the loads just issued, so
// every chunk waited a whole memory latency.  Every load is unconditional (clamped indices); only the
// last partial chunk guards its steps.  The (0,0) column differs only in where its values are kept (a
// per-lane choice of store and of load): an instance of its own would diverge from the other lanes of
// its wavefront and run the whole chain twice.
template <int kTC>
__device__ __forceinline__ void thomas_tab_up(const double *Tab, long long fs, int k0, int hi, double (&v)[kTC]) {
#pragma unroll
    for (int t = 0; t < kTC; t++) v[t] = Tab[min(k0 + t, hi) * fs];
}
template <int kTC>
__device__ __forceinline__ void thomas_tab_down(const double *Tab, long long fs, int k0, double (&v)[kTC]) {
#pragma unroll
    for (int t = 0; t < kTC; t++) v[t] = Tab[max(k0 - t, 0) * fs];
}
// p_kk = (x_kk / (ni nj) - a_k p_{kk-1}) z_kk for the chunk's levels kk = k0 .. k0+kTC-1 (< N unless FULL)
template <bool FULL, int kTC, typename T>
__device__ __forceinline__ void thomas_fwd_chunk(const ThomasCoef &co, const double (&z)[kTC], int k0, int N, double size2d,
                                                 double rsize, T *x, int xs, bool m0, double *mean, double &p) {
    double v[kTC], ac[kTC];
#pragma unroll
    for (int t = 0; t < kTC; t++) {
        const int kk = FULL ? k0 + t : min(k0 + t, N - 1);
        v[t] = double(x[kk * xs]);
        ac[t] = co.ac[kk];
    }
#pragma unroll
    for (int t = 0; t < kTC; t++) {
        if (FULL || k0 + t < N) p = (div_exact(v[t], size2d, rsize) - ac[t] * p) * z[t];
        v[t] = p;
    }
#pragma unroll
    for (int t = 0; t < kTC; t++) {
        if (FULL || k0 + t < N) {
            if (m0) mean[2 * (k0 + t)] = v[t];
            else x[(k0 + t) * xs] = T(v[t]);
        }
    }
}
// x_kk = y_kk - F_kk x_{kk+1} for kk = k0 .. k0-kTC+1 (>= 0 unless FULL)
template <typename R, bool FULL, int kTC, typename T>
__device__ __forceinline__ void thomas_back_chunk(const ThomasCoef &co, const double (&z)[kTC], int k0, T *x, int xs, bool m0,
                                                  const double *mean, double &p) {
    double v[kTC], f[kTC];
#pragma unroll
    for (int t = 0; t < kTC; t++) {
        const int kk = FULL ? k0 - t : max(k0 - t, 0);
        const double vm = mean[2 * kk], vx = double(x[kk * xs]);
        v[t] = m0 ? vm : vx;
        f[t] = co.cc[kk] * z[t];
    }
#pragma unroll
    for (int t = 0; t < kTC; t++) {
        if (FULL || k0 - t >= 0) p = v[t] - f[t] * p;
        v[t] = p;
    }
#pragma unroll
    for (int t = 0; t < kTC; t++)
        if (FULL || k0 - t >= 0) x[(k0 - t) * xs] = T(R(v[t]));
}
// Z: the column's pivots, one every fs; R: the type the results are rounded to, whatever type T holds them
template <typename R, int kTC = kThomasChunk, typename T>
__device__ __forceinline__ void thomas_part(const ThomasArgs &ta, const ThomasCoef &co, int kx, int ky, const double *Z, long long fs, T *x, int xs,
                                            double *mean) {
    const int N = ta.nk - 2;
    const double size2d = (double)(ta.ni * ta.nj), rsize = 1.0 / size2d;
    const bool m0 = (kx == 0 && ky == 0);
    double A[kTC], B[kTC], p = 0.0;
    // full chunks two at a time (one path through the loop, so the loads of the set not in use stay in
    // flight across its back edge), then the levels left
    thomas_tab_up<kTC>(Z, fs, 0, N - 1, A);
    int k0 = 0;
    for (; k0 + 2 * kTC <= N; k0 += 2 * kTC) {
        thomas_tab_up<kTC>(Z, fs, k0 + kTC, N - 1, B);
        thomas_fwd_chunk<true, kTC>(co, A, k0, N, size2d, rsize, x, xs, m0, mean, p);
        thomas_tab_up<kTC>(Z, fs, k0 + 2 * kTC, N - 1, A);
        thomas_fwd_chunk<true, kTC>(co, B, k0 + kTC, N, size2d, rsize, x, xs, m0, mean, p);
    }
    if (k0 < N) {
        thomas_tab_up<kTC>(Z, fs, k0 + kTC, N - 1, B);
        if (k0 + kTC <= N) thomas_fwd_chunk<true, kTC>(co, A, k0, N, size2d, rsize, x, xs, m0, mean, p);
        else thomas_fwd_chunk<false, kTC>(co, A, k0, N, size2d, rsize, x, xs, m0, mean, p);
        if (k0 + kTC < N) thomas_fwd_chunk<false, kTC>(co, B, k0 + kTC, N, size2d, rsize, x, xs, m0, mean, p);
    }
    if (m0) p = 0.0;  // OUT3D(0,0,NZ-2) = 0
    x[(N - 1) * xs] = T(R(p));
    if (N < 2) return;
    // back substitution x_kk = y_kk - F_kk x_{kk+1} for kk = N-2 .. 0, walking down in chunks
    thomas_tab_down<kTC>(Z, fs, N - 2, A);
    k0 = N - 2;
    for (; k0 - 2 * kTC + 1 >= 0; k0 -= 2 * kTC) {
        thomas_tab_down<kTC>(Z, fs, k0 - kTC, B);
        thomas_back_chunk<R, true, kTC>(co, A, k0, x, xs, m0, mean, p);
        thomas_tab_down<kTC>(Z, fs, k0 - 2 * kTC, A);
        thomas_back_chunk<R, true, kTC>(co, B, k0 - kTC, x, xs, m0, mean, p);
    }
    if (k0 >= 0) {
        thomas_tab_down<kTC>(Z, fs, k0 - kTC, B);
        if (k0 - kTC + 1 >= 0) thomas_back_chunk<R, true, kTC>(co, A, k0, x, xs, m0, mean, p);
        else thomas_back_chunk<R, false, kTC>(co, A, k0, x, xs, m0, mean, p);
        if (k0 - kTC >= 0) thomas_back_chunk<R, false, kTC>(co, B, k0 - kTC, x, xs, m0, mean, p);
    }
}

// q_kk = x_kk - F_{kk-1} q_{kk-1} for the chunk's levels kk = k0 .. k0+kTC-1 (< N unless FULL), z[t] = z_{k0+t-1}
template <bool FULL, int kTC, typename T>
__device__ __forceinline__ void thomas_t_fwd_chunk(const ThomasCoef &co, const double (&z)[kTC], int k0, int N, T *x, int xs, double &q) {
    double v[kTC], f[kTC];
#pragma unroll
    for (int t = 0; t < kTC; t++) {
        const int kk = FULL ? k0 + t : min(k0 + t, N - 1);
        v[t] = double(x[kk * xs]);
        f[t] = co.cc[kk - 1] * z[t];
    }
#pragma unroll
    for (int t = 0; t < kTC; t++) {
        if (FULL || k0 + t < N) q = v[t] - f[t] * q;
        v[t] = q;
    }
#pragma unroll
    for (int t = 0; t < kTC; t++)
        if (FULL || k0 + t < N) x[(k0 + t) * xs] = T(v[t]);
}
// b_kk = z_kk (q_kk - a_{kk+2} b_{kk+1}), stored as b / (ni nj), for kk = k0 .. k0-kTC+1 (>= 0 unless FULL)
template <typename R, bool FULL, int kTC, typename T>
__device__ __forceinline__ void thomas_t_back_chunk(const ThomasCoef &co, const double (&z)[kTC], int k0, double size2d, double rsize,
                                                    T *x, int xs, double &b) {
    double v[kTC], ac[kTC];
#pragma unroll
    for (int t = 0; t < kTC; t++) {
        const int kk = FULL ? k0 - t : max(k0 - t, 0);
        v[t] = double(x[kk * xs]);
        ac[t] = co.ac[kk + 1];
    }
#pragma unroll
    for (int t = 0; t < kTC; t++) {
        if (FULL || k0 - t >= 0) b = (v[t] - ac[t] * b) * z[t];
        v[t] = div_exact(b, size2d, rsize);
    }
#pragma unroll
    for (int t = 0; t < kTC; t++)
        if (FULL || k0 - t >= 0) x[(k0 - t) * xs] = T(R(v[t]));
}
// Transpose of thomas_part (the adjoint's vertical solve), in place.  The forward map is p = L'^{-1} x / S
// (L' lower bidiagonal: 1/z_k on the diagonal, a_k below) followed by x_k = p_k - F_k x_{k+1}; for the
// (0,0) column p_N is replaced by 0.  The transpose runs the two bidiagonal solves transposed and in
// reverse order: q_1 = x_1, q_k = x_k - F_{k-1} q_{k-1} (q_N = 0 for (0,0)), then b_N = z_N q_N,
// b_k = z_k (q_k - a_{k+1} b_{k+1}), result b / S.  The singular last pivot of (0,0) is never used.
// The table entries come in chunks through two register sets that take turns, as in thomas_part.
template <typename R, int kTC = kThomasChunk, typename T>
__device__ __forceinline__ void thomas_part_t(const ThomasArgs &ta, const ThomasCoef &co, int kx, int ky, const double *Z, long long fs,
                                              T *x, int xs) {
    const int N = ta.nk - 2;
    const double size2d = (double)(ta.ni * ta.nj), rsize = 1.0 / size2d;
    const bool m0 = (kx == 0 && ky == 0);
    double A[kTC], B[kTC];
    // q_kk = x_kk - F_{kk-1} q_{kk-1}, kk = 1 .. N-1 (q_0 = x_0)
    double q = double(x[0]);
    thomas_tab_up<kTC>(Z, fs, 0, N - 2, A);
    int k0 = 1;
    for (; k0 + 2 * kTC <= N; k0 += 2 * kTC) {
        thomas_tab_up<kTC>(Z, fs, k0 + kTC - 1, N - 2, B);
        thomas_t_fwd_chunk<true, kTC>(co, A, k0, N, x, xs, q);
        thomas_tab_up<kTC>(Z, fs, k0 + 2 * kTC - 1, N - 2, A);
        thomas_t_fwd_chunk<true, kTC>(co, B, k0 + kTC, N, x, xs, q);
    }
    if (k0 < N) {
        thomas_tab_up<kTC>(Z, fs, k0 + kTC - 1, N - 2, B);
        if (k0 + kTC <= N) thomas_t_fwd_chunk<true, kTC>(co, A, k0, N, x, xs, q);
        else thomas_t_fwd_chunk<false, kTC>(co, A, k0, N, x, xs, q);
        if (k0 + kTC < N) thomas_t_fwd_chunk<false, kTC>(co, B, k0 + kTC, N, x, xs, q);
    }
    // b_{N-1} = z_{N-1} q_{N-1} (0 for (0,0)); b_kk = z_kk (q_kk - a_{kk+2} b_{kk+1}), kk = N-2 .. 0
    double b = m0 ? 0.0 : double(x[(N - 1) * xs]) * Z[(N - 1) * fs];
    x[(N - 1) * xs] = T(R(div_exact(b, size2d, rsize)));
    if (N < 2) return;
    thomas_tab_down<kTC>(Z, fs, N - 2, A);
    k0 = N - 2;
    for (; k0 - 2 * kTC + 1 >= 0; k0 -= 2 * kTC) {
        thomas_tab_down<kTC>(Z, fs, k0 - kTC, B);
        thomas_t_back_chunk<R, true, kTC>(co, A, k0, size2d, rsize, x, xs, b);
        thomas_tab_down<kTC>(Z, fs, k0 - 2 * kTC, A);
        thomas_t_back_chunk<R, true, kTC>(co, B, k0 - kTC, size2d, rsize, x, xs, b);
    }
    if (k0 >= 0) {
        thomas_tab_down<kTC>(Z, fs, k0 - kTC, B);
        if (k0 - kTC + 1 >= 0) thomas_t_back_chunk<R, true, kTC>(co, A, k0, size2d, rsize, x, xs, b);
        else thomas_t_back_chunk<R, false, kTC>(co, A, k0, size2d, rsize, x, xs, b);
        if (k0 - kTC >= 0) thomas_t_back_chunk<R, false, kTC>(co, B, k0 - kTC, size2d, rsize, x, xs, b);
    }
}

// Global <-> LDS copies of one kx slab: n complex values (re, im interleaved) at spec[base + 2 idx], in
// the LDS planes at (idx / nk2) * P2 + idx % nk2.  Each thread issues kU global loads (clamped indices, so
// no load sits behind a branch) before it writes any of them: a guarded load inside the loop made the
// compiler wait for each one before issuing the next.
constexpr int kSlabU = 8;
template <typename T>
__device__ __forceinline__ void slab_to_lds(const T *__restrict__ spec, long long base, int n, int nk2, int P2, T *re, T *im) {
    const int nt = (int)blockDim.x, dk = nt % nk2, dy = nt / nk2;
    int kk = (int)threadIdx.x % nk2, ky = (int)threadIdx.x / nk2;
    for (int i0 = (int)threadIdx.x; i0 < n; i0 += kSlabU * nt) {
        T vr[kSlabU], vi[kSlabU];
#pragma unroll
        for (int u = 0; u < kSlabU; u++) {
            ld2(spec + base + 2LL * min(i0 + u * nt, n - 1), vr[u], vi[u]);
        }
#pragma unroll
        for (int u = 0; u < kSlabU; u++) {
            if (i0 + u * nt < n) {
                re[ky * P2 + kk] = vr[u];
                im[ky * P2 + kk] = vi[u];
            }
            kk += dk;
            ky += dy;
            if (kk >= nk2) {
                kk -= nk2;
                ky++;
            }
        }
    }
}
template <typename T>
__device__ __forceinline__ void lds_to_slab(T *__restrict__ spec, long long base, int n, int nk2, int P2, const T *re, const T *im) {
    const int nt = (int)blockDim.x, dk = nt % nk2, dy = nt / nk2, last = n / nk2 - 1;
    int kk = (int)threadIdx.x % nk2, ky = (int)threadIdx.x / nk2;
    for (int i0 = (int)threadIdx.x; i0 < n; i0 += kSlabU * nt) {
        T vr[kSlabU], vi[kSlabU];
#pragma unroll
        for (int u = 0; u < kSlabU; u++) {
            const int e = min(ky, last) * P2 + kk;  // rows past the slab read its last row (not stored)
            vr[u] = re[e];
            vi[u] = im[e];
            kk += dk;
            ky += dy;
            if (kk >= nk2) {
                kk -= nk2;
                ky++;
            }
        }
#pragma unroll
        for (int u = 0; u < kSlabU; u++) {
            const int idx = i0 + u * nt;
            if (idx < n) st2(spec + base + 2LL * idx, vr[u], vi[u]);
        }
    }
}

// Q2 (fused): forward DFT along j, FP64 tridiagonal solve, backward DFT along j for one kx, with the
// whole (j, k) slab of that kx resident in LDS
template <typename T, bool TR, bool POW2 = true, int MAXB = ypass_maxb<T>()>
__device__ __forceinline__ void ypass_block(T *__restrict__ spec, int nk2, const Radix &rady, const double *twy, const ThomasArgs &ta,
                                            int pad, int kx, unsigned char *smem) {
    const int nj = rady.n, P2 = nk2 + pad;
    T *re = (T *)smem, *im = re + nj * P2;
    double *mean = (double *)(re + 2 * nj * P2);  // 2*nj*P2 elements of T: 8-byte aligned
    T *twl = (T *)(mean + 4 * nk2 + 1);
    const ThomasCoef co = thomas_coef(ta, nk2, mean + 2 * nk2);
    load_twiddles(twl, twy, nj);
    const long long base = (long long)kx * nj * nk2 * 2;
    slab_to_lds(spec, base, nj * nk2, nk2, P2, re, im);
    __syncthreads();
    lds_fft_ip<T, MAXB, POW2>(re, im, rady, nk2, P2, 1, twl, -1);
    if ((int)threadIdx.x < 2 * nj) {
        // one thread per real sequence: threads [0, nj) take the real parts, [nj, 2 nj) the imaginary parts
        const int part = (int)threadIdx.x >= nj, ky = (int)threadIdx.x - part * nj;
        T *x = (part ? im : re) + ky * P2;
        const double *Z = ta.zpiv + (long long)kx * nj * nk2 + ky;
        if (TR) thomas_part_t<T>(ta, co, kx, ky, Z, nj, x, 1);
        else thomas_part<T>(ta, co, kx, ky, Z, nj, x, 1, mean + part);
    }
    __syncthreads();
    lds_fft_ip<T, MAXB, POW2>(re, im, rady, nk2, P2, 1, twl, +1);
    lds_to_slab(spec, base, nj * nk2, nk2, P2, re, im);
}

template <typename T, int MAXB>
__global__ void __launch_bounds__(kThreadsX) k_div_rfft_x(Geo g, Cols c, const T *__restrict__ UP, const T *__restrict__ VP,
                                                         const T *__restrict__ WP, T *__restrict__ spec, Radix rad, const double *tw,
                                                         int nk2, int kc, double step, const T *__restrict__ src, bool wide) {
    extern __shared__ unsigned char smem[];
    const TileXY t = xcd_tile_xy();
    div_rfft_x_block<T, MAXB>(g, c, UP, VP, WP, spec, rad, tw, nk2, kc, step, src, t.x, t.y, smem, wide);
}

template <typename T, int MAXB>
__global__ void __launch_bounds__(kThreadsX) k_irfft_x_out(Geo g, const T *__restrict__ spec, T *__restrict__ PI, Radix rad,
                                                          const double *tw, int nk2, int kc, int half) {
    extern __shared__ unsigned char smem[];
    const TileXY t = xcd_tile_xy();
    irfft_x_out_block<T, MAXB>(g, spec, PI, rad, tw, nk2, kc, t.x, t.y, smem, half);
}

// The same after the half-slab j pass, one block per row pair (j', jhalf + j') and chunk of kc levels:
// it reads v0 (row j') and v1 (row jhalf + j') once for both rows (v0 + v1 and v0 - v1), and transforms
// the two rows as one batch of kc level pairs.  Values as irfft_x_out_block's, bit for bit.
template <typename T, int MAXB = kMaxBX>
__device__ __forceinline__ void irfft_x_out_pair_block(const Geo &g, const T *__restrict__ spec, T *__restrict__ PI, const Radix &rad,
                                                       const double *tw, int nk2, int kc, int jp, int chunk, unsigned char *smem,
                                                       int jhalf) {
    const int n = rad.n, P = kc / 2, B = 2 * P, half = n / 2;  // B: batch of both rows' level pairs
    T *re = (T *)smem, *im = re + n * B, *twl = im + n * B;
    const int kk0 = chunk * kc;
    load_twiddles(twl, tw, n);
#pragma unroll 2
    for (int idx = threadIdx.x; idx < n * P; idx += blockDim.x) {
        int pp = idx % P, m = idx / P;
        int ka = kk0 + 2 * pp, kb = ka + 1;
        int ms = m <= half ? m : n - m;
        const long long o0 = ((long long)ms * g.NY + jp) * nk2, o1 = ((long long)ms * g.NY + jhalf + jp) * nk2;
        T e[4] = {T(0), T(0), T(0), T(0)}, o[4] = {T(0), T(0), T(0), T(0)};  // a re, a im, b re, b im
        if (kb < nk2 && (nk2 & 1) == 0) {  // the pair's four values in one load
            ld4(spec + (o0 + ka) * 2, e);
            ld4(spec + (o1 + ka) * 2, o);
        } else {
            if (ka < nk2) {
                ld2(spec + (o0 + ka) * 2, e[0], e[1]);
                ld2(spec + (o1 + ka) * 2, o[0], o[1]);
            }
            if (kb < nk2) {
                ld2(spec + (o0 + kb) * 2, e[2], e[3]);
                ld2(spec + (o1 + kb) * 2, o[2], o[3]);
            }
        }
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const T sg = r == 0 ? T(1) : T(-1);
            T ar = T(0), ai = T(0), br = T(0), bi = T(0);
            if (ka < nk2) {
                ar = e[0] + sg * o[0];
                ai = e[1] + sg * o[1];
            }
            if (kb < nk2) {
                br = e[2] + sg * o[2];
                bi = e[3] + sg * o[3];
            }
            if (ms == 0 || 2 * ms == n) {  // self-conjugate wavenumbers: only the real part is kept
                ai = T(0);
                bi = T(0);
            }
            if (m > half) {  // conjugate mirror
                ai = -ai;
                bi = -bi;
            }
            re[m * B + r * P + pp] = ar - bi;
            im[m * B + r * P + pp] = ai + br;
        }
    }
    __syncthreads();
    lds_fft_ip<T, MAXB>(re, im, rad, B, B, 1, twl, +1);
    const int shift = g.NX - 6;
    for (int idx = threadIdx.x; idx < 2 * n * kc; idx += blockDim.x) {
        const int r = idx / (n * kc), rem = idx - r * (n * kc);
        const int b = rem % kc, i = rem / kc;
        const int kk = kk0 + b;
        if (kk >= nk2) continue;
        const int q = r * P + (b >> 1);
        T v = (b & 1) ? im[i * B + q] : re[i * B + q];
        const int j = r == 0 ? jp : jhalf + jp;
        int ia = i + 3, k = kk + 1;
        int ks[3] = {k, -1, -1};
        if (kk == 0) ks[1] = 0;
        if (kk == nk2 - 1) ks[2] = g.NZ - 1;
        for (int t = 0; t < 3; t++) {
            if (ks[t] < 0) continue;
            PI[IX(ia, j, ks[t])] = v;
            if (ia >= shift && ia < shift + 3) PI[IX(ia - shift, j, ks[t])] = v;
            if (ia >= 3 && ia < 6) PI[IX(ia + shift, j, ks[t])] = v;
        }
    }
}

template <typename T, int MAXB>
__global__ void __launch_bounds__(kThreadsX) k_irfft_x_out_pair(Geo g, const T *__restrict__ spec, T *__restrict__ PI, Radix rad,
                                                               const double *tw, int nk2, int kc, int jhalf) {
    extern __shared__ unsigned char smem[];
    const TileXY t = xcd_tile_xy();
    irfft_x_out_pair_block<T, MAXB>(g, spec, PI, rad, tw, nk2, kc, t.x, t.y, smem, jhalf);
}

// Q2 on half slabs (even nj, L = nj/2): the j transform's first radix-2 split (decimation in frequency)
// is done while loading, so block (kx, h) holds only a_h(j') = (x(j') + (-1)^h x(j'+L)) W^(h j'),
// W = exp(-2 pi i / nj), j' < L, whose length-L transform is X(2m + h).  It solves the columns
// ky = 2m + h, transforms back, and stores v_h(j') = conj(W)^(h j') u_h(j') in rows h L + j' of `out`; the
// inverse along i combines row j of the full inverse as v_0(j') + (-1)^q v_1(j'), j = j' + qL.  Both
// blocks of a kx read every row of `in`, so they write to a second array.
template <typename T, bool TR>
__device__ __forceinline__ void ypass_half_block(const T *__restrict__ in, T *__restrict__ out, int nk2, const Radix &rh,
                                                 const double *twy, const ThomasArgs &ta, int pad, int kx, int h, unsigned char *smem) {
    const int L = rh.n, nj = 2 * L, P2 = nk2 + pad;
    T *re = (T *)smem, *im = re + L * P2;
    double *mean = (double *)(re + 2 * L * P2);
    T *twl = (T *)(mean + 4 * nk2 + 1);
    const ThomasCoef co = thomas_coef(ta, nk2, mean + 2 * nk2);
    // the length-L table is every other entry of the length-nj one
    for (int e = threadIdx.x; e < L; e += blockDim.x) {
        twl[2 * e] = T(twy[4 * e]);
        twl[2 * e + 1] = T(twy[4 * e + 1]);
    }
    const long long base = (long long)kx * nj * nk2 * 2, second = 2LL * L * nk2;
    // kU elements per thread per round, every global load of a round issued (clamped indices) before any
    // is used: a load behind the loop's bound check made the compiler wait for each in turn
    constexpr int kU = 4;
    const int ne = L * nk2, nt = (int)blockDim.x;
    for (int idx0 = (int)threadIdx.x; idx0 < ne; idx0 += kU * nt) {
        T a[kU][4];
        double w[kU][2];
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const int idx = min(idx0 + u * nt, ne - 1), jp = idx / nk2;
            const long long o = base + 2LL * idx;
            ld2(in + o, a[u][0], a[u][1]);
            ld2(in + o + second, a[u][2], a[u][3]);
            if (h == 1) {
                w[u][0] = twy[2 * jp];
                w[u][1] = twy[2 * jp + 1];
            }
        }
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const int idx = idx0 + u * nt, jp = idx / nk2, kk = idx - jp * nk2;
            T ar, ai;
            if (h == 0) {
                ar = a[u][0] + a[u][2];
                ai = a[u][1] + a[u][3];
            } else {
                const T dr = a[u][0] - a[u][2], di = a[u][1] - a[u][3];
                ar = dr;
                ai = di;
                cmul(ar, ai, T(w[u][0]), T(w[u][1]));
            }
            if (idx < ne) {
                re[jp * P2 + kk] = ar;
                im[jp * P2 + kk] = ai;
            }
        }
    }
    __syncthreads();
    lds_fft_pow2<T, half_maxb<T>()>(re, im, rh, nk2, P2, 1, twl, -1);
    if ((int)threadIdx.x < 2 * L) {
        const int part = (int)threadIdx.x >= L, m = (int)threadIdx.x - part * L;
        T *x = (part ? im : re) + m * P2;
        const double *Z = ta.zpiv + (long long)kx * nj * nk2 + 2 * m + h;
        if (TR) thomas_part_t<T>(ta, co, kx, 2 * m + h, Z, nj, x, 1);
        else thomas_part<T>(ta, co, kx, 2 * m + h, Z, nj, x, 1, mean + part);
    }
    __syncthreads();
    lds_fft_pow2<T, half_maxb<T>()>(re, im, rh, nk2, P2, 1, twl, +1);
    for (int idx0 = (int)threadIdx.x; idx0 < ne; idx0 += kU * nt) {
        T vr[kU], vi[kU];
        double w[kU][2];
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const int idx = min(idx0 + u * nt, ne - 1), jp = idx / nk2, kk = idx - jp * nk2;
            vr[u] = re[jp * P2 + kk];
            vi[u] = im[jp * P2 + kk];
            if (h == 1) {
                w[u][0] = twy[2 * jp];
                w[u][1] = twy[2 * jp + 1];
            }
        }
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const int idx = idx0 + u * nt;
            if (h == 1) cmul(vr[u], vi[u], T(w[u][0]), -T(w[u][1]));
            if (idx < ne) {
                st2(out + base + 2LL * ((long long)h * L * nk2 + idx), vr[u], vi[u]);
            }
        }
    }
}

template <typename T, bool TR = false>
__global__ void __launch_bounds__(half_threads<T>()) k_ypass_half(const T *__restrict__ in, T *__restrict__ out, int nk2, Radix rh,
                                                                   const double *twy, ThomasArgs ta, int pad) {
    extern __shared__ unsigned char smem[];
    ypass_half_block<T, TR>(in, out, nk2, rh, twy, ta, pad, blockIdx.x >> 1, blockIdx.x & 1, smem);
}

template <typename T, bool TR>
__global__ void __launch_bounds__(ypass_threads<T>()) k_ypass(T *__restrict__ spec, int nk2, Radix rady, const double *twy, ThomasArgs ta,
                                                              int pad) {
    extern __shared__ unsigned char smem[];
    ypass_block<T, TR>(spec, nk2, rady, twy, ta, pad, blockIdx.x, smem);
}

// Q2 by matrix products (dyn_dft.hpp): the whole (j, k) slab of one kx in LDS as rows of 2 nk2 doubles (real
// and imaginary parts side by side), in place throughout: rows i and n-i hold E(i) and D(i) while the
// products run, X(i) and X(n-i) afterwards.  A wavefront keeps up to PT tiles' results in registers across
// the barrier before they replace the operands; the last columns of a tile past 2 nk2 hold the next row's
// values and their results are dropped.  The bits are those of k_dft_y, k_thomas_staged and k_dft_y in turn
// (64 bits from the first products to the sweeps' results, which are rounded to the storage type).
// One launch serves slabs of few tiles (a pair of products per wavefront, PT = 1: 48x48x40 FP32 a step of 138 us
// against 143 with three launches, and the radix passes, a chain of two barriers per radix, take 19 us
// instead of 14); with more, the matrix units of nkx CUs are outrun by three launches spread over all of them
// (a step at 96x96x40 FP32, forced to products, 206 against 181 us), except in an ensemble's batch.
inline int dft_y_tiles(int nk2) { return (2 * nk2 + 15) / 16; }
inline int dft_y_pairs(int n, int nk2) { return dft_pad(n) / 16 * dft_y_tiles(nk2); }  // (row tile, column tile)
// doubles per row: 14 or 18 modulo 32, so that the two rows a half-wavefront of the products reads overlap in
// few banks and the sweeps' columns (one row apart) in none
__host__ __device__ __forceinline__ int ypass_dft_pitch(int nk2) {
    int p = 2 * nk2;
    while (p % 32 != 14 && p % 32 != 18) p += 2;
    return p;
}
inline size_t ypass_dft_lds(int n, int nk2) { return 8 * ((size_t)n * ypass_dft_pitch(nk2) + 16 + 4 * (size_t)nk2); }
constexpr int kYDftWaves = 16, kEnsYDftPairs = 3;

// whether a slab fits the LDS and `pt` pairs of products per wavefront, with a thread per sequence of the sweeps
inline bool ypass_dft_fits(const PressurePlan &pp, int pt) {
    return ypass_dft_lds(pp.nj, pp.nk2) <= pp.lds_max && dft_y_pairs(pp.nj, pp.nk2) <= kYDftWaves * pt && 2 * pp.nj <= 64 * kYDftWaves;
}

template <typename T, bool TR, int PT>
__device__ __forceinline__ void ypass_dft_block(T *__restrict__ spec, int n, const double *__restrict__ tab, int nk2, const ThomasArgs &ta,
                                                int kx, unsigned char *smem) {
    const int pitch = ypass_dft_pitch(nk2), h = dft_rows(n), p = dft_pad(n), steps = (h + 3) / 4, ncol = 2 * nk2, nct = (ncol + 15) / 16;
    double *X = (double *)smem, *mean = X + n * pitch + 16;
    const ThomasCoef co = thomas_coef(ta, nk2, mean + 2 * nk2);
    T *x = spec + (long long)kx * n * ncol;
    const int nt = (int)blockDim.x;
    // load and fold row pairs (i, n-i); kU pairs per thread per round, their loads issued together
    constexpr int kU = 4;
    for (int i0 = (int)threadIdx.x; i0 < h * nk2; i0 += kU * nt) {
        T a[kU][2], m[kU][2];
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const int idx = min(i0 + u * nt, h * nk2 - 1), i = idx / nk2, kk = idx - i * nk2, im = i == 0 ? 0 : n - i;
            ld2(x + (long long)i * ncol + 2 * kk, a[u][0], a[u][1]);
            ld2(x + (long long)im * ncol + 2 * kk, m[u][0], m[u][1]);
        }
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const int idx = i0 + u * nt, i = idx / nk2, kk = idx - i * nk2;
            if (idx >= h * nk2) break;
            const bool self = i == 0 || 2 * i == n;
            double *e = X + i * pitch + 2 * kk;
            if (self) {
                e[0] = double(a[u][0]);
                e[1] = double(a[u][1]);
            } else {
                double *d = X + (n - i) * pitch + 2 * kk;
                e[0] = double(a[u][0]) + double(m[u][0]);
                e[1] = double(a[u][1]) + double(m[u][1]);
                d[0] = double(a[u][0]) - double(m[u][0]);
                d[1] = double(a[u][1]) - double(m[u][1]);
            }
        }
    }
    if ((int)threadIdx.x < 16) X[n * pitch + threadIdx.x] = 0.0;
    __syncthreads();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, row = lane >> 4, col = lane & 15;
    const int pairs = p / 16 * nct, per = (pairs + kYDftWaves - 1) / kYDftWaves;  // a wavefront's pairs are consecutive
    dvec4 pc[PT], ps[PT];
    auto products = [&]() {
#pragma unroll
        for (int t = 0; t < PT; t++) {
            const int pr = wave * per + t;
            pc[t] = dvec4{0.0, 0.0, 0.0, 0.0};
            ps[t] = dvec4{0.0, 0.0, 0.0, 0.0};
            if (t >= per || pr >= pairs) continue;
            const int m0 = pr / nct * 16, c0 = pr % nct * 16;
            const double *ca = tab + (size_t)row * p + m0 + col, *sa = ca + (size_t)p * p;
            double ac[2][4], as[2][4];
            auto fetch = [&](int k, double (&fc)[4], double (&fs)[4]) {
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const size_t o = (size_t)min(k + u, steps - 1) * 4 * p;
                    fc[u] = ca[o];
                    fs[u] = sa[o];
                }
            };
            auto use = [&](int k, const double (&fc)[4], const double (&fs)[4]) {
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    if (k + u >= steps) break;
                    const int i = (k + u) * 4 + row;  // rows past h-1 meet zeros of the matrices
                    pc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(fc[u], X[i * pitch + c0 + col], pc[t], 0, 0, 0);
                    ps[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(fs[u], X[(i == 0 ? 0 : n - i) * pitch + c0 + col], ps[t], 0, 0, 0);
                }
            };
            fetch(0, ac[0], as[0]);
            for (int k = 0; k < steps; k += 8) {
                fetch(k + 4, ac[1], as[1]);
                use(k, ac[0], as[0]);
                fetch(k + 8, ac[0], as[0]);
                use(k + 4, ac[1], as[1]);
            }
        }
    };
    // put(row, column, value) for every result: X(m) = P + s i Q and X(n-m) = P - s i Q (see k_dft_y)
    auto results = [&](int sign, auto put) {
        const double sg = (lane & 1) != (sign < 0) ? 1.0 : -1.0;
#pragma unroll
        for (int t = 0; t < PT; t++) {
            const int pr = wave * per + t;
            if (t >= per || pr >= pairs) continue;
            const int m0 = pr / nct * 16, q = pr % nct * 16 + col;
#pragma unroll
            for (int v4 = 0; v4 < 4; v4++) {
                const int m = m0 + row + 4 * v4;
                const double o = sg * lane_pair(ps[t][v4]);
                if (m < h && q < ncol) {
                    put(m, q, pc[t][v4] + o);
                    if (m > 0 && 2 * m != n) put(n - m, q, pc[t][v4] - o);
                }
            }
        }
    };
    products();
    __syncthreads();
    results(-1, [&](int r, int q, double v) { X[r * pitch + q] = v; });
    __syncthreads();
    if ((int)threadIdx.x < 2 * n) {  // neighbouring lanes take the real and the imaginary part of a column
        const int ky = (int)threadIdx.x >> 1, part = (int)threadIdx.x & 1;
        const double *Z = ta.zpiv + (long long)kx * n * nk2 + ky;
        double *xc = X + ky * pitch + part;
        if (TR) thomas_part_t<T>(ta, co, kx, ky, Z, n, xc, 2);
        else thomas_part<T>(ta, co, kx, ky, Z, n, xc, 2, mean + part);
    }
    __syncthreads();
    for (int idx = (int)threadIdx.x; idx < (n - 1) / 2 * ncol; idx += nt) {
        const int i = idx / ncol + 1, q = idx - (i - 1) * ncol;
        double *e = X + i * pitch + q, *d = X + (n - i) * pitch + q;
        const double a = *e, m = *d;
        *e = a + m;
        *d = a - m;
    }
    __syncthreads();
    products();
    results(+1, [&](int r, int q, double v) { x[(long long)r * ncol + q] = T(v); });
}
template <typename T, bool TR>
__global__ void __launch_bounds__(64 * kYDftWaves) k_ypass_dft(T *__restrict__ spec, int n, const double *__restrict__ tab, int nk2,
                                                              ThomasArgs ta) {
    extern __shared__ __align__(16) unsigned char smem[];
    ypass_dft_block<T, TR, 1>(spec, n, tab, nk2, ta, blockIdx.x, smem);
}

// ---- batched over the members of an ensemble: one launch per pass, blocks walk a work list that
// concatenates the members' (row, level chunk) or (kx) items -------------------------------------------

constexpr int kEnsTiles = 2;  // column tiles per block of a member's matrix products
// Threads of a batch's j pass: 512 where every member's slab leaves room for two blocks on a CU and its butterflies fit
// (one block's sweeps then run beside the other's transforms: 113 us a launch against 207, 16 FP32 members of 96 to
// 192 points a side and 40 levels), else 1024, and with matrix products
constexpr int kEnsYNarrow = 512;
constexpr int ens_ymaxb(int threads) { return threads == kEnsYNarrow ? 6 : kMaxBY; }
template <typename T, bool DFT, int MAXB>
__global__ void __launch_bounds__(kThreadsX) k_ens_div_rfft_x(const EnsMember *mem, int nmem, EnsRoles roles, int total, double step) {
    extern __shared__ __align__(16) unsigned char smem[];
    {
        const int item = xcd_tile(blockIdx.x, gridDim.x);
        const EnsMember &e = mem[ens_member(mem, nmem, item, &EnsMember::px0)];
        if (DFT && e.dftx) {
            div_dft_x_block<T, kEnsTiles, false>(e.g, e.c, (const T *)e.buf[DYN_U][roles.r[DYN_U][DYN_ROLE_P]],
                                                 (const T *)e.buf[DYN_V][roles.r[DYN_V][DYN_ROLE_P]],
                                                 (const T *)e.buf[DYN_W][roles.r[DYN_W][DYN_ROLE_P]], (T *)e.spec, e.ni, e.dftx, e.nk2, step,
                                                 (const T *)nullptr, item - e.px0, smem);
            return;
        }
        const int local = item - e.px0, nch = (e.nk2 + e.kcx - 1) / e.kcx;
        div_rfft_x_block<T, MAXB>(e.g, e.c, (const T *)e.buf[DYN_U][roles.r[DYN_U][DYN_ROLE_P]], (const T *)e.buf[DYN_V][roles.r[DYN_V][DYN_ROLE_P]],
                            (const T *)e.buf[DYN_W][roles.r[DYN_W][DYN_ROLE_P]], (T *)e.spec, e.rx, e.twx, e.nk2, e.kcx, step,
                            (const T *)nullptr, local / nch, local % nch, smem, e.dfty != nullptr);
    }
}

template <typename T, bool DFT, int MAXB>
__global__ void __launch_bounds__(kThreadsX) k_ens_irfft_x_out(const EnsMember *mem, int nmem, int total) {
    extern __shared__ __align__(16) unsigned char smem[];
    {
        const int item = xcd_tile(blockIdx.x, gridDim.x);
        const EnsMember &e = mem[ens_member(mem, nmem, item, &EnsMember::px0)];
        if (DFT && e.dftx) {
            idft_x_out_block<T, kEnsTiles>(e.g, (const T *)e.spec, (T *)e.pi, e.ni, e.dftx, e.nk2, item - e.px0, smem);
            return;
        }
        const int local = item - e.px0, nch = (e.nk2 + e.kcx - 1) / e.kcx;
        irfft_x_out_block<T, MAXB>(e.g, (const T *)e.spec, (T *)e.pi, e.rx, e.twx, e.nk2, e.kcx, local / nch, local % nch, smem);
    }
}

template <typename T, int THREADS, bool DFT>
__global__ void __launch_bounds__(THREADS) k_ens_ypass(const EnsMember *mem, int nmem, int total) {
    extern __shared__ __align__(16) unsigned char smem[];
    {
        const int item = xcd_tile(blockIdx.x, gridDim.x);
        const EnsMember &e = mem[ens_member(mem, nmem, item, &EnsMember::py0)];
        ThomasArgs ta{e.acoef, e.ccoef, e.zpiv, e.ni, e.nj, e.g.NZ};
        if constexpr (DFT) {
            if (e.ydft) {
                ypass_dft_block<T, false, kEnsYDftPairs>((T *)e.spec, e.nj, e.dfty, e.nk2, ta, item - e.py0, smem);
                return;
            }
        }
        // the generic transform passes (the straight-line power-of-two ones measured no faster here)
        ypass_block<T, false, false, ens_ymaxb(THREADS)>((T *)e.spec, e.nk2, e.ry, e.twy, ta, 1, item - e.py0, smem);
    }
}

// Q2 (staged): tridiagonal solve of tg columns of one kx with their values and pivots in LDS (coalesced in and
// out): the whole block loads and stores, 2 tg of its threads run the sweeps
constexpr int kThomasThreads = 256;
template <typename T, bool TR, typename TI>
__global__ void __launch_bounds__(kThomasThreads) k_thomas_staged(const TI *in, T *spec, int nk2, ThomasArgs ta, int tg) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int P2 = 2 * nk2 + 1;
    double *zl = (double *)smem, *mean = zl + tg * nk2;
    TI *x = (TI *)(mean + 4 * nk2);
    const ThomasCoef co = thomas_coef(ta, nk2, mean + 2 * nk2);
    const int kx = blockIdx.x, ky0 = blockIdx.y * tg;
    const int ncol = min(tg, ta.nj - ky0);
    const long long base = ((long long)kx * ta.nj + ky0) * nk2 * 2;
    const double *zg = ta.zpiv + (long long)kx * ta.nj * nk2 + ky0;
    // kU elements per thread per round, every load of a round issued (clamped indices) before any is used
    constexpr int kU = 5;
    const int ne = ncol * nk2, nt = (int)blockDim.x;
    for (int i0 = (int)threadIdx.x; i0 < ne; i0 += kU * nt) {
        double z[kU];
        TI vr[kU], vi[kU];
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const int idx = min(i0 + u * nt, ne - 1), kk = idx / ncol;
            z[u] = zg[(long long)kk * ta.nj + idx - kk * ncol];
            ld2(in + base + 2LL * idx, vr[u], vi[u]);
        }
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const int idx = min(i0 + u * nt, ne - 1), kk = idx / ncol, col = idx / nk2, k2 = idx - col * nk2;
            zl[kk * tg + idx - kk * ncol] = z[u];
            x[col * P2 + 2 * k2] = vr[u];
            x[col * P2 + 2 * k2 + 1] = vi[u];
        }
    }
    __syncthreads();
    {
        // two threads per column: even lanes the real part, odd lanes the imaginary part (interleaved)
        const int colx = (int)threadIdx.x >> 1, part = threadIdx.x & 1;
        if (colx < ncol) {
            if (TR) thomas_part_t<T>(ta, co, kx, ky0 + colx, zl + colx, tg, x + colx * P2 + part, 2);
            else thomas_part<T>(ta, co, kx, ky0 + colx, zl + colx, tg, x + colx * P2 + part, 2, mean + part);
        }
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < ncol * nk2; idx += blockDim.x) {
        const int col = idx / nk2, kk = idx - col * nk2;
        st2(spec + base + 2LL * idx, T(x[col * P2 + 2 * kk]), T(x[col * P2 + 2 * kk + 1]));
    }
}

// Radix passes of a length-n transform: 4, 2, 3 and 5 first (the butterflies), then the remaining prime
// factors in increasing order (direct sums, dft_radix); false when n needs more than kMaxRad passes.
bool factorize(int n, Radix &rad) {
    rad.n = n;
    rad.nr = 0;
    int m = n;
    while (m > 1 && rad.nr < kMaxRad) {
        int r = (m % 4 == 0) ? 4 : (m % 2 == 0) ? 2 : (m % 3 == 0) ? 3 : (m % 5 == 0) ? 5 : 0;
        if (r == 0) {
            r = 7;
            while (m % r != 0) r++;  // smallest prime factor of m (every smaller factor was divided out)
        }
        rad.r[rad.nr++] = r;
        m /= r;
    }
    return m == 1;
}

int level_chunk(int n, size_t elt, int nk2);
size_t x_pass_lds(int ni, int kc, size_t elt);

int max_butterflies(const Radix &r, int nbatch, int nthr);
// The i passes hold a thread's butterflies of a radix pass in registers: the instance with no more of them than the
// grid's pass needs (FP32 86 registers with four, 69 with three and 52 with two, so two, three and four blocks on a
// CU; FP64 148, 120 and 92, so one, two and two).  192x192x40 FP32 dry 390 -> 345 us a step, 512x256x40 FP64 1867 ->
// 1745.
template <typename T>
auto div_rfft_x_kernel(const Radix &rx, int kc) {
    const int b = max_butterflies(rx, kc / 2, kThreadsX);
    return b <= 2 ? k_div_rfft_x<T, 2> : b <= 3 ? k_div_rfft_x<T, 3> : k_div_rfft_x<T, kMaxBX>;
}
// the inverse i pass into `out`: after the half-slab j pass (half = nj/2) one block per row pair and
// chunk of an even number of levels, at most kc/2 (same LDS and butterflies per thread as kc levels of
// one row); otherwise one block per row and chunk of kc levels
template <typename T>
void launch_irfft_x_out(Ctx *c, const T *spec, T *out, const Radix &rx, int kc, int half) {
    const PressurePlan &pp = c->pp;
    const Geo &g = c->geo;
    const size_t shx = x_pass_lds(pp.ni, kc, sizeof(T));
    const int kcp = (kc / 2) & ~1;
    if (half && kcp >= 2) {
        const int b = max_butterflies(rx, 2 * (kcp / 2), kThreadsX);
        auto k = b <= 2 ? k_irfft_x_out_pair<T, 2> : b <= 3 ? k_irfft_x_out_pair<T, 3> : k_irfft_x_out_pair<T, kMaxBX>;
        hipLaunchKernelGGL(k, dim3(half, (pp.nk2 + kcp - 1) / kcp), dim3(kThreadsX), shx, c->stream, g, spec, out, rx,
                           pp.twx, pp.nk2, kcp, half);
        return;
    }
    const int b = max_butterflies(rx, kc / 2, kThreadsX);
    auto k = b <= 2 ? k_irfft_x_out<T, 2> : b <= 3 ? k_irfft_x_out<T, 3> : k_irfft_x_out<T, kMaxBX>;
    hipLaunchKernelGGL(k, dim3(g.NY, (pp.nk2 + kc - 1) / kc), dim3(kThreadsX), shx, c->stream, g, spec, out, rx, pp.twx,
                       pp.nk2, kc, half);
}

// launches of the matrix-product transforms (dyn_dft.hpp) with 4, 2 or 1 column tiles per block; src: transform
// that field instead of the divergence
template <typename T, int NT>
void launch_div_dft_x_t(Ctx *c, T *spec, double step, const T *src) {
    const PressurePlan &pp = c->pp;
    const int ncol = pp.nj * pp.nk2, nc = 16 * NT;
    const dim3 grid((ncol + nc - 1) / nc), blk(dft_threads(pp.ni));
    const size_t sh = dft_lds(pp.ni, nc);
    if (src) {
        hipLaunchKernelGGL((k_div_dft_x<T, NT, true>), grid, blk, sh, c->stream, c->geo, c->cols, src, src, src, spec, pp.ni, pp.dftx, pp.nk2,
                           step, src);
        return;
    }
    hipLaunchKernelGGL((k_div_dft_x<T, NT, false>), grid, blk, sh, c->stream, c->geo, c->cols, (const T *)c->prog[DYN_U][2],
                       (const T *)c->prog[DYN_V][2], (const T *)c->prog[DYN_W][2], spec, pp.ni, pp.dftx, pp.nk2, step, src);
}
template <typename T>
void launch_div_dft_x(Ctx *c, T *spec, double step, const T *src = nullptr) {
    const int nt = dft_tiles(c->pp.ni, 1, c->pp.nj * c->pp.nk2, c->pp.cus);
    if (nt == 4) launch_div_dft_x_t<T, 4>(c, spec, step, src);
    else if (nt == 2) launch_div_dft_x_t<T, 2>(c, spec, step, src);
    else launch_div_dft_x_t<T, 1>(c, spec, step, src);
}
template <typename T>
int dft_lds_limits() {  // their operands may take more than 64 KiB: kDftMax with one column tile, 80 KiB with more
    const void *k[] = {(const void *)k_div_dft_x<T, 1, false>, (const void *)k_div_dft_x<T, 2, false>, (const void *)k_div_dft_x<T, 4, false>,
                       (const void *)k_div_dft_x<T, 1, true>, (const void *)k_div_dft_x<T, 2, true>, (const void *)k_div_dft_x<T, 4, true>,
                       (const void *)k_idft_x_out<T, 1>, (const void *)k_idft_x_out<T, 2>, (const void *)k_idft_x_out<T, 4>,
                       (const void *)k_dft_y<T, T, 1>, (const void *)k_dft_y<T, T, 2>, (const void *)k_dft_y<T, T, 4>,
                       (const void *)k_dft_y<T, double, 1>, (const void *)k_dft_y<T, double, 2>, (const void *)k_dft_y<T, double, 4>};
    for (const void *f : k) DYN_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024));
    return DYN_OK;
}
template <typename T>
void launch_idft_x_out(Ctx *c, const T *spec, T *out, int half) {
    const PressurePlan &pp = c->pp;
    const int ncol = pp.nj * pp.nk2, nt = dft_tiles(pp.ni, 1, ncol, pp.cus), nc = 16 * nt;
    const dim3 grid((ncol + nc - 1) / nc), blk(dft_threads(pp.ni));
    const size_t sh = dft_lds(pp.ni, nc);
    if (nt == 4) hipLaunchKernelGGL((k_idft_x_out<T, 4>), grid, blk, sh, c->stream, c->geo, spec, out, pp.ni, pp.dftx, pp.nk2, half);
    else if (nt == 2) hipLaunchKernelGGL((k_idft_x_out<T, 2>), grid, blk, sh, c->stream, c->geo, spec, out, pp.ni, pp.dftx, pp.nk2, half);
    else hipLaunchKernelGGL((k_idft_x_out<T, 1>), grid, blk, sh, c->stream, c->geo, spec, out, pp.ni, pp.dftx, pp.nk2, half);
}
template <typename T, typename TO>
void launch_dft_y(Ctx *c, const T *in, TO *out, int nrows, int sign) {
    const PressurePlan &pp = c->pp;
    const int nt = dft_tiles(pp.nj, nrows, 2 * pp.nk2, pp.cus), nc = 16 * nt;
    const dim3 grid(nrows, (2 * pp.nk2 + nc - 1) / nc), blk(dft_threads(pp.nj));
    const size_t sh = dft_lds(pp.nj, nc);
    if (nt == 4) hipLaunchKernelGGL((k_dft_y<T, TO, 4>), grid, blk, sh, c->stream, in, out, pp.nj, pp.dfty, pp.nk2, sign);
    else if (nt == 2) hipLaunchKernelGGL((k_dft_y<T, TO, 2>), grid, blk, sh, c->stream, in, out, pp.nj, pp.dfty, pp.nk2, sign);
    else hipLaunchKernelGGL((k_dft_y<T, TO, 1>), grid, blk, sh, c->stream, in, out, pp.nj, pp.dfty, pp.nk2, sign);
}
// the 64-bit half spectrum between k_dft_y and the sweeps: behind the FP32 one in the plan's buffer
inline size_t wide_spec_at(const PressurePlan &pp) { return ((size_t)(pp.ni / 2 + 1) * pp.nj * pp.nk2 * 8 + 15) & ~(size_t)15; }
inline double *wide_spec(const PressurePlan &pp) { return (double *)((char *)pp.spec + wide_spec_at(pp)); }

// one j transform of the three-kernel j pass over nrows kx rows: the matrix products where the plan has them, the
// power-of-two kernel when nj is a power of two and its plan fits, else the mixed-radix one
template <typename T>
void launch_fft_y(Ctx *c, T *spec, int nrows, const Radix &ry, int sign) {
    const PressurePlan &pp = c->pp;
    if (pp.dfty) {
        if (sizeof(T) == 4 && sign < 0) return launch_dft_y(c, (const T *)spec, wide_spec(pp), nrows, sign);
        return launch_dft_y(c, (const T *)spec, spec, nrows, sign);
    }
    Radix rp{};
    const int kcp = pow2_plan48(pp.nj, rp, true) ? fft_y_pow2_chunk<T>(rp, pp.nk2) : 0;
    if (kcp > 0) {
        hipLaunchKernelGGL((k_fft_y_pow2<T, kFftYMaxB>), dim3(nrows, (pp.nk2 + kcp - 1) / kcp), dim3(kFftYThreads),
                           fft_y_pow2_lds(pp.nj, kcp, sizeof(T)), c->stream, spec, pp.nj, pp.nk2, rp, pp.twy, kcp, sign);
        return;
    }
    const int kcy = level_chunk(pp.nj, sizeof(T), pp.nk2);
    hipLaunchKernelGGL(k_fft_y<T>, dim3(nrows, (pp.nk2 + kcy - 1) / kcy), dim3(kThreads), 4 * (size_t)pp.nj * kcy * sizeof(T), c->stream,
                       spec, pp.nj, pp.nk2, ry, pp.twy, kcy, sign);
}

int level_chunk(int n, size_t elt, int nk2) {
    // two ping-pong buffers of n*kc complex values must fit the LDS budget
    int kc = (int)(kLdsBudget / (4 * (size_t)n * elt));
    if (kc > 32) kc = 32;
    if (kc > nk2) kc = nk2;
    if (kc < 1) kc = 1;
    return kc;
}

double *upload_twiddles(int n, hipStream_t s) {
    std::vector<double> h(2 * (size_t)n);
    for (int e = 0; e < n; e++) {
        double a = 2.0 * kTrigPi * (double)e / (double)n;
        h[2 * e] = std::cos(a);
        h[2 * e + 1] = -std::sin(a);
    }
    double *d = nullptr;
    if (hipMalloc(&d, sizeof(double) * h.size()) != hipSuccess) return nullptr;
    if (hipMemcpy(d, h.data(), sizeof(double) * h.size(), hipMemcpyHostToDevice) != hipSuccess) return nullptr;
    return d;
}

// butterflies a thread holds in the worst pass; a pass of prime radix above 5 holds outputs instead, 5
// per radix-5 butterfly's worth of registers
int max_butterflies(const Radix &r, int nbatch, int nthr) {
    int mb = 0;
    for (int s = 0; s < r.nr; s++) {
        if (r.r[s] > 5) mb = std::max(mb, ((r.n * nbatch + nthr - 1) / nthr + 4) / 5);
        else mb = std::max(mb, (r.n / r.r[s] * nbatch + nthr - 1) / nthr);
    }
    return mb;
}

// LDS of the i passes for kc levels (kc/2 packed pairs) and of the fused j pass, twiddle tables included
size_t x_pass_lds(int ni, int kc, size_t elt) { return (2 * (size_t)ni * (kc / 2) + 2 * (size_t)ni) * elt + 32 * (size_t)kc; }
size_t y_pass_lds(int nj, int nk2, size_t elt) {
    return 2 * (size_t)nj * (nk2 + 1) * elt + 8 * (4 * (size_t)nk2 + 1) + 2 * (size_t)nj * elt + 8;
}
// levels per block of the i passes (even: two levels per complex transform), within the LDS budget and
// the butterflies a thread holds.  One grid alone wants enough blocks to fill the chip (about 512 rows x
// chunks); a batch of members has blocks to spare, so there every row takes all its levels at once
// (`fill` false), which keeps the row segments long.
int x_level_chunk(const PressurePlan &pp, const Geo &g, const Radix &rx, size_t elt, bool fill = true) {
    int kc = (int)((kLdsBudget - 2 * (size_t)pp.ni * elt) / (2 * (size_t)pp.ni * elt)) * 2;
    // about 512 blocks per pass in FP32; FP64 takes half the levels per block down to 16 (256x256x64:
    // 1.909 -> 1.869 ms per step with 16 levels instead of 30; FP32 is slower with fewer than 32, and
    // FP64 at 192x192x40 with 6 instead of 14)
    int want = fill ? std::max(2, ((pp.nk2 * g.NY / 512) + 1) & ~1) : (pp.nk2 + 1) & ~1;
    if (fill && elt == 8 && want > 16) want = std::max(16, (want / 2) & ~1);
    kc = std::max(2, std::min(kc, want));
    while (kc > 2 && (max_butterflies(rx, kc / 2, kThreadsX) > kMaxBX || x_pass_lds(pp.ni, kc, elt) > kLdsBudget)) kc -= 2;
    return kc;
}

// The j pass of a solve while no form is asked for: the one-slab form by matrix products where a slab has few
// tiles, three launches with them up to kDftYThree (96x96x40 FP64: 210 us per step against 235 with the radix
// passes' slab; 96x96x48 FP32: 42 us a solve with products on both sides against 53), the nominal forms beyond
// (128x128x64 FP32: the slab takes 26 us, three launches 38).
int jpass_in_use(const Ctx *c) {
    if (c->tune[DYN_TUNE_PRESSURE_JPASS]) return fused_shape(c, DYN_TUNE_PRESSURE_JPASS);
    if (c->pp.ydft) return 1;
    // (in FP32 a product along i goes with one along j, see pressure_init)
    const bool three = c->pp.nj <= kDftYThree || (c->prec == DYN_FP32 && c->pp.dftx);
    return c->pp.dfty && three ? 2 : fused_shape(c, DYN_TUNE_PRESSURE_JPASS);
}
// LDS of k_thomas_staged for tg columns; columns per block: 32 (64 running threads, one wavefront), fewer
// where their values and pivots exceed half the LDS of a CU
size_t thomas_lds(int tg, int nk2, size_t elt) { return 8 * ((size_t)tg * nk2 + 4 * (size_t)nk2) + (size_t)tg * (2 * (size_t)nk2 + 1) * elt; }
int thomas_group(int nk2, size_t elt) {
    int tg = 32;
    while (tg > 1 && thomas_lds(tg, nk2, elt) > 80 * 1024) tg /= 2;
    return tg;
}
template <typename T, bool TR>
void launch_thomas(Ctx *c, T *spec, int nkx) {
    const PressurePlan &pp = c->pp;
    const bool wide = sizeof(T) == 4 && pp.dfty;  // the products left the spectrum in 64 bits
    const size_t elt = wide ? 8 : sizeof(T);
    const int tg = thomas_group(pp.nk2, elt);
    const dim3 grid(nkx, (pp.nj + tg - 1) / tg);
    const size_t sh = thomas_lds(tg, pp.nk2, elt);
    if (wide)
        hipLaunchKernelGGL((k_thomas_staged<T, TR, double>), grid, dim3(kThomasThreads), sh, c->stream, (const double *)wide_spec(pp), spec,
                           pp.nk2, thomas_args(pp, c->g.nz), tg);
    else
        hipLaunchKernelGGL((k_thomas_staged<T, TR, T>), grid, dim3(kThomasThreads), sh, c->stream, (const T *)spec, spec, pp.nk2,
                           thomas_args(pp, c->g.nz), tg);
}
// the LDS-resident j pass: by matrix products where the plan has them, else by radix passes
template <typename T, bool TR>
void launch_ypass(Ctx *c, T *spec, int nkx, const Radix &ry) {
    const PressurePlan &pp = c->pp;
    const ThomasArgs ta = thomas_args(pp, c->g.nz);
    if (pp.ydft) {
        hipLaunchKernelGGL((k_ypass_dft<T, TR>), dim3(nkx), dim3(64 * kYDftWaves), ypass_dft_lds(pp.nj, pp.nk2), c->stream, spec, pp.nj,
                           pp.dfty, pp.nk2, ta);
        return;
    }
    hipLaunchKernelGGL((k_ypass<T, TR>), dim3(nkx), dim3(ypass_threads<T>()), y_pass_lds(pp.nj, pp.nk2, sizeof(T)), c->stream, spec, pp.nk2,
                       ry, pp.twy, ta, 1);
}

template <typename T>
int solve_t(Ctx *c, double step, bool halos, PressureHook after_i, void *arg) {
    PressurePlan &pp = c->pp;
    const Geo &g = c->geo;
    Radix rx{}, ry{};
    factorize(pp.ni, rx);
    factorize(pp.nj, ry);
    if (halos) {  // periodic_uvw_boundaries (boundaries.cpp:546-555)
        void *uvw[3] = {c->prog[DYN_U][2], c->prog[DYN_V][2], c->prog[DYN_W][2]};
        int rc = launch_periodic(c, uvw, 3);
        if (rc) return rc;
    }
    T *spec = (T *)pp.spec;
    const double pts = (double)pp.ni * pp.nj * pp.nk2;
    const ThomasArgs ta = thomas_args(pp, c->g.nz);
    // half-spectrum transforms, except along i for lengths with a prime factor above 5 that have no matrix
    // products: those take the full complex spectrum
    if (pp.smooth_x || pp.dftx) {
        const int nkx = pp.ni / 2 + 1;
        const int kc = x_level_chunk(pp, g, rx, sizeof(T));
        const size_t shx = x_pass_lds(pp.ni, kc, sizeof(T));
        dim3 gx(g.NY, (pp.nk2 + kc - 1) / kc);
        if (pp.dftx) {
            Timed _t(c, "p1_div_dft_x", pts);
            launch_div_dft_x<T>(c, spec, step);
        } else {
            Timed _t(c, "p1_div_rfft_x", pts);
            hipLaunchKernelGGL(div_rfft_x_kernel<T>(rx, kc), gx, dim3(kThreadsX), shx, c->stream, g, c->cols, (const T *)c->prog[DYN_U][2],
                               (const T *)c->prog[DYN_V][2], (const T *)c->prog[DYN_W][2], spec, rx, pp.twx, pp.nk2, kc, step,
                               (const T *)nullptr, pp.dfty != nullptr);
        }
        DYN_LAUNCH_CHECK();
        if (after_i) {
            const int rc = after_i(c, arg);
            if (rc) return rc;
        }
        const int pad = 1;
        const int jpass = jpass_in_use(c);
        int half = 0;
        if (jpass == 1) {
            Timed _t(c, pp.ydft ? "p2_ypass_dft" : "p2_ypass", pts);
            launch_ypass<T, false>(c, spec, nkx, ry);
            DYN_LAUNCH_CHECK();
        } else if (jpass == 3) {
            Radix rh{};
            pow2_plan48(pp.nj / 2, rh, sizeof(T) == 8);
            half = pp.nj / 2;
            Timed _t(c, "p2_ypass", pts);
            hipLaunchKernelGGL((k_ypass_half<T>), dim3(2 * nkx), dim3(half_threads<T>()), y_pass_lds(half, pp.nk2, sizeof(T)), c->stream,
                               (const T *)spec, (T *)pp.spec2, pp.nk2, rh, pp.twy, ta, pad);
            DYN_LAUNCH_CHECK();
        } else {
            {
                Timed _t(c, pp.dfty ? "p2_dft_y" : "p2_fft_y", pts);
                launch_fft_y<T>(c, spec, nkx, ry, -1);
            }
            DYN_LAUNCH_CHECK();
            {
                Timed _t(c, "p3_thomas", pts);
                launch_thomas<T, false>(c, spec, nkx);
            }
            DYN_LAUNCH_CHECK();
            {
                Timed _t(c, pp.dfty ? "p4_idft_y" : "p4_ifft_y", pts);
                launch_fft_y<T>(c, spec, nkx, ry, +1);
            }
            DYN_LAUNCH_CHECK();
        }
        if (pp.dftx) {
            Timed _t(c, "p5_idft_x_out", pts);
            launch_idft_x_out<T>(c, half ? (const T *)pp.spec2 : spec, (T *)c->pi, half);
        } else {
            Timed _t(c, "p5_irfft_x_out", pts);
            launch_irfft_x_out<T>(c, half ? (const T *)pp.spec2 : spec, (T *)c->pi, rx, kc, half);
        }
        DYN_LAUNCH_CHECK();
        return DYN_OK;
    }
    // full complex spectrum, out-of-place transforms
    int kcx = level_chunk(pp.ni, sizeof(T), pp.nk2), kcy = level_chunk(pp.nj, sizeof(T), pp.nk2);
    size_t shx = 4 * (size_t)pp.ni * kcx * sizeof(T), shy = 4 * (size_t)pp.nj * kcy * sizeof(T);
    dim3 gx(g.NY, (pp.nk2 + kcx - 1) / kcx), gy(pp.ni, (pp.nk2 + kcy - 1) / kcy);
    {
        Timed _t(c, "p1_div_fft_x", pts);
        hipLaunchKernelGGL(k_div_fft_x<T>, gx, dim3(kThreads), shx, c->stream, g, c->cols, (const T *)c->prog[DYN_U][2],
                           (const T *)c->prog[DYN_V][2], (const T *)c->prog[DYN_W][2], spec, rx, pp.twx, pp.nk2, kcx, step);
    }
    DYN_LAUNCH_CHECK();
    if (after_i) {
        const int rc = after_i(c, arg);
        if (rc) return rc;
    }
    {
        Timed _t(c, "p2_fft_y", pts);
        hipLaunchKernelGGL(k_fft_y<T>, gy, dim3(kThreads), shy, c->stream, spec, pp.nj, pp.nk2, ry, pp.twy, kcy, -1);
    }
    DYN_LAUNCH_CHECK();
    int nq = pp.ni * pp.nj;
    {
        Timed _t(c, "p3_thomas", pts);
        hipLaunchKernelGGL(k_thomas<T>, dim3((nq + 127) / 128), dim3(128), 0, c->stream, spec, pp.ni, pp.nj, g.NZ, pp.acoef, pp.ccoef,
                           pp.zpiv);
    }
    DYN_LAUNCH_CHECK();
    {
        Timed _t(c, "p4_ifft_y", pts);
        hipLaunchKernelGGL(k_fft_y<T>, gy, dim3(kThreads), shy, c->stream, spec, pp.nj, pp.nk2, ry, pp.twy, kcy, +1);
    }
    DYN_LAUNCH_CHECK();
    {
        Timed _t(c, "p5_ifft_x_out", pts);
        hipLaunchKernelGGL(k_ifft_x_out<T>, gx, dim3(kThreads), shx, c->stream, g, (const T *)spec, (T *)c->pi, rx, pp.twx, pp.nk2, kcx);
    }
    DYN_LAUNCH_CHECK();
    return DYN_OK;
}


// ---- adjoint of the solve (transposed projection for the hand-written adjoint) -----------------------
// Transpose of the pressure-gradient force (solver.cpp:123-135) over [1,NX-1) x [1,NY-1), which gathers PI's adjoint
// at a point from the forecast velocities' (they pass through), and of P5's output stage: the value v(i, j, kk)
// was written to PI at (i+3, j, kk+1), at the ghost level 0 (kk = 0) or NZ-1 (kk = nk2-1), and at the periodic halo
// copies; its adjoint is the sum of the adjoints of every location it was written to.
template <typename T>
__global__ void k_adj_pi_fold(Geo g, Cols c, const T *__restrict__ UH, const T *__restrict__ VH, const T *__restrict__ WH,
                              T *__restrict__ R, int nk2, T step) {
    // levels, rows and columns one after another over the lanes
    const unsigned q = (unsigned)xcd_tile(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x, row = q / (unsigned)nk2;
    const int kk = (int)(q - row * (unsigned)nk2), j = (int)(row % (unsigned)g.NY), ia = (int)(row / (unsigned)g.NY) + 3;
    if (ia >= g.NX - 3) return;
    auto inr = [&](int ii, int jj, int kz) { return ii >= 1 && ii < g.NX - 1 && jj >= 1 && jj < g.NY - 1 && kz >= 1 && kz <= g.NZ - 2; };
    const T sx = step * T(g.dtx), sy = step * T(g.dty);
    auto pgf = [&](int i, int k) -> T {
        const long long p = IX(i, j, k);
        T acc = T(0);
        if (inr(i, j, k)) acc -= sx * UH[p] + sy * VH[p];
        if (inr(i + 1, j, k)) acc += sx * UH[p + g.NYNZ];
        if (inr(i, j + 1, k)) acc += sy * VH[p + g.NZ];
        if (inr(i, j, k) && k >= 2) acc -= step * (T(g.dtz) * T(c.mw[k])) * WH[p];
        if (inr(i, j, k + 1) && k + 1 >= 2) acc += step * (T(g.dtz) * T(c.mw[k + 1])) * WH[p + 1];
        return acc;
    };
    const int shift = g.NX - 6, k = kk + 1;
    const int ks[3] = {k, kk == 0 ? 0 : -1, kk == nk2 - 1 ? g.NZ - 1 : -1};
    T v = T(0);
    for (int t = 0; t < 3; t++) {
        if (ks[t] < 0) continue;
        v += pgf(ia, ks[t]);
        if (ia >= shift && ia < shift + 3) v += pgf(ia - shift, ks[t]);
        if (ia >= 3 && ia < 6) v += pgf(ia + shift, ks[t]);
    }
    R[IX(ia, j, k)] = v;
}

// Transpose of P1's divergence prologue (divergence3d_periodic, pressure.cpp:1390-1424): the adjoint of the
// right-hand side r(ia, j, k) (rows 0 and NY-1 fold onto the mirrored rows 1 and NY-2) is spread back onto
// the forecast velocities, one gathering thread per velocity point.
template <typename T>
__global__ void k_adj_div(Geo g, Cols c, const T *__restrict__ R, T *__restrict__ UH, T *__restrict__ VH, T *__restrict__ WH,
                          double step) {
    const long long q = (long long)xcd_tile(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    if (q >= (long long)g.NX * g.NYNZ) return;
    const int x = (int)(q / g.NYNZ), r = (int)(q - (long long)x * g.NYNZ), y = r / g.NZ, k = r - y * g.NZ;
    const T sdt = T(step * g.dt);
    auto Rf = [&](int ia, int yy, int kk) -> T {
        if (ia < 3 || ia >= g.NX - 3 || yy < 1 || yy > g.NY - 2 || kk < 1 || kk > g.NZ - 2) return T(0);
        T v = R[IX(ia, yy, kk)];
        if (yy == 1) v += R[IX(ia, 0, kk)];
        if (yy == g.NY - 2) v += R[IX(ia, g.NY - 1, kk)];
        return v;
    };
    T uh = T(0), vh = T(0), wh = T(0);
    if (x >= 3 && x < g.NX - 3 && k >= 1 && k <= g.NZ - 2) {
        const T a = T(c.rhou[k]) * T(g.one_d_dx) / sdt, b = T(c.rhou[k]) * T(g.one_d_dy) / sdt;
        // UP(x) enters column ia as UP(ie) with ie = ia + 1 (ie = 3 for ia = NX-4) and as UP(ia)
        const int iae = x == 3 ? g.NX - 4 : x - 1;
        uh = a * (Rf(iae, y, k) - Rf(x, y, k));
        vh = b * (Rf(x, y - 1, k) - Rf(x, y, k));
    }
    if (x >= 3 && x < g.NX - 3) {
        const T rw = T(c.rhow[k]), odz = T(g.one_d_dz);
        if (k >= 2) wh += rw * (odz * T(c.mu[k - 1])) * Rf(x, y, k - 1) / sdt;
        if (k >= 1 && k <= g.NZ - 2) wh -= rw * (odz * T(c.mu[k])) * Rf(x, y, k) / sdt;
    }
    const long long p = IX(x, y, k);
    UH[p] += uh;
    VH[p] += vh;
    WH[p] += wh;
}

template <typename T>
int solve_adjoint_t(Ctx *c, double step, T *uh, T *vh, T *wh, T *r1, T *r2) {
    PressurePlan &pp = c->pp;
    const Geo &g = c->geo;
    if (pp.ni % 2 != 0 || !pp.smooth_x) {
        set_error("adjoint pressure solve: needs an even ni of factors 2, 3 and 5 (half-spectrum transform), got ni=" +
                  std::to_string(pp.ni));
        return DYN_E_UNSUPPORTED;
    }
    Radix rx{}, ry{};
    factorize(pp.ni, rx);
    factorize(pp.nj, ry);
    const double pts = (double)pp.ni * pp.nj * pp.nk2;
    {
        Timed _t(c, "adj_pi_fold", pts);
        hipLaunchKernelGGL(k_adj_pi_fold<T>, dim3((unsigned)(((long long)pp.ni * g.NY * pp.nk2 + 255) / 256)), dim3(256), 0, c->stream, g,
                           c->cols, (const T *)uh, (const T *)vh, (const T *)wh, r1, pp.nk2, T(step));
        DYN_LAUNCH_CHECK();
    }
    T *spec = (T *)pp.spec;
    const ThomasArgs ta = thomas_args(pp, c->g.nz);
    const int nkx = pp.ni / 2 + 1;
    const int kc = x_level_chunk(pp, g, rx, sizeof(T));
    const size_t shx = x_pass_lds(pp.ni, kc, sizeof(T));
    dim3 gx(g.NY, (pp.nk2 + kc - 1) / kc);
    if (pp.dftx) {
        Timed _t(c, "adj_dft_x", pts);
        launch_div_dft_x<T>(c, spec, step, (const T *)r1);
    } else {
        Timed _t(c, "adj_rfft_x", pts);
        hipLaunchKernelGGL(div_rfft_x_kernel<T>(rx, kc), gx, dim3(kThreadsX), shx, c->stream, g, c->cols, (const T *)nullptr, (const T *)nullptr,
                           (const T *)nullptr, spec, rx, pp.twx, pp.nk2, kc, step, (const T *)r1, false);
    }
    DYN_LAUNCH_CHECK();
    const int pad = 1;
    const int jpass = jpass_in_use(c);
    int half = 0;
    if (jpass == 1) {
        Timed _t(c, pp.ydft ? "adj_ypass_dft" : "adj_ypass", pts);
        launch_ypass<T, true>(c, spec, nkx, ry);
        DYN_LAUNCH_CHECK();
    } else if (jpass == 3) {
        Radix rh{};
        pow2_plan48(pp.nj / 2, rh, sizeof(T) == 8);
        half = pp.nj / 2;
        Timed _t(c, "adj_ypass", pts);
        hipLaunchKernelGGL((k_ypass_half<T, true>), dim3(2 * nkx), dim3(half_threads<T>()), y_pass_lds(half, pp.nk2, sizeof(T)),
                           c->stream, (const T *)spec, (T *)pp.spec2, pp.nk2, rh, pp.twy, ta, pad);
        DYN_LAUNCH_CHECK();
    } else {
        Timed _t(c, pp.dfty ? "adj_dft_y" : "adj_ypass", pts);
        launch_fft_y<T>(c, spec, nkx, ry, -1);
        DYN_LAUNCH_CHECK();
        launch_thomas<T, true>(c, spec, nkx);
        DYN_LAUNCH_CHECK();
        launch_fft_y<T>(c, spec, nkx, ry, +1);
        DYN_LAUNCH_CHECK();
    }
    {
        Timed _t(c, "adj_irfft_x", pts);
        if (pp.dftx) launch_idft_x_out<T>(c, half ? (const T *)pp.spec2 : spec, r2, half);
        else launch_irfft_x_out<T>(c, half ? (const T *)pp.spec2 : spec, r2, rx, kc, half);
    }
    DYN_LAUNCH_CHECK();
    {
        Timed _t(c, "adj_div", (double)c->npts);
        hipLaunchKernelGGL(k_adj_div<T>, dim3((unsigned)(((long long)g.NX * g.NYNZ + 255) / 256)), dim3(256), 0, c->stream, g, c->cols,
                           (const T *)r2, uh, vh, wh, step);
    }
    DYN_LAUNCH_CHECK();
    return DYN_OK;
}

template <typename T>
int y_lds_limits(int most) {
    const void *k[] = {(const void *)k_ypass<T, false>, (const void *)k_ypass<T, true>, (const void *)k_thomas_staged<T, false, T>,
                       (const void *)k_thomas_staged<T, true, T>, (const void *)k_thomas_staged<T, false, double>,
                       (const void *)k_thomas_staged<T, true, double>, (const void *)k_ypass_dft<T, false>, (const void *)k_ypass_dft<T, true>};
    for (const void *f : k) DYN_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, most));
    return DYN_OK;
}

}  // namespace

// Bytes of a spectrum buffer: the full complex spectrum in 64 bits, or the two half spectra of an FP32 context's products
// (more than that on the narrowest grids)
size_t pressure_spec_bytes(const PressurePlan &pp) {
    const size_t col = (size_t)pp.nj * pp.nk2 * 2 * sizeof(double);
    return std::max(col * pp.ni, wide_spec_at(pp) + col * (pp.ni / 2 + 1));
}

int pressure_init(Ctx *c) {
    PressurePlan &pp = c->pp;
    const int NZ = c->g.nz;
    pp.ni = c->g.nx - 6;
    pp.nj = c->g.ny;
    pp.nk2 = NZ - 2;
    Radix rx{}, ry{};
    if (!factorize(pp.ni, rx) || !factorize(pp.nj, ry)) {
        set_error("pressure solver: transform sizes need at most 8 radix passes (ni=" + std::to_string(pp.ni) +
                  ", nj=" + std::to_string(pp.nj) + ")");
        return DYN_E_UNSUPPORTED;
    }
    auto smooth = [](const Radix &r) {
        for (int q = 0; q < r.nr; q++)
            if (r.r[q] > 5) return false;
        return true;
    };
    pp.smooth_x = smooth(rx);
    pp.smooth_y = smooth(ry);
    pp.twx = upload_twiddles(pp.ni, c->stream);
    pp.twy = upload_twiddles(pp.nj, c->stream);
    if (!pp.twx || !pp.twy) {
        set_error("pressure solver: twiddle upload failed");
        return DYN_E_HIP;
    }
    DYN_HIP(hipMalloc(&pp.spec, pressure_spec_bytes(pp)));
    int dev = 0, lds = 0;
    DYN_HIP(hipGetDevice(&dev));
    DYN_HIP(hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
    pp.lds_max = (size_t)lds;
    DYN_HIP(hipDeviceGetAttribute(&pp.cus, hipDeviceAttributeMultiprocessorCount, dev));
    // the fused j pass keeps a whole (j, k) slab of one kx in LDS when it fits (FP32 at 256x64, FP64 up to
    // about 192x40) and one thread per real sequence of the solve exists; otherwise the j transforms and
    // the solve run as three kernels
    const size_t need = y_pass_lds(pp.nj, pp.nk2, c->elt);
    const bool f32 = c->prec == DYN_FP32;
    const int nthr = f32 ? ypass_threads<float>() : ypass_threads<double>();
    const int maxb = f32 ? ypass_maxb<float>() : ypass_maxb<double>();
    pp.fused_y = pp.smooth_y && need <= pp.lds_max && 2 * pp.nj <= nthr && max_butterflies(ry, pp.nk2, nthr) <= maxb;
    // Which sides go by matrix products: lengths with a prime factor above 5, and short smooth ones.
    // FP32 is choosier.  The longest waves' columns are nearly singular systems, the more so the wider the domain is
    // for its depth, and what a factored FP32 transform rounds away on one side the products' 64 bits on the
    // other don't give back (pi of 160x128x40, 6 steps, is 2 to 6e-6 off a 64-bit run either way, at 313 and
    // 314 us a step).  So smooth sides (even along i) take products on both or on neither, and only in domains up
    // to twice as many points wide as deep, where the change of rounding stays at 1e-5 of pi and below (2e-4 at
    // 190x190x12 after two steps).  Dry domains wider than that keep the passes without products whatever their
    // factors.  Neither time nor the accuracy of a solve speaks for that: with the same winds, a dry context and a
    // moist one (which takes the products) give, us a solve and pi's rms distance from a 64-bit solve, 303 and 2.3e-7
    // against 95 and 5.7e-8 at 184x150x57, 449 and 2.1e-7 against 57 and 7.6e-8 at 194x100x40, 589 and 6.1e-7 against
    // 36 and 6.9e-8 at 97x97x40, 39 and 1.7e-6 against 32 and 1.1e-6 at 45x75x30.  It keeps the results of dry
    // runs: their pi is 2e-5 to 8e-4 off a 64-bit run after two steps by the winds' own rounding, whatever the
    // transforms, and a change of transform moves it by as much.
    // Dry grids with smooth sides past 64 points keep those passes at every width that an ensemble can hold: its
    // members' bits are those of runs alone, and a batch of 32 members of 96 to 192 points takes 4.82 ms a step
    // without products and 4.87 with them.  Single runs pay for it (us a solve without and with products, 46 and 36
    // at 72x72x40, 44 and 37 at 80x80x40, 53 and 42 at 96x96x48); batches of members of 65 to 95 points were not
    // measured.
    const int widest = std::max(pp.ni, pp.nj);
    const bool shallow = widest > 2 * c->g.nz, dry = !c->g.microphysics;
    bool prod_x = pp.ni <= (!pp.smooth_x ? kDftMax : f32 ? dft_x_smooth<float>() : dft_x_smooth<double>());
    bool prod_y = pp.nj <= (!pp.smooth_y ? kDftMax : kDftYSmooth);
    if (f32 && pp.smooth_x && pp.smooth_y && pp.ni % 2 == 0) {
        const bool y_taken = prod_y && (pp.nj <= kDftYThree || !pp.fused_y);
        const bool batched = dry && fused_waves(c) == 1 && widest > 64;
        prod_x = prod_y = prod_x && y_taken && !shallow && !batched;
    } else if (f32 && dry && shallow) {
        prod_x = prod_y = false;
    }
    auto matrices = [](int n, double **out) -> int {
        const std::vector<double> h = dft_matrices(n);
        DYN_HIP(hipMalloc(out, sizeof(double) * h.size()));
        DYN_HIP(hipMemcpy(*out, h.data(), sizeof(double) * h.size(), hipMemcpyHostToDevice));
        return DYN_OK;
    };
    int rc = prod_x ? matrices(pp.ni, &pp.dftx) : DYN_OK;
    if (!rc && prod_y) rc = matrices(pp.nj, &pp.dfty);
    if (!rc && (pp.dftx || pp.dfty)) rc = f32 ? dft_lds_limits<float>() : dft_lds_limits<double>();
    if (rc) return rc;
    pp.ydft = pp.dfty && ypass_dft_fits(pp, 1);
    rc = f32 ? y_lds_limits<float>(lds) : y_lds_limits<double>(lds);
    if (rc) return rc;
    // half slabs (power-of-two nj/2): what a slab of nj/2 rows needs, with one thread per real sequence
    // of the solve
    if (pp.nj % 2 == 0 && pp.nj >= 4 && ((pp.nj / 2) & (pp.nj / 2 - 1)) == 0) {
        Radix rh{};
        const bool ok = pow2_plan48(pp.nj / 2, rh, !f32);
        const size_t needh = y_pass_lds(pp.nj / 2, pp.nk2, c->elt);
        const int hthr = f32 ? half_threads<float>() : half_threads<double>();
        const int hmaxb = f32 ? half_maxb<float>() : half_maxb<double>();
        bool fits = ok && needh <= pp.lds_max && pp.nj <= hthr;
        for (int st = 0; fits && st < rh.nr; st++) {  // butterflies a thread holds in each pass
            const int items = rh.n / rh.r[st] * pp.nk2, per = (items + hthr - 1) / hthr;
            fits = per <= (rh.r[st] == 8 ? pow2_maxb8(hmaxb) : hmaxb);
        }
        pp.half_y = fits && pp.smooth_x;
        if (pp.half_y) {
            DYN_HIP(hipMalloc(&pp.spec2, sizeof(double) * 2 * (size_t)pp.ni * pp.nj * pp.nk2));
            if (f32) {
                DYN_HIP(hipFuncSetAttribute((const void *)k_ypass_half<float>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)needh));
                DYN_HIP(hipFuncSetAttribute((const void *)k_ypass_half<float, true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)needh));
            } else {
                DYN_HIP(hipFuncSetAttribute((const void *)k_ypass_half<double>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)needh));
                DYN_HIP(hipFuncSetAttribute((const void *)k_ypass_half<double, true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)needh));
            }
        }
    }
    // the power-of-two j transforms of the three-kernel j pass may take more than 64 KiB of LDS
    if (f32) DYN_HIP(hipFuncSetAttribute((const void *)k_fft_y_pow2<float, kFftYMaxB>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kFftYLds));
    else DYN_HIP(hipFuncSetAttribute((const void *)k_fft_y_pow2<double, kFftYMaxB>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kFftYLds));
    DYN_HIP(hipMalloc(&pp.zpiv, sizeof(double) * (size_t)pp.ni * pp.nj * pp.nk2));
    DYN_HIP(hipMalloc(&pp.coskx, sizeof(double) * pp.ni));
    DYN_HIP(hipMalloc(&pp.cosly, sizeof(double) * pp.nj));
    DYN_HIP(hipMalloc(&pp.acoef, sizeof(double) * NZ));
    DYN_HIP(hipMalloc(&pp.ccoef, sizeof(double) * NZ));
    // cos(kwave[i]), cos(lwave[j]) exactly as init_fft3d forms them (pressure.cpp:751-752)
    std::vector<double> ck(pp.ni), cl(pp.nj);
    for (int i = 0; i < pp.ni; i++) ck[i] = std::cos((double)i * 2 * kTrigPi / ((double)pp.ni));
    for (int j = 0; j < pp.nj; j++) cl[j] = std::cos((double)j * 2 * kTrigPi / ((double)pp.nj));
    DYN_HIP(hipMemcpy(pp.coskx, ck.data(), sizeof(double) * pp.ni, hipMemcpyHostToDevice));
    DYN_HIP(hipMemcpy(pp.cosly, cl.data(), sizeof(double) * pp.nj, hipMemcpyHostToDevice));
    return DYN_OK;
}

// coefficients that depend on the columns (acoef, ccoef, F2): called once the columns are set
int pressure_coefficients(Ctx *c) {
    PressurePlan &pp = c->pp;
    const int nk = c->g.nz;
    const double dz = c->g.dz;
    const double *mu = c->colhost + (size_t)DYN_COL_MU * nk, *mw = c->colhost + (size_t)DYN_COL_MW * nk;
    const double *rhow = c->colhost + (size_t)DYN_COL_RHOW * nk;
    std::vector<double> a(nk, 0.0), cc(nk, 0.0);
    for (int k = 1; k < nk - 1; k++) {
        a[k] = mu[k] * mw[k] * rhow[k] / (dz * dz);
        cc[k] = mu[k] * mw[k + 1] * rhow[k + 1] / (dz * dz);
    }
    a[1] = 0;
    cc[nk - 2] = 0;
    DYN_HIP(hipMemcpy(pp.acoef, a.data(), sizeof(double) * nk, hipMemcpyHostToDevice));
    DYN_HIP(hipMemcpy(pp.ccoef, cc.data(), sizeof(double) * nk, hipMemcpyHostToDevice));
    int nq = pp.ni * pp.nj;
    hipLaunchKernelGGL(k_thomas_factors, dim3((nq + 127) / 128), dim3(128), 0, c->stream, pp.ni, pp.nj, nk, pp.coskx, pp.cosly,
                       c->cols.rhou, c->cols.rhow, c->cols.mu, c->cols.mw, pp.acoef, pp.ccoef, c->g.dx, dz, pp.zpiv);
    DYN_LAUNCH_CHECK();
    DYN_HIP(hipStreamSynchronize(c->stream));
    return DYN_OK;
}

int pressure_free(Ctx *c) {
    PressurePlan &pp = c->pp;
    void *ptrs[] = {pp.twx, pp.twy, pp.dftx, pp.dfty, pp.spec, pp.spec2, pp.zpiv, pp.coskx, pp.cosly, pp.acoef, pp.ccoef};
    for (void *p : ptrs)
        if (p) (void)hipFree(p);
    pp = PressurePlan{};
    return DYN_OK;
}

// the form of the j pass in force (the full complex spectrum has the one with three kernels)
int pressure_jpass(const Ctx *c) { return c->pp.smooth_x || c->pp.dftx ? jpass_in_use(c) : 2; }

int launch_solve_pressure(Ctx *c, double step, bool halos, PressureHook after_i, void *arg) {
    return c->prec == DYN_FP32 ? solve_t<float>(c, step, halos, after_i, arg) : solve_t<double>(c, step, halos, after_i, arg);
}



// the pressure part of an ensemble member's table entry; false when the member cannot join the batched
// solve (FP64, the full complex spectrum, or a (j, k) slab too large for the LDS-resident j pass)
bool pressure_ens_fill(Ctx *c, EnsMember &e, size_t &lds_x, size_t &lds_y) {
    PressurePlan &pp = c->pp;
    const int jpass = jpass_in_use(c);
    const bool by_products = (jpass == 1 && pp.ydft) || (jpass == 2 && pp.dfty);
    if (c->prec != DYN_FP32 || (!pp.smooth_x && !pp.dftx) || (by_products ? !ypass_dft_fits(pp, kEnsYDftPairs) : jpass != 1)) return false;
    if (!factorize(pp.ni, e.rx) || !factorize(pp.nj, e.ry)) return false;
    e.kcx = x_level_chunk(pp, c->geo, e.rx, sizeof(float), false);
    e.ni = pp.ni;
    e.nj = pp.nj;
    e.nk2 = pp.nk2;
    e.spec = pp.spec;
    e.twx = pp.twx;
    e.twy = pp.twy;
    e.zpiv = pp.zpiv;
    e.acoef = pp.acoef;
    e.ccoef = pp.ccoef;
    // by matrix products where the member's own solve takes them, so its bits are those of a step on its own
    e.dftx = pp.dftx;
    e.dfty = pp.dfty;
    e.ydft = by_products;
    e.pxn = pp.dftx ? (pp.nj * pp.nk2 + 16 * kEnsTiles - 1) / (16 * kEnsTiles) : c->g.ny * ((pp.nk2 + e.kcx - 1) / e.kcx);
    lds_x = pp.dftx ? dft_lds(pp.ni, 16 * kEnsTiles) : x_pass_lds(pp.ni, e.kcx, sizeof(float));
    if (pp.dftx && lds_x > pp.lds_max) return false;
    e.xform = pp.dftx ? 2 : max_butterflies(e.rx, e.kcx / 2, kThreadsX) <= 3 ? 0 : 1;
    if (e.ydft) {
        lds_y = ypass_dft_lds(pp.nj, pp.nk2);
        return true;
    }
    lds_y = y_pass_lds(pp.nj, pp.nk2, sizeof(float));
    e.ynarrow = 2 * lds_y <= pp.lds_max && 2 * pp.nj <= kEnsYNarrow && max_butterflies(e.ry, pp.nk2, kEnsYNarrow) <= ens_ymaxb(kEnsYNarrow);
    return lds_y <= pp.lds_max && 2 * pp.nj <= 1024 && max_butterflies(e.ry, pp.nk2, 1024) <= kMaxBY;
}

// the batched passes may take more than 64 KiB of LDS
int pressure_ens_prepare(const Ctx *c) {
    const void *k[] = {(const void *)k_ens_div_rfft_x<float, false, 3>, (const void *)k_ens_irfft_x_out<float, false, 3>,
                       (const void *)k_ens_div_rfft_x<float, false, kMaxBX>, (const void *)k_ens_irfft_x_out<float, false, kMaxBX>,
                       (const void *)k_ens_div_rfft_x<float, true, kMaxBX>, (const void *)k_ens_irfft_x_out<float, true, kMaxBX>,
                       (const void *)k_ens_ypass<float, kEnsYNarrow, false>,
                       (const void *)k_ens_ypass<float, 1024, false>, (const void *)k_ens_ypass<float, 1024, true>};
    for (const void *f : k) DYN_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)c->pp.lds_max));
    return DYN_OK;
}

// solve_pressure(step) of every member without the uvw halo copy (as in the fused step): three launches
int launch_pressure_ens(Ctx *c0, const EnsMember *d, int nmem, const EnsRoles &ro, double step, int tot_px, int tot_py, size_t lds_x,
                        size_t lds_y, int xform, int yform) {
    {
        const int grid = tot_px;
        Timed _t(c0, "ens_p1_div_rfft_x", 0.0);
        auto k = xform == 0   ? k_ens_div_rfft_x<float, false, 3>
                 : xform == 1 ? k_ens_div_rfft_x<float, false, kMaxBX>
                              : k_ens_div_rfft_x<float, true, kMaxBX>;
        hipLaunchKernelGGL(k, dim3(grid), dim3(kThreadsX), lds_x, c0->stream, d, nmem, ro, tot_px, step);
        DYN_LAUNCH_CHECK();
    }
    {
        const int grid = tot_py;
        Timed _t(c0, "ens_p2_ypass", 0.0);
        auto k = yform == 0 ? k_ens_ypass<float, kEnsYNarrow, false> : yform == 1 ? k_ens_ypass<float, 1024, false> : k_ens_ypass<float, 1024, true>;
        hipLaunchKernelGGL(k, dim3(grid), dim3(yform == 0 ? kEnsYNarrow : 1024), lds_y, c0->stream, d, nmem, tot_py);
        DYN_LAUNCH_CHECK();
    }
    {
        const int grid = tot_px;
        Timed _t(c0, "ens_p5_irfft_x_out", 0.0);
        auto k = xform == 0   ? k_ens_irfft_x_out<float, false, 3>
                 : xform == 1 ? k_ens_irfft_x_out<float, false, kMaxBX>
                              : k_ens_irfft_x_out<float, true, kMaxBX>;
        hipLaunchKernelGGL(k, dim3(grid), dim3(kThreadsX), lds_x, c0->stream, d, nmem, tot_px);
        DYN_LAUNCH_CHECK();
    }
    return DYN_OK;
}

// adjoint of the gradient force and of solve_pressure(step) minus its periodic_uvw_boundaries: PI's adjoint from the
// forecast-velocity adjoints, to which the adjoint of the divergence input is added; r1, r2 are scratch fields of
// the context's element type
int launch_pressure_adjoint(Ctx *c, double step, void *uh, void *vh, void *wh, void *r1, void *r2) {
    if (c->prec == DYN_FP32)
        return solve_adjoint_t<float>(c, step, (float *)uh, (float *)vh, (float *)wh, (float *)r1, (float *)r2);
    return solve_adjoint_t<double>(c, step, (double *)uh, (double *)vh, (double *)wh, (double *)r1, (double *)r2);
}

}  // namespace dyn
