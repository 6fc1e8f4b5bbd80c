// Turbulence parameterization (turbulence.cpp, USE_TURBULENT_STRESS) for the serial periodic path
// without terrain or surface heat flux: mixing coefficients and stored tendencies at the start of each
// step (calculate_diff_tend, driver_serial.cpp:194), added to the forecasts in every stage
// (apply_velocity_diffusion, solver.cpp:104; apply_scalar_diffusion / apply_moisture_diffusion,
// driver_serial.cpp:218, 231).  The fused step adds them inside its stage kernels; the per-operator one
// through the kernels at the end of this file.
//
// The reference walks i-slabs and carries the stress tensor of slab i-1 over as the west stress of slab
// i, and the flux through the top of a level over as the bottom flux of the level above.  Every such
// value is a pure function of its position, so here one thread computes one point and re-evaluates the
// stress components and fluxes it needs; the values are those of the carried ones, in the reference's
// expression order (the library is built without FMA contraction).
#include <cmath>

#include "dyn_internal.hpp"

namespace dyn {
namespace {

constexpr double kCmixV = 0.15, kCmixH = 0.05;   // turbulence.cpp:48-49
constexpr double kPrInv = 3.0, kLvMax = 200.0, kCs = 0.25;  // turbulence.cpp:56-58

// (the tendencies in the order of DYN_U .. DYN_QR)
enum { TK = 0, TKH, TUF, TVF, TWF, TTD, TQV, TQC, TQR, TCOUNT };

struct TurbArgs {
    const double *vml2, *vkmax, *landsea;
    double kmixh_max, lH;
};

// the fields the coefficients and tendencies read: the M buffers, the basic state, pi and the
// saturation flags Kessler leaves
template <typename T>
struct TurbIn {
    const T *um, *vm, *wm, *thm, *qvm, *qcm, *qrm;
    const T *ub, *vb, *wb, *thb, *qb, *pb, *pi;
    const unsigned char *sat;
    int moist;
};

#define IX3(i, j, k) ((long long)(i) * g.NYNZ + (long long)(j) * g.NZ + (k))

// Threads take the levels of neighbouring columns one after another (kTurbThreads of them, whole columns while a
// column fits), so that a 40-level column leaves no lanes idle, and a block stays in one i-slab: the slabs' bases
// are scalars and one 32-bit offset per thread reaches every neighbour.  Consecutive blocks sit behind one L2.
constexpr int kTurbThreads = 256;

// a point's neighbours: at(F, di, dj, dk)
template <typename T>
struct Near {
    long long slab;  // i * NYNZ
    long long nynz;
    int nz;
    unsigned o;      // j * NZ + k
    __device__ __forceinline__ T operator()(const T *F, int di, int dj, int dk) const {
        const T *b = F + (slab + di * nynz);
        return *(const T *)((const char *)b + (size_t)((o + (unsigned)(dj * nz + dk)) * (unsigned)sizeof(T)));
    }
};

template <typename T>
__device__ __forceinline__ T odz(const Geo &g, const Cols &c, int k) { return T(g.one_d_dz) * T(c.mu[k]); }
template <typename T>
__device__ __forceinline__ T odzw(const Geo &g, const Cols &c, int k) { return T(g.one_d_dz) * T(c.mw[k]); }

// S^2 = D11^2 + ... + D23^2, turbulence.cpp:596-624
template <typename T>
__device__ __forceinline__ T deformation2(const Geo &g, const Cols &c, const TurbIn<T> &f, const Near<T> &A, int k) {
    const T *UM = f.um, *VM = f.vm, *WM = f.wm, *UB = f.ub, *VB = f.vb, *WB = f.wb;
    const T odx = T(g.one_d_dx), ody = T(g.one_d_dy), dzw = odzw<T>(g, c, k);
    T D11 = T(0.50) * (A(UM, 1, 0, 0) + A(UM, 1, 0, -1) - A(UM, -1, 0, 0) - A(UM, -1, 0, -1) +
                       A(UB, 1, 0, 0) + A(UB, 1, 0, -1) - A(UB, -1, 0, 0) - A(UB, -1, 0, -1)) * odx;
    T D22 = T(0.50) * (A(VM, 0, 1, 0) + A(VM, 0, 1, -1) - A(VM, 0, -1, 0) - A(VM, 0, -1, -1) +
                       A(VB, 0, 1, 0) + A(VB, 0, 1, -1) - A(VB, 0, -1, 0) - A(VB, 0, -1, -1)) * ody;
    T D33 = T(1.0) * (A(WM, 0, 0, 1) - A(WM, 0, 0, -1) + A(WB, 0, 0, 1) - A(WB, 0, 0, -1)) * dzw;
    T D12 = T(0.5) * ((A(UM, 0, 1, 0) + A(UM, 0, 1, -1) - A(UM, 0, -1, 0) - A(UM, 0, -1, -1) +
                       A(UB, 0, 1, 0) + A(UB, 0, 1, -1) - A(UB, 0, -1, 0) - A(UB, 0, -1, -1)) * ody +
                      (A(VM, 1, 0, 0) + A(VM, 1, 0, -1) - A(VM, -1, 0, 0) - A(VM, -1, 0, -1) +
                       A(VB, 1, 0, 0) + A(VB, 1, 0, -1) - A(VB, -1, 0, 0) - A(VB, -1, 0, -1)) * odx);
    T D13 = T(0.5) * ((A(UM, 0, 0, 0) + A(UM, 1, 0, 0) - A(UM, 0, 0, -1) - A(UM, 1, 0, -1) +
                       A(UB, 0, 0, 0) + A(UB, 1, 0, 0) - A(UB, 0, 0, -1) - A(UB, 1, 0, -1)) * dzw +
                      (A(WM, 1, 0, 0) - A(WM, -1, 0, 0) + A(WB, 1, 0, 0) - A(WB, -1, 0, 0)) * odx);
    T D23 = T(0.5) * ((A(VM, 0, 0, 0) + A(VM, 0, 1, 0) - A(VM, 0, 0, -1) - A(VM, 0, 1, -1) +
                       A(VB, 0, 0, 0) + A(VB, 0, 1, 0) - A(VB, 0, 0, -1) - A(VB, 0, 1, -1)) * dzw +
                      (A(WM, 0, 1, 0) - A(WM, 0, -1, 0) + A(WB, 0, 1, 0) - A(WB, 0, -1, 0)) * ody);
    return D11 * D11 + D22 * D22 + D33 * D33 + D12 * D12 + D13 * D13 + D23 * D23;
}

// What the stability of a level needs of each of the two it lies between: the virtual potential temperature,
// and where the air is saturated the temperature and the potential temperature of the moist form (with its
// pow and exp, so they are worth forming once a level)
template <typename T>
struct StabilityLevel {
    T thetav, temp, thetam;
    int sat;
};
template <typename T>
__device__ __forceinline__ StabilityLevel<T> stability_level(const Geo &g, const Cols &c, const TurbIn<T> &f, const Near<T> &A,
                                                             long long h, int k) {
    StabilityLevel<T> s;
    s.sat = f.moist ? f.sat[h] : 0;
    T qh = f.moist ? A(f.qvm, 0, 0, 0) + A(f.qb, 0, 0, 0) + T(c.qb[k]) : T(c.qb[k]);
    T th = A(f.thm, 0, 0, 0) + A(f.thb, 0, 0, 0) + T(c.tb[k]);
    s.thetav = th * (T(1) + T(0.61) * qh);
    s.temp = T(0);
    s.thetam = T(0);
    if (s.sat) {
        const T cp = T(kCp), Lv = T(kLv);
        const T cpRd = T(kCp / kRd);
        const T pbh = A(f.pb, 0, 0, 0), pih = A(f.pi, 0, 0, 0);
        s.temp = th * (pbh + pih / (cp * T(c.tbv[k])));
        T pd = T(kP0) * pow(pbh, cpRd) + pih * T(c.rhou[k]);
        T esl = T(611.2) * exp(T(17.67) * (s.temp - T(273.15)) / (s.temp - T(29.65)));
        T qvsat = T(0.62197) * esl / (pd - esl);
        s.thetam = th * (T(1) + Lv * qvsat / (cp * s.temp));
    }
    return s;
}

// Brunt-Vaisala frequency: get_Kmix_dry (turbulence.cpp:781-791), get_Kmix (:627-690), from the levels k (H) and
// k-1 (L)
template <typename T>
__device__ __forceinline__ T brunt_vaisala(const Geo &g, const Cols &c, const TurbIn<T> &f, const Near<T> &A, const StabilityLevel<T> &H,
                                           const StabilityLevel<T> &L, int k) {
    if (!H.sat || !L.sat) {
        T dTheta = H.thetav - L.thetav;
        return T(2.0) * T(kGrav) / (T(c.tbv[k]) + T(c.tbv[k - 1])) * dTheta * odzw<T>(g, c, k);
    }
    const T cp = T(kCp), Lv = T(kLv), Rd = T(kRd), grav = T(kGrav);
    T temp = T(0.5) * (H.temp + L.temp);
    T dQL = A(f.qcm, 0, 0, 0) + A(f.qrm, 0, 0, 0) - A(f.qcm, 0, 0, -1) - A(f.qrm, 0, 0, -1) + A(f.qvm, 0, 0, 0) - A(f.qvm, 0, 0, -1) +
            A(f.qb, 0, 0, 0) - A(f.qb, 0, 0, -1) + T(c.qb[k]) - T(c.qb[k - 1]);
    T qv = T(0.5) * (A(f.qvm, 0, 0, 0) + A(f.qvm, 0, 0, -1) + A(f.qb, 0, 0, 0) + A(f.qb, 0, 0, -1) + T(c.qb[k]) + T(c.qb[k - 1]));
    T dTheta = H.thetam - L.thetam;
    T Acoef = (grav / T(c.tbw[k])) * (T(1.0) + Lv * qv / (Rd * temp)) / (T(1.0) + T(0.622) * Lv * Lv * qv / (cp * Rd * temp * temp));
    return (Acoef * dTheta - grav * dQL) * odzw<T>(g, c, k);
}

// get_Kmix / get_Kmix_dry, turbulence.cpp:563-831: one thread per level; the horizontal coefficient of level
// k-1 is set with level k, from level k-1's final and level k's raw value (levels 1 and NZ-1 are 0).  What a
// level hands the one above goes through LDS, so the deformation and the moist thermodynamics of a level are
// formed once (194x100x40 FP32 38 -> 16 us, 150x126x50 FP64 95 -> 44; the rest is the 60 neighbour
// loads of the deformation, from L1 and L2).  Columns longer than the block take several, which overlap by one level.
template <typename T>
__global__ void __launch_bounds__(kTurbThreads) k_turb_kmix(Geo g, Cols c, TurbIn<T> f, TurbArgs ta, T *__restrict__ K, T *__restrict__ KH,
                                                            int il, int jl, int jh, int rows, int nbj, int nbk) {
    __shared__ StabilityLevel<T> lev[kTurbThreads];
    __shared__ T lfin[kTurbThreads];
    const int t = xcd_tile(blockIdx.x, gridDim.x);
    const int kb = t % nbk, jb = t / nbk % nbj, i = t / (nbk * nbj) + il;
    const int q = threadIdx.x, per = min(g.NZ, kTurbThreads), k0 = kb * (kTurbThreads - 1);
    const int r = q / per, k = k0 + q - r * per, j = jl + jb * rows + r;
    const bool in = r < rows && j < jh && k < g.NZ;
    const Near<T> A{(long long)i * g.NYNZ, g.NYNZ, g.NZ, in ? (unsigned)(j * g.NZ + k) : 0u};
    const long long p = A.slab + A.o;
    StabilityLevel<T> H{};
    if (in && k >= 1 && k <= g.NZ - 2) H = stability_level<T>(g, c, f, A, p, k);
    lev[q] = H;
    __syncthreads();
    // raw and final (bounded) coefficient of level k; a block's first level has no level below in LDS: 1 has
    // the value 0, and further up it is the overlap, whose final value is formed from memory
    T raw = T(0), fin = T(0);
    if (in && k >= 2 && k <= g.NZ - 2) {
        StabilityLevel<T> L;
        if (q > 0) {
            L = lev[q - 1];
        } else {
            Near<T> B = A;
            B.o -= 1;
            L = stability_level<T>(g, c, f, B, p - 1, k - 1);
        }
        T S2 = deformation2<T>(g, c, f, A, k);
        T bruntv = brunt_vaisala<T>(g, c, f, A, H, L, k);
        if (S2 - T(kPrInv) * bruntv > T(0)) {
            T cc = T(ta.vml2[k]) * T(kCs) * T(kCs);
            raw = cc * sqrt(S2 - T(kPrInv) * bruntv);
            fin = raw > T(ta.vkmax[k]) ? T(ta.vkmax[k]) : raw;
        }
    }
    lfin[q] = fin;
    __syncthreads();
    if (!in || k < 1 || (kb > 0 && q == 0)) return;
    K[p] = fin;
    if (k == 1 || k == g.NZ - 1) return;
    const T finl = lfin[q - 1];
    const T lH = T(ta.lH);
    T kh;
    if (raw > T(0)) {
        kh = T(0.5) * (finl / T(ta.vml2[k - 1]) + raw / T(ta.vml2[k])) * lH * lH;
        if (kh > T(ta.kmixh_max)) kh = T(ta.kmixh_max);
    } else {
        kh = T(0) + T(0.5) * finl / T(ta.vml2[k - 1]) * lH * lH;
    }
    KH[p - 1] = kh;
}

// Stress components at (i + di, j + dj, k + dk) (turbulence.cpp:913-933); k is the level of the point `A` stands on,
// level 0 of tau_33, tau_13, tau_23 is zero
template <typename T>
struct Stress {
    const Geo &g;
    const Cols &c;
    const TurbIn<T> &f;
    const Near<T> &A;
    int k;
    __device__ __forceinline__ T t11(int di, int dj, int dk) const {
        return T(2.0) * (A(f.um, di + 1, dj, dk) - A(f.um, di, dj, dk)) * T(g.one_d_dx);
    }
    __device__ __forceinline__ T t22(int di, int dj, int dk) const {
        return T(2.0) * (A(f.vm, di, dj + 1, dk) - A(f.vm, di, dj, dk)) * T(g.one_d_dy);
    }
    __device__ __forceinline__ T t33(int dk) const {
        return k + dk < 1 ? T(0) : T(2.0) * (A(f.wm, 0, 0, dk + 1) - A(f.wm, 0, 0, dk)) * odz<T>(g, c, k + dk);
    }
    __device__ __forceinline__ T t13(int di, int dj, int dk) const {
        if (k + dk < 1) return T(0);
        return (A(f.wm, di + 1, dj, dk + 1) - A(f.wm, di, dj, dk + 1)) * T(g.one_d_dx) +
               (A(f.um, di + 1, dj, dk + 1) - A(f.um, di + 1, dj, dk)) * odzw<T>(g, c, k + dk + 1);
    }
    __device__ __forceinline__ T t23(int di, int dj, int dk) const {
        if (k + dk < 1) return T(0);
        return (A(f.wm, di, dj + 1, dk + 1) - A(f.wm, di, dj, dk + 1)) * T(g.one_d_dy) +
               (A(f.vm, di, dj + 1, dk + 1) - A(f.vm, di, dj + 1, dk)) * odzw<T>(g, c, k + dk + 1);
    }
    __device__ __forceinline__ T t12(int di, int dj, int dk) const {
        return (A(f.um, di + 1, dj + 1, dk) - A(f.um, di + 1, dj, dk)) * T(g.one_d_dy) +
               (A(f.vm, di + 1, dj + 1, dk) - A(f.vm, di, dj + 1, dk)) * T(g.one_d_dx);
    }
};

// The tendencies at (i, j, k), k in [1, NZ-1), in one pass (they share the coefficients):
//   turbulent_diffusion_velocity, turbulence.cpp:839-1020: friction of u, v, w; the bottom flux of level 1 is the
//   bulk surface stress (turbulence.cpp:885-907);
//   turbulent_diffusion_theta / turbulent_diffusion_scalars, turbulence.cpp:1027-1276: theta (and qv, qc, qr); no
//   flux through the ground.
// Bound by the neighbour loads (40 of the winds and coefficients, 7 a scalar); measured with the packed
// lanes and the one pass against a kernel each and a wavefront a column: 194x100x40 FP32 40 -> 25 us,
// 150x126x50 FP64 88 -> 58.
template <typename T>
__global__ void __launch_bounds__(kTurbThreads) k_turb_tendencies(Geo g, Cols c, TurbIn<T> f, TurbArgs ta, const T *__restrict__ K,
                                                                  const T *__restrict__ KH, T *__restrict__ UF, T *__restrict__ VF,
                                                                  T *__restrict__ WF, T *__restrict__ TD, T *__restrict__ QVD,
                                                                  T *__restrict__ QCD, T *__restrict__ QRD, int il, int jl, int jh, int nbq) {
    const int t = xcd_tile(blockIdx.x, gridDim.x);
    const int i = t / nbq + il;
    const int n = g.NZ - 2, q = t % nbq * kTurbThreads + threadIdx.x;  // (row, active level) of the slab
    const int r = q / n, j = jl + r, k = q - r * n + 1;
    if (j >= jh) return;
    const Near<T> A{(long long)i * g.NYNZ, g.NYNZ, g.NZ, (unsigned)(j * g.NZ + k)};
    const Stress<T> tau{g, c, f, A, k};
    const long long p = A.slab + A.o;
    const T odx = T(g.one_d_dx), ody = T(g.one_d_dy);
    auto KM = [&](int di, int dj, int dk) -> T { return A(K, di, dj, dk); };
    auto KHM = [&](int di, int dj, int dk) -> T { return A(KH, di, dj, dk); };
    T tau_u_zl, tau_v_zl;
    if (k == 1) {
        const T um = A(f.um, 0, 0, 0), ub = A(f.ub, 0, 0, 0), vm = A(f.vm, 0, 0, 0), vb = A(f.vb, 0, 0, 0);
        T wind_speed = sqrt((um + ub) * (um + ub) + (vm + vb) * (vm + vb));
        T wind_speed_base = sqrt(ub * ub + vb * vb);
        if (ta.landsea[(long long)i * g.NY + j] < 0.5) {
            tau_u_zl = T(0.003) * (wind_speed * um + (wind_speed - wind_speed_base) * ub);
            tau_v_zl = T(0.003) * (wind_speed * vm + (wind_speed - wind_speed_base) * vb);
        } else {
            T drag_coef = (T(1.1e-3) + T(4.0e-5) * wind_speed);
            tau_u_zl = drag_coef * (wind_speed * um + (wind_speed - wind_speed_base) * ub);
            tau_v_zl = drag_coef * (wind_speed * vm + (wind_speed - wind_speed_base) * vb);
        }
    } else {  // the top flux of level k-1
        T uK13V_l = T(0.50) * (KM(0, 0, 0) + KM(-1, 0, 0));
        T vK23V_l = T(0.5) * (KM(0, 0, 0) + KM(0, -1, 0));
        tau_u_zl = uK13V_l * tau.t13(-1, 0, -1);
        tau_v_zl = vK23V_l * tau.t23(0, -1, -1);
    }
    T uK11H_h = KHM(0, 0, 0);
    T uK11H_l = KHM(-1, 0, 0);
    T uK12H_h = T(0.25) * (KHM(0, 0, 0) + KHM(-1, 0, 0) + KHM(-1, 1, 0) + KHM(0, 1, 0));
    T uK12H_l = T(0.25) * (KHM(0, -1, 0) + KHM(-1, -1, 0) + KHM(-1, 0, 0) + KHM(0, 0, 0));
    T uK13V_h = T(0.50) * (KM(0, 0, 1) + KM(-1, 0, 1));
    T vK12H_h = T(0.25) * (KHM(0, -1, 0) + KHM(0, 0, 0) + KHM(1, -1, 0) + KHM(1, 0, 0));
    T vK12H_l = uK12H_l;
    T vK22H_h = KHM(0, 0, 0);
    T vK22H_l = KHM(0, -1, 0);
    T vK23V_h = T(0.5) * (KM(0, 0, 1) + KM(0, -1, 1));
    T wK13H_h = T(0.25) * (KHM(0, 0, 0) + KHM(0, 0, -1) + KHM(1, 0, 0) + KHM(1, 0, -1));
    T wK13H_l = T(0.25) * (KHM(0, 0, 0) + KHM(0, 0, -1) + KHM(-1, 0, 0) + KHM(-1, 0, -1));
    T wK23H_h = T(0.25) * (KHM(0, 0, 0) + KHM(0, 0, -1) + KHM(0, 1, 0) + KHM(0, 1, -1));
    T wK23H_l = T(0.25) * (KHM(0, 0, 0) + KHM(0, 0, -1) + KHM(0, -1, 0) + KHM(0, -1, -1));
    T wK33V_h = T(0.50) * (KM(0, 0, 0) + KM(0, 0, 1));
    T wK33V_l = T(0.50) * (KM(0, 0, 0) + KM(0, 0, -1));
    T ufric = (uK11H_h * tau.t11(0, 0, 0) - uK11H_l * tau.t11(-1, 0, 0)) * odx +
              (uK12H_h * tau.t12(-1, 0, 0) - uK12H_l * tau.t12(-1, -1, 0)) * ody +
              (uK13V_h * tau.t13(-1, 0, 0) - tau_u_zl) * odz<T>(g, c, k);
    T vfric = (vK12H_h * tau.t12(0, -1, 0) - vK12H_l * tau.t12(-1, -1, 0)) * odx +
              (vK22H_h * tau.t22(0, 0, 0) - vK22H_l * tau.t22(0, -1, 0)) * ody +
              (vK23V_h * tau.t23(0, -1, 0) - tau_v_zl) * odz<T>(g, c, k);
    T wfric = (wK13H_h * tau.t13(0, 0, -1) - wK13H_l * tau.t13(-1, 0, -1)) * odx +
              (wK23H_h * tau.t23(0, 0, -1) - wK23H_l * tau.t23(0, -1, -1)) * ody +
              (wK33V_h * tau.t33(0) - wK33V_l * tau.t33(-1)) * odzw<T>(g, c, k);
    UF[p] = ufric;
    VF[p] = vfric;
    WF[p] = wfric;
    // the scalars: shared coefficients of the faces, then a flux difference each
    const T Pr = T(kPrInv);
    const T KHn = T(0.5) * (Pr * KHM(0, 1, 0) + Pr * KHM(0, 0, 0));
    const T KHs = T(0.5) * (Pr * KHM(0, 0, 0) + Pr * KHM(0, -1, 0));
    const T KHe = T(0.5) * (Pr * KHM(1, 0, 0) + Pr * KHM(0, 0, 0));
    const T KHw = T(0.5) * (Pr * KHM(0, 0, 0) + Pr * KHM(-1, 0, 0));
    const T KVh = -Pr * KM(0, 0, 1), KVl = -Pr * KM(0, 0, 0);
    const T dzh = odzw<T>(g, c, k + 1), dzl = odzw<T>(g, c, k), dz = odz<T>(g, c, k);
    auto diffuse = [&](const T *S) -> T {
        const T s0 = A(S, 0, 0, 0);
        // the diffusive fluxes through the top and the bottom, turbulence.cpp:1128-1131, 1226
        T tau_h = KVh * (A(S, 0, 0, 1) - s0) * dzh;
        T tau_l = k == 1 ? T(0) : KVl * (s0 - A(S, 0, 0, -1)) * dzl;
        T t22h = -KHn * (A(S, 0, 1, 0) - s0) * ody;
        T t22l = -KHs * (s0 - A(S, 0, -1, 0)) * ody;
        T t11h = -KHe * (A(S, 1, 0, 0) - s0) * odx;
        T t11l = -KHw * (s0 - A(S, -1, 0, 0)) * odx;
        return -((t11h - t11l) * odx + (t22h - t22l) * ody + (tau_h - tau_l) * dz);
    };
    TD[p] = diffuse(f.thm);
    if (f.moist) {
        QVD[p] = diffuse(f.qvm);
        QCD[p] = diffuse(f.qcm);
        QRD[p] = diffuse(f.qrm);
    }
}

// apply_velocity_diffusion, turbulence.cpp:233-258 (w from level 2)
template <typename T>
__global__ void k_turb_apply_uvw(Geo g, const T *__restrict__ UF, const T *__restrict__ VF, const T *__restrict__ WF, T *__restrict__ UP,
                                 T *__restrict__ VP, T *__restrict__ WP, T deltaT, int il, int jl, int jh) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x + 1;
    const int j = blockIdx.y + jl, i = blockIdx.z + il;
    if (k >= g.NZ - 1 || j >= jh) return;
    const long long p = IX3(i, j, k);
    UP[p] += UF[p] * deltaT;
    VP[p] += VF[p] * deltaT;
    if (k >= 2) WP[p] += WF[p] * deltaT;
}

// apply_scalar_diffusion (THP += t * step * dt) and apply_moisture_diffusion (QP += q * (step*dt)),
// turbulence.cpp:263-292
template <typename T>
__global__ void k_turb_apply_scalars(Geo g, const T *__restrict__ D0, const T *__restrict__ D1, const T *__restrict__ D2,
                                     T *__restrict__ P0, T *__restrict__ P1, T *__restrict__ P2, int nf, int theta, T step, T dt,
                                     int il, int jl, int jh) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x + 1;
    const int j = blockIdx.y + jl, i = blockIdx.z + il;
    if (k >= g.NZ - 1 || j >= jh) return;
    const long long p = IX3(i, j, k);
    if (theta) {
        P0[p] += D0[p] * step * dt;
        return;
    }
    const T deltaT = step * dt;
    P0[p] += D0[p] * deltaT;
    if (nf > 1) P1[p] += D1[p] * deltaT;
    if (nf > 2) P2[p] += D2[p] * deltaT;
}

#undef IX3

template <typename T>
TurbIn<T> turb_inputs(Ctx *c) {
    TurbIn<T> f{};
    auto M = [&](int fld) { return (const T *)c->prog[fld][DYN_ROLE_M]; };
    f.um = M(DYN_U);
    f.vm = M(DYN_V);
    f.wm = M(DYN_W);
    f.thm = M(DYN_TH);
    f.moist = c->g.microphysics != 0;
    if (f.moist) {
        f.qvm = M(DYN_QV);
        f.qcm = M(DYN_QC);
        f.qrm = M(DYN_QR);
    }
    f.ub = (const T *)c->bar[0];
    f.vb = (const T *)c->bar[1];
    f.wb = (const T *)c->bar[2];
    f.thb = (const T *)c->bar[3];
    f.qb = (const T *)c->bar[4];
    f.pb = (const T *)c->bar[5];
    f.pi = (const T *)c->pi;
    f.sat = c->turb.sat;
    return f;
}

TurbArgs turb_args(const Ctx *c) {
    return TurbArgs{c->turb.vml2, c->turb.vkmax, c->turb.landsea, c->turb.kmixh_max, c->turb.lH};
}

dim3 grid3(const Ctx *c, int il, int ih, int jl, int jh, int kblock) {
    return dim3((c->g.nz + kblock - 1) / kblock, (unsigned)(jh - jl), (unsigned)(ih - il));
}

template <typename T>
int launch_diff_tend(Ctx *c, int il, int ih, int jl, int jh) {
    TurbIn<T> f = turb_inputs<T>(c);
    TurbArgs ta = turb_args(c);
    T **b = (T **)c->turb.buf;
    const int ni = ih - il, nj = jh - jl, NZ = c->g.nz;
    {
        const int rows = std::max(1, kTurbThreads / NZ), nbj = (nj + rows - 1) / rows;
        const int nbk = NZ <= kTurbThreads ? 1 : (NZ - 2) / (kTurbThreads - 1) + 1;
        hipLaunchKernelGGL(k_turb_kmix<T>, dim3((unsigned)ni * nbj * nbk), dim3(kTurbThreads), 0, c->stream, c->geo, c->cols, f, ta, b[TK],
                           b[TKH], il, jl, jh, rows, nbj, nbk);
        DYN_LAUNCH_CHECK();
    }
    const int nbq = (nj * (NZ - 2) + kTurbThreads - 1) / kTurbThreads;
    hipLaunchKernelGGL(k_turb_tendencies<T>, dim3((unsigned)ni * nbq), dim3(kTurbThreads), 0, c->stream, c->geo, c->cols, f, ta,
                       (const T *)b[TK], (const T *)b[TKH], b[TUF], b[TVF], b[TWF], b[TTD], b[TQV], b[TQC], b[TQR], il, jl, jh, nbq);
    DYN_LAUNCH_CHECK();
    return DYN_OK;
}

template <typename T>
int launch_apply_velocity(Ctx *c, double step, int il, int ih, int jl, int jh) {
    T **b = (T **)c->turb.buf;
    auto P = [&](int fld) { return (T *)c->prog[fld][DYN_ROLE_P]; };
    const double deltaT = step * c->g.dt;
    hipLaunchKernelGGL(k_turb_apply_uvw<T>, grid3(c, il, ih, jl, jh, 64), dim3(64), 0, c->stream, c->geo, (const T *)b[TUF],
                       (const T *)b[TVF], (const T *)b[TWF], P(DYN_U), P(DYN_V), P(DYN_W), T(deltaT), il, jl, jh);
    DYN_LAUNCH_CHECK();
    return DYN_OK;
}

template <typename T>
int launch_apply_scalars(Ctx *c, double step, int il, int ih, int jl, int jh, bool theta) {
    T **b = (T **)c->turb.buf;
    auto P = [&](int fld) { return (T *)c->prog[fld][DYN_ROLE_P]; };
    if (theta)
        hipLaunchKernelGGL(k_turb_apply_scalars<T>, grid3(c, il, ih, jl, jh, 64), dim3(64), 0, c->stream, c->geo, (const T *)b[TTD],
                           (const T *)nullptr, (const T *)nullptr, P(DYN_TH), (T *)nullptr, (T *)nullptr, 1, 1, T(step), T(c->g.dt), il,
                           jl, jh);
    else
        hipLaunchKernelGGL(k_turb_apply_scalars<T>, grid3(c, il, ih, jl, jh, 64), dim3(64), 0, c->stream, c->geo, (const T *)b[TQV],
                           (const T *)b[TQC], (const T *)b[TQR], P(DYN_QV), P(DYN_QC), P(DYN_QR), 3, 0, T(step), T(c->g.dt), il, jl,
                           jh);
    DYN_LAUNCH_CHECK();
    return DYN_OK;
}

int check_turb(Ctx *c, const char *who, int il, int ih, int jl, int jh, int lo_i, int hi_i, int lo_j, int hi_j) {
    if (!c) {
        set_error(std::string(who) + ": null context");
        return DYN_E_ARG;
    }
    if (!c->turb.on) {
        set_error(std::string(who) + ": turbulence is off (dyn_set_turbulence)");
        return DYN_E_STATE;
    }
    if (il < lo_i || ih > hi_i || jl < lo_j || jh > hi_j || il >= ih || jl >= jh) {
        set_error(std::string(who) + ": bounds outside the range the reference uses");
        return DYN_E_ARG;
    }
    return DYN_OK;
}

}  // namespace

void turb_release(Ctx *c) {
    for (void *&p : c->turb.buf)
        if (p) {
            (void)hipFree(p);
            p = nullptr;
        }
    void *ptrs[] = {c->turb.sat, c->turb.landsea, c->turb.vml2, c->turb.vkmax};
    for (void *p : ptrs)
        if (p) (void)hipFree(p);
    c->turb = Turbulence{};
}

int turb_step_begin(Ctx *c) {
    const int NX = c->g.nx, NY = c->g.ny;
    return c->prec == DYN_FP32 ? launch_diff_tend<float>(c, 1, NX - 1, 1, NY - 1) : launch_diff_tend<double>(c, 1, NX - 1, 1, NY - 1);
}
const void *turb_tendency(const Ctx *c, int field) { return c->turb.buf[TUF + field]; }
int turb_apply_velocity(Ctx *c, double step) {
    const int NX = c->g.nx, NY = c->g.ny;
    return c->prec == DYN_FP32 ? launch_apply_velocity<float>(c, step, 3, NX - 3, 3, NY - 3)
                               : launch_apply_velocity<double>(c, step, 3, NX - 3, 3, NY - 3);
}
int turb_apply_scalars(Ctx *c, double step, bool theta) {
    const int NX = c->g.nx, NY = c->g.ny;
    return c->prec == DYN_FP32 ? launch_apply_scalars<float>(c, step, 1, NX - 1, 1, NY - 1, theta)
                               : launch_apply_scalars<double>(c, step, 1, NX - 1, 1, NY - 1, theta);
}

}  // namespace dyn

using namespace dyn;

extern "C" {

int dyn_set_turbulence(dyn_ctx *ctx, int on, const double *landsea, size_t count) {
    Ctx *c = reinterpret_cast<Ctx *>(ctx);
    if (!c) {
        set_error("dyn_set_turbulence: null context");
        return DYN_E_ARG;
    }
    const size_t n2 = (size_t)c->g.nx * c->g.ny;
    if (landsea && count != n2) {
        set_error("dyn_set_turbulence: the land-sea mask needs NX*NY values");
        return DYN_E_ARG;
    }
    if (int rc = dyn_synchronize(ctx)) return rc;
    drop_graph(c);  // the step's kernel sequence changes
    if (!on) {
        turb_release(c);
        return DYN_OK;
    }
    if (fused_supported(c))
        if (int rc = fused_lds_limits(c, true)) return rc;
    Turbulence &t = c->turb;
    if (!t.buf[0]) {
        for (void *&p : t.buf) {
            if (hipMalloc(&p, c->npts * c->elt) != hipSuccess || hipMemset(p, 0, c->npts * c->elt) != hipSuccess) {
                turb_release(c);
                set_error("dyn_set_turbulence: out of device memory");
                return DYN_E_HIP;
            }
        }
        if (hipMalloc(&t.sat, c->npts) != hipSuccess || hipMemset(t.sat, 0, c->npts) != hipSuccess ||
            hipMalloc(&t.landsea, n2 * 8) != hipSuccess || hipMalloc(&t.vml2, (size_t)c->g.nz * 8) != hipSuccess ||
            hipMalloc(&t.vkmax, (size_t)c->g.nz * 8) != hipSuccess) {
            turb_release(c);
            set_error("dyn_set_turbulence: out of device memory");
            return DYN_E_HIP;
        }
    }
    // init_kmix, turbulence.cpp:85-147, with zlevs = ZU = zsu (driver_serial.cpp:52)
    const int NZ = c->g.nz;
    const double *zsu = c->colhost + (size_t)DYN_COL_ZSU * NZ;
    std::vector<double> vml2(NZ, 0.0), vkmax(NZ, 0.0), ls(n2, 1.0);
    for (int k = 1; k < NZ; k++) {
        double deltaZ = zsu[k] - zsu[k - 1];
        vml2[k] = deltaZ > kLvMax ? kLvMax * kLvMax : deltaZ * deltaZ;
        vkmax[k] = kCmixV * vml2[k] / c->g.dt;
    }
    if (landsea)
        for (size_t n = 0; n < n2; n++) ls[n] = landsea[n];
    t.kmixh_max = kCmixH * c->g.dx * c->g.dx / c->g.dt;
    t.lH = c->g.dx / 4.0;
    DYN_HIP(hipMemcpy(t.vml2, vml2.data(), NZ * 8, hipMemcpyHostToDevice));
    DYN_HIP(hipMemcpy(t.vkmax, vkmax.data(), NZ * 8, hipMemcpyHostToDevice));
    DYN_HIP(hipMemcpy(t.landsea, ls.data(), n2 * 8, hipMemcpyHostToDevice));
    t.on = true;
    return DYN_OK;
}

int dyn_calculate_diff_tend(dyn_ctx *ctx, int il, int ih, int jl, int jh) {
    Ctx *c = reinterpret_cast<Ctx *>(ctx);
    if (int rc = check_turb(c, "calculate_diff_tend", il, ih, jl, jh, 1, c ? c->g.nx - 1 : 0, 1, c ? c->g.ny - 1 : 0)) return rc;
    return c->prec == DYN_FP32 ? launch_diff_tend<float>(c, il, ih, jl, jh) : launch_diff_tend<double>(c, il, ih, jl, jh);
}

int dyn_apply_velocity_diffusion(dyn_ctx *ctx, double step, int il, int ih, int jl, int jh) {
    Ctx *c = reinterpret_cast<Ctx *>(ctx);
    if (int rc = check_turb(c, "apply_velocity_diffusion", il, ih, jl, jh, 1, c ? c->g.nx - 1 : 0, 1, c ? c->g.ny - 1 : 0)) return rc;
    return c->prec == DYN_FP32 ? launch_apply_velocity<float>(c, step, il, ih, jl, jh) : launch_apply_velocity<double>(c, step, il, ih, jl, jh);
}

int dyn_apply_scalar_diffusion(dyn_ctx *ctx, double step, int il, int ih, int jl, int jh) {
    Ctx *c = reinterpret_cast<Ctx *>(ctx);
    if (int rc = check_turb(c, "apply_scalar_diffusion", il, ih, jl, jh, 1, c ? c->g.nx - 1 : 0, 1, c ? c->g.ny - 1 : 0)) return rc;
    return c->prec == DYN_FP32 ? launch_apply_scalars<float>(c, step, il, ih, jl, jh, true)
                               : launch_apply_scalars<double>(c, step, il, ih, jl, jh, true);
}

int dyn_apply_moisture_diffusion(dyn_ctx *ctx, double step, int il, int ih, int jl, int jh) {
    Ctx *c = reinterpret_cast<Ctx *>(ctx);
    if (int rc = check_turb(c, "apply_moisture_diffusion", il, ih, jl, jh, 1, c ? c->g.nx - 1 : 0, 1, c ? c->g.ny - 1 : 0)) return rc;
    if (!c->g.microphysics) {
        set_error("apply_moisture_diffusion: context has no moisture fields");
        return DYN_E_STATE;
    }
    return c->prec == DYN_FP32 ? launch_apply_scalars<float>(c, step, il, ih, jl, jh, false)
                               : launch_apply_scalars<double>(c, step, il, ih, jl, jh, false);
}

int dyn_get_turbulence(dyn_ctx *ctx, int which, double *values, size_t count) {
    Ctx *c = reinterpret_cast<Ctx *>(ctx);
    if (!c || !c->turb.on || which < 0 || which > TCOUNT || !values || count != c->npts) {
        set_error("dyn_get_turbulence: turbulence off, bad array id or count other than NX*NY*NZ");
        return DYN_E_ARG;
    }
    DYN_HIP(hipStreamSynchronize(c->stream));
    if (which == TCOUNT) {  // the saturation flags
        std::vector<unsigned char> tmp(c->npts);
        DYN_HIP(hipMemcpy(tmp.data(), c->turb.sat, c->npts, hipMemcpyDeviceToHost));
        for (size_t n = 0; n < c->npts; n++) values[n] = tmp[n];
        return DYN_OK;
    }
    if (c->prec == DYN_FP64) {
        DYN_HIP(hipMemcpy(values, c->turb.buf[which], c->npts * 8, hipMemcpyDeviceToHost));
        return DYN_OK;
    }
    std::vector<float> tmp(c->npts);
    DYN_HIP(hipMemcpy(tmp.data(), c->turb.buf[which], c->npts * 4, hipMemcpyDeviceToHost));
    for (size_t n = 0; n < c->npts; n++) values[n] = tmp[n];
    return DYN_OK;
}

}  // extern "C"
