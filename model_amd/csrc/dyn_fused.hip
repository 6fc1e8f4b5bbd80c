// Fused stage advection for gfx950: advect_uvw_velocity + advect_theta + advect_microphysics_cell
// (+ the fall speed and the interior part of zero_moisture) in one pass over HBM.
//
// Mapping: a block of tj j-rows, one lane per level of a row (RowMap), marches along i over a chunk of ti
// columns, as the reference's slab loop does (advection.cpp:313-325):
//   * i-stencils come from per-thread register queues (own j,k; columns i-3..i+3) and the east-face
//     flux of column i is carried as the west face of column i+1 (fluxes.cpp:891,1322,1504);
//   * j- and k-stencils read LDS planes of tj+6 rows; U/UB are kept for planes i and i+1, V/VB/W/WB for
//     planes i-1 and i (staggered advecting velocities), the scalars for plane i;
//   * north and top faces are computed once per point and exchanged through LDS as the south and
//     bottom faces of the neighbours.
// Every face and tendency uses the same expression tree as the per-operator kernels, so the fused and
// unfused paths agree to the last bit.
#include <algorithm>

#include "dyn_internal.hpp"

namespace dyn {
namespace {

constexpr int KP = 64;  // lanes per row (levels)

template <typename T>
__device__ __forceinline__ T sgn(T x) { return x > T(0) ? T(1) : T(-1); }

// interpolants of fluxes.cpp:110-206 (face_i5, face_i3)
template <typename T>
__device__ __forceinline__ T i5(T pm2, T pm1, T p0, T p1, T p2, T p3, T sign) { return face_i5(pm2, pm1, p0, p1, p2, p3, sign); }
template <typename T>
__device__ __forceinline__ T i3(T pm1, T p0, T p1, T p2, T sign) { return face_i3(pm1, p0, p1, p2, sign); }
template <typename T>
__device__ __forceinline__ T i2(T p0, T p1) { return T(0.5) * (p1 + p0); }

// Neighbouring levels of a column sit in neighbouring lanes.  Level k+1 and level k-1 come by the
// wavefront shifts of DPP (wave_shl:1 and wave_shr:1, a modifier of a VALU move: no LDS round trip); a
// lane whose source lies outside the wavefront keeps its own value.  That is the clamp the callers want at
// level 0 and at the last lane, and where packed rows cross a wavefront's edge the callers overwrite it
// from LDS.  Lanes past NZ-1 hold the values loaded at level NZ-1 (clamped loads) or values no
// active lane reads.  A fixed level comes by readlane (lane index uniform).
__device__ __forceinline__ int dpp_next(int x) { return __builtin_amdgcn_update_dpp(x, x, 0x130, 0xf, 0xf, false); }
__device__ __forceinline__ int dpp_prev(int x) { return __builtin_amdgcn_update_dpp(x, x, 0x138, 0xf, 0xf, false); }
__device__ __forceinline__ float lane_next(float x) { return __int_as_float(dpp_next(__float_as_int(x))); }
__device__ __forceinline__ float lane_prev(float x) { return __int_as_float(dpp_prev(__float_as_int(x))); }
__device__ __forceinline__ float lane_read(float x, int lane) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane)); }
__device__ __forceinline__ double lane_next(double x) {
    const long long b = __double_as_longlong(x);
    const unsigned lo = (unsigned)dpp_next((int)b), hi = (unsigned)dpp_next((int)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ double lane_prev(double x) {
    const long long b = __double_as_longlong(x);
    const unsigned lo = (unsigned)dpp_prev((int)b), hi = (unsigned)dpp_prev((int)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ double lane_read(double x, int lane) {
    const long long b = __double_as_longlong(x);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)b, lane), hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Element offsets are 32-bit (the host checks that a field is below 4 GiB): the base pointer stays in
// SGPRs and one VGPR byte offset serves every field at the same point.
template <typename T>
__device__ __forceinline__ T ld(const void *base, unsigned idx) {
    return *(const T *)((const char *)base + (size_t)(idx * (unsigned)sizeof(T)));
}
template <typename T>
__device__ __forceinline__ void st(void *base, unsigned idx, T v) {
    *(T *)((char *)base + (size_t)(idx * (unsigned)sizeof(T))) = v;
}

// Tile t = jblock + nbj * ichunk, placed by xcd_tile: neighbouring j-blocks of one i-chunk (which share
// halo rows) sit behind the same L2.

struct StageArgs {
    const void *cur[7];   // U V W TH QV QC QR (current)
    const void *mprev[7]; // M buffers
    void *out[7];         // P buffers
    const void *bar[5];   // UB VB WB THB QB
    void *vt;
    int il, ih, jl, jh;   // advected box
    int ti;               // columns one block marches
    int nbj;              // j-blocks
    int tj;               // rows per block
    // TURB: the step's turbulence tendencies of U V W TH QV QC QR, added to the new values
    const void *tend[7];
    double tdt;           // step * dt, in 64 bits
};

// Rows of a block.  Two mappings of levels and rows onto lanes, chosen on the host by the level count:
//   * one wavefront per row (PACK false, 57 <= NZ <= 64): lane = level, TJ rows per block;
//   * packed rows (PACK true, every other NZ up to 128): the block's rows lie one after another over its
//     lanes, lane q holding level q % NZ of row q / NZ.  A 40-level column fills 40 lanes instead of 64 and
//     an 80-level one 80 instead of 128; what bounds these kernels is the instructions each wavefront
//     issues, so an idle lane costs as much as a busy one.  A wavefront's edge may fall anywhere in a
//     column: the values that cross it go through a few LDS words (xch, xw, xb).
// Measured against a wavefront (two above 64 levels) per row, each at its best launch shape, FP32 moist: the
// momentum and scalar kernels 34 and 47 -> 26 and 37 us at 192x192x40, 57 and 74 -> 33 and 48 us at
// 160x120x90; FP64 78 and 159 -> 53 and 107 us at 192x192x40.
template <int TJ, bool PACK>
struct RowMap {
    int tj;     // rows per block
    int pitch;  // lanes (and LDS words of one field) per row
    int r, k;   // this lane's row and level; packed lanes past the last row repeat its last level
    int wave, lane;
    __device__ __forceinline__ RowMap(int tj_, int NZ) {
        tj = PACK ? tj_ : TJ;
        pitch = PACK ? NZ : KP;
        if (PACK) {
            const int q = min((int)threadIdx.x, tj * NZ - 1);
            r = q / NZ;
            k = q - r * NZ;
            wave = threadIdx.x / KP;
            lane = threadIdx.x % KP;
        } else {
            r = threadIdx.y;
            k = threadIdx.x;
            wave = r;
            lane = k;
        }
    }
};
// halo rows (and W rows) a lane loads: a block of tj rows has six halo rows and tj + 1 W rows
template <int TJ>
constexpr int halo_loads() { return TJ >= 6 ? 1 : TJ >= 3 ? 2 : 3; }

// Two or four neighbouring LDS words in one access (the addresses are multiples of the access's size)
template <typename T>
struct LdsVec;
template <>
struct LdsVec<float> {
    typedef float v2 __attribute__((ext_vector_type(2)));
};
template <>
struct LdsVec<double> {
    typedef double v2 __attribute__((ext_vector_type(2)));
};
template <typename T>
__device__ __forceinline__ void lds_ld2(const T *p, T &x, T &y) {
    const typename LdsVec<T>::v2 v = *(const typename LdsVec<T>::v2 *)p;
    x = v.x;
    y = v.y;
}
template <typename T>
__device__ __forceinline__ void lds_st2(T *p, T x, T y) {
    typename LdsVec<T>::v2 v;
    v.x = x;
    v.y = y;
    *(typename LdsVec<T>::v2 *)p = v;
}

// ---- momentum: advect_uvw_velocity (u, v fluxes and Coriolis; w = buoyancy, advection.cpp:304-339) -------
// LDS: (U, UB) of planes i, i+1 and (V, VB) of planes i-1, i on rows j0-3 .. j0+tj+2, (W, WB) of planes i-1, i
// on rows j0-1 .. j0+tj-1, each in a ring of three slots (plane p in slot p % 3); north faces of rows
// j0-1 .. j0+tj-1.  The fields of a pair lie side by side, so one LDS access moves both.
// Register queues hold U UB V VB of the own row at columns i-2 .. i+3.
template <typename T>
struct MomLds {
    __host__ __device__ static constexpr size_t uv(int tj, int pitch) { return 3 * 4 * (size_t)(tj + 6) * pitch; }  // [slot][u, v][row][k][2]
    __host__ __device__ static constexpr size_t w(int tj, int pitch) { return 3 * 2 * (size_t)(tj + 1) * pitch; }   // [slot][row][k][2]
    __host__ __device__ static constexpr size_t nf(int tj, int pitch) { return 2 * (size_t)(tj + 1) * pitch; }      // [row + 1][k][u v]
    static constexpr size_t x = 3 * 16;  // packed rows: top faces and buoyancy from each wavefront to the next
    static constexpr size_t bytes(int tj, int pitch) { return (uv(tj, pitch) + w(tj, pitch) + nf(tj, pitch) + x) * sizeof(T); }
};

// one tile (tj rows x ti columns x all levels) of the momentum stage; every thread of the block calls it
// TURB: apply_velocity_diffusion (turbulence.cpp:233-258) in the same pass; its box is the advected one.  The
// tendencies of a column are loaded ahead of the next column's prefetch, so the wait for them is not one for it.
template <typename T, int TJ, bool MOIST, bool PACK, bool TURB = false>
__device__ __forceinline__ void adv_momentum_tile(const Geo &g, const Cols &c, const StageArgs &a, T step, int t, unsigned char *smem_raw) {
    const RowMap<TJ, PACK> map(a.tj, g.NZ);
    const int tj = map.tj, KPW = map.pitch, k = map.k, r = map.r;
    const int R = tj + 6, RW = tj + 1;
    constexpr int HH = halo_loads<TJ>(), HW = 2;  // halo / W plane rows per lane
    T *uvp = (T *)smem_raw;
    T *wpl = uvp + MomLds<T>::uv(tj, KPW);
    T *nface = wpl + MomLds<T>::w(tj, KPW);
    T *xch = nface + MomLds<T>::nf(tj, KPW);

    const int j0 = a.jl + (t % a.nbj) * tj;
    const int i0 = a.il + (t / a.nbj) * a.ti;
    const int i1 = min(i0 + a.ti, a.ih);
    const int NZ = g.NZ, NY = g.NY;
    const unsigned NYNZ = (unsigned)g.NYNZ;
    const int j = j0 + r;
    const bool active = j < a.jh && k >= 1 && k <= NZ - 2;
    const int kc = min(k, NZ - 1), jc = min(j, NY - 1);
    const int km1 = max(kc - 1, 0), kp1 = min(kc + 1, NZ - 1), kp2 = min(kc + 2, NZ - 1);
    const unsigned rowoff = (unsigned)(jc * NZ + kc);
    const int RO = r + 3, WO = r + 1;  // own row in the U/V and W planes

    // the pair (U, UB) (p = 0) or (V, VB) (p = 1), and (W, WB), of a plane row at level kk
    auto UV = [&](int slot, int p, int row, int kk) -> T * { return uvp + (((slot * 2 + p) * R + row) * KPW + kk) * 2; };
    auto WW = [&](int slot, int row, int kk) -> T * { return wpl + ((slot * RW + row) * KPW + kk) * 2; };
    const void *qsrc[4] = {a.cur[0], a.bar[0], a.cur[1], a.bar[1]};
    T q[4][6], qs[4];  // U UB V VB of the own row at columns i-2 .. i+3 (i-3 .. i+2 in the prologue)

    // plane rows: U UB of plane iu, V VB W WB of plane iv.  The own row of U UB V VB comes from the
    // queues (which hold those columns already); only the six halo rows j0-3..j0-1, j0+tj..j0+tj+2 are
    // loaded
    auto halo_row = [&](int hh) { return hh < 3 ? hh : tj + hh; };
    T su[HH][4], sw[HW][2];
    auto fetch_planes = [&](int iu, int iv) {
#pragma unroll
        for (int h = 0; h < HH; h++) {
            const int hh = r + h * tj;
            if (hh < 6) {
                const int rr = halo_row(hh);
                const int jj = min(max(j0 - 3 + rr, 0), NY - 1);
                const unsigned pu = (unsigned)iu * NYNZ + (unsigned)(jj * NZ + kc), pv = (unsigned)iv * NYNZ + (unsigned)(jj * NZ + kc);
                su[h][0] = ld<T>(a.cur[0], pu);
                su[h][1] = ld<T>(a.bar[0], pu);
                su[h][2] = ld<T>(a.cur[1], pv);
                su[h][3] = ld<T>(a.bar[1], pv);
            }
        }
#pragma unroll
        for (int h = 0; h < HW; h++) {
            const int rr = r + h * tj;
            if (rr < RW) {
                const int jj = min(max(j0 - 1 + rr, 0), NY - 1);
                const unsigned pv = (unsigned)iv * NYNZ + (unsigned)(jj * NZ + kc);
                sw[h][0] = ld<T>(a.cur[2], pv);
                sw[h][1] = ld<T>(a.bar[2], pv);
            }
        }
    };
    // qu, qv: queue positions of columns iu and iv
    auto store_planes = [&](int iu, int iv, int qu, int qv) {
        const int su_slot = iu % 3, sv_slot = iv % 3;
        lds_st2(UV(su_slot, 0, RO, k), q[0][qu], q[1][qu]);
        lds_st2(UV(sv_slot, 1, RO, k), q[2][qv], q[3][qv]);
#pragma unroll
        for (int h = 0; h < HH; h++) {
            const int hh = r + h * tj;
            if (hh < 6) {
                const int rr = halo_row(hh);
                lds_st2(UV(su_slot, 0, rr, k), su[h][0], su[h][1]);
                lds_st2(UV(sv_slot, 1, rr, k), su[h][2], su[h][3]);
            }
        }
#pragma unroll
        for (int h = 0; h < HW; h++) {
            const int rr = r + h * tj;
            if (rr < RW) lds_st2(WW(sv_slot, rr, k), sw[h][0], sw[h][1]);
        }
    };
    // own-column inputs of column i: the buoyancy term's theta', qv, qc, qr and the M values of u, v, w
    T cb[7] = {}, sb[7] = {};
    auto fetch_col = [&](int i, T *b) {
        const unsigned p = (unsigned)i * NYNZ + rowoff;
        b[0] = ld<T>(a.cur[3], p);
        if (MOIST) {
            b[1] = ld<T>(a.cur[4], p);
            b[2] = ld<T>(a.cur[5], p);
            b[3] = ld<T>(a.cur[6], p);
        }
        b[4] = ld<T>(a.mprev[0], p);
        b[5] = ld<T>(a.mprev[1], p);
        b[6] = ld<T>(a.mprev[2], p);
    };

    // prologue: queues at columns i0-3 .. i0+2, planes U(i0, i0+1), V/W(i0-1, i0)
#pragma unroll
    for (int f = 0; f < 4; f++)
#pragma unroll
        for (int d = 0; d < 6; d++) q[f][d] = ld<T>(qsrc[f], (unsigned)(i0 - 3 + d) * NYNZ + rowoff);
    fetch_planes(i0, i0 - 1);
    store_planes(i0, i0 - 1, 3, 2);
    fetch_planes(i0 + 1, i0);
    store_planes(i0 + 1, i0, 4, 3);
    fetch_col(i0, cb);

    const T dtx = T(g.dtx), dty = T(g.dty), dt = T(g.dt);
    const T DTZ = T(g.dtz) * T(c.mu[kc]);
    const T rw1 = T(c.rhow[kp1]), rw0 = T(c.rhow[kc]), odr = T(c.one_d_rhou[kc]);
    const T fj = T(c.f[jc]);
    // read once: a load inside the march would be waited for together with the next column's prefetch
    const T tbvk = T(c.tbv[kc]);
    const T tdt = T(a.tdt);
    const bool low = (k == 1 || k == NZ - 2);

    // east faces of the queue's centre column (u_east, v_east; fluxes.cpp:1384-1592); slot: the U plane of the
    // column east of the centre, read at row j-1
    auto east_faces = [&](int slot, T *e) {
        T Ujm1, UBjm1;
        lds_ld2(UV(slot, 0, RO - 1, k), Ujm1, UBjm1);
        {
            T ua = T(0.5) * (q[0][3] + q[0][2]);
            T uba = T(0.5) * (q[1][3] + q[1][2]);
            T ue = i5(q[0][0], q[0][1], q[0][2], q[0][3], q[0][4], q[0][5], sgn(uba + ua));
            T ube = i5(q[1][0], q[1][1], q[1][2], q[1][3], q[1][4], q[1][5], sgn(ua));
            e[0] = ua * ube + (uba + ua) * ue;
        }
        {
            T ua = T(0.5) * (q[0][3] + Ujm1);
            T uba = T(0.5) * (q[1][3] + UBjm1);
            T ve = i5(q[2][0], q[2][1], q[2][2], q[2][3], q[2][4], q[2][5], sgn(uba + ua));
            T vbe = i5(q[3][0], q[3][1], q[3][2], q[3][3], q[3][4], q[3][5], sgn(ua));
            e[1] = ua * vbe + (uba + ua) * ve;
        }
    };
    __syncthreads();
    T west[2], east[2];
    east_faces(i0 % 3, west);  // column i0-1
#pragma unroll
    for (int f = 0; f < 4; f++) {
#pragma unroll
        for (int d = 0; d < 5; d++) q[f][d] = q[f][d + 1];
        q[f][5] = ld<T>(qsrc[f], (unsigned)(i0 + 3) * NYNZ + rowoff);
    }
    // Every prologue load has landed before the march starts: a load still outstanding at the loop's
    // entry makes the compiler wait, inside every iteration, for the next column's prefetch as well.
    __builtin_amdgcn_s_waitcnt(0);

    for (int i = i0; i < i1; i++) {
        const bool more = i + 1 < i1;
        const int c0 = i % 3, cm1 = (i + 2) % 3, cp1 = (i + 1) % 3;
        const unsigned p = (unsigned)i * NYNZ + rowoff;
        T du = T(0), dv = T(0), dw = T(0);
        if (TURB) {
            du = ld<T>(a.tend[0], p);
            dv = ld<T>(a.tend[1], p);
            dw = ld<T>(a.tend[2], p);
        }
        // loads for the next column go out first, its M values included
        if (more) {
#pragma unroll
            for (int f = 0; f < 4; f++) qs[f] = ld<T>(qsrc[f], (unsigned)(i + 4) * NYNZ + rowoff);
            fetch_planes(i + 2, i + 1);
            fetch_col(i + 1, sb);
        }
        const T um = cb[4], vm = cb[5], wm = cb[6];

        east_faces(cp1, east);
        // north faces (u_north, v_north) of row RR of the U/V planes
        auto north_faces = [&](int RR, T *nf) {
            T v[6], vb[6], vm1, vbm1;
#pragma unroll
            for (int d = 0; d < 6; d++) lds_ld2(UV(c0, 1, RR - 2 + d, k), v[d], vb[d]);
            lds_ld2(UV(cm1, 1, RR + 1, k), vm1, vbm1);
            {
                T va = T(0.5) * (v[3] + v[2]);
                T vba = T(0.5) * (vb[3] + vb[2]);
                T vn = i5(v[0], v[1], v[2], v[3], v[4], v[5], sgn(vba + va));
                T vbn = i5(vb[0], vb[1], vb[2], vb[3], vb[4], vb[5], sgn(va));
                nf[1] = va * vbn + (vba + va) * vn;
            }
            {
                T va = T(0.5) * (v[3] + vm1);
                T vba = T(0.5) * (vb[3] + vbm1);
#pragma unroll
                for (int d = 0; d < 6; d++) lds_ld2(UV(c0, 0, RR - 2 + d, k), v[d], vb[d]);
                T un = i5(v[0], v[1], v[2], v[3], v[4], v[5], sgn(vba + va));
                T ubn = i5(vb[0], vb[1], vb[2], vb[3], vb[4], vb[5], sgn(va));
                nf[0] = va * ubn + (vba + va) * un;
            }
        };
        T nf[2];
        north_faces(RO, nf);
        lds_st2(nface + ((r + 1) * KPW + k) * 2, nf[0], nf[1]);
        if (r == 0) {
            T sf[2];
            north_faces(RO - 1, sf);
            lds_st2(nface + k * 2, sf[0], sf[1]);
        }
        // top faces (u_top, v_top) of this level; level 0 has none
        T tf[2];
        T w1, wb1;  // w, wbar at k+1
        lds_ld2(WW(c0, WO, kp1), w1, wb1);
        auto top_face = [&](int pr, T wo, T wbo) -> T {
            T wa = T(0.5) * (w1 + wo);
            T wba = T(0.5) * (wb1 + wbo);
            T s0, s1, b0, b1, st_, bt;
            lds_ld2(UV(c0, pr, RO, kc), s0, b0);
            lds_ld2(UV(c0, pr, RO, kp1), s1, b1);
            if (low) {
                st_ = i2(s0, s1);
                bt = i2(b0, b1);
            } else {
                T sm, bm, s2, b2;
                lds_ld2(UV(c0, pr, RO, km1), sm, bm);
                lds_ld2(UV(c0, pr, RO, kp2), s2, b2);
                st_ = i3(sm, s0, s1, s2, sgn(wba + wa));
                bt = i3(bm, b0, b1, b2, sgn(wa));
            }
            return wa * bt + (wba + wa) * st_;
        };
        {
            T wo, wbo;
            lds_ld2(WW(cm1, WO, kp1), wo, wbo);
            tf[0] = top_face(0, wo, wbo);
            lds_ld2(WW(c0, WO - 1, kp1), wo, wbo);
            tf[1] = top_face(1, wo, wbo);
        }
        if (k == 0) tf[0] = tf[1] = T(0);
        // bottom face of level k = top face of level k-1; buoyancy of level k-1 (advection.cpp:42-58)
        T bu = lane_prev(tf[0]), bv = lane_prev(tf[1]);
        T bk = cb[0] / tbvk;
        if (MOIST) bk = cb[0] / tbvk + T(0.61) * cb[1] - cb[2] - cb[3];
        T bkm = lane_prev(bk);
        // packed rows: a wavefront's first lane takes the last lane's values of the wavefront before it
        if (PACK && map.lane == KP - 1) {
            xch[3 * map.wave] = tf[0];
            xch[3 * map.wave + 1] = tf[1];
            xch[3 * map.wave + 2] = bk;
        }
        __syncthreads();
        if (PACK && map.lane == 0 && map.wave > 0) {
            bu = xch[3 * map.wave - 3];
            bv = xch[3 * map.wave - 2];
            bkm = xch[3 * map.wave - 1];
        }
        T ou = T(0), ov = T(0), ow = T(0);  // this level's new values, stored after the barrier below
        if (active) {
            T su0, sv0;
            lds_ld2(nface + (r * KPW + k) * 2, su0, sv0);
            {  // u (advection.cpp:73-99)
                T other = T(0.25) * (UV(c0, 1, RO, k)[0] + UV(c0, 1, RO + 1, k)[0] + UV(cm1, 1, RO, k)[0] + UV(cm1, 1, RO + 1, k)[0]);
                T tend = -dtx * (east[0] - west[0]) - dty * (nf[0] - su0) - DTZ * (rw1 * tf[0] - rw0 * bu) * odr + dt * fj * other;
                ou = um + step * tend;
            }
            {  // v (advection.cpp:104-128)
                T other = T(0.25) * (UV(c0, 0, RO, k)[0] + UV(cp1, 0, RO, k)[0] + UV(c0, 0, RO - 1, k)[0] + UV(cp1, 0, RO - 1, k)[0]);
                T tend = -dtx * (east[1] - west[1]) - dty * (nf[1] - sv0) - DTZ * (rw1 * tf[1] - rw0 * bv) * odr - dt * fj * other;
                ov = vm + step * tend;
            }
            ow = wm + step * dt * T(kGrav) * T(0.5) * (bk + bkm);  // advection.cpp:329-337
            if (TURB) {
                ou += du * tdt;
                ov += dv * tdt;
                ow += dw * tdt;  // (stored from level 2)
            }
        }
        west[0] = east[0];
        west[1] = east[1];
        if (more) {
            store_planes(i + 2, i + 1, 4, 3);
#pragma unroll
            for (int f = 0; f < 4; f++) {
#pragma unroll
                for (int d = 0; d < 5; d++) q[f][d] = q[f][d + 1];
                q[f][5] = qs[f];
            }
#pragma unroll
            for (int f = 0; f < 7; f++) cb[f] = sb[f];
        }
        // Drained on every path, so the compiler does not carry this column's prefetch as possibly
        // outstanding into the next iteration (where it would wait on it, and on the stores below, at the
        // first reuse of those registers).  On the main path the plane update has already waited.
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        // stored after the next column's planes are written: a store issued earlier would hold up the
        // wait for the next column's prefetched values (the memory counter completes them in order)
        if (active) {
            st<T>(a.out[0], p, ou);
            st<T>(a.out[1], p, ov);
            if (k >= 2) st<T>(a.out[2], p, ow);
        }
    }
}

// ---- scalars: advect_theta (+ advect_microphysics_cell, the fall speed and the interior zero_moisture) ----
// LDS: the pairs (theta', thetabar) ((qv, qbar), (qc, qr)) of plane i on rows j0-3 .. j0+tj+2 in a ring of two
// slots, north faces of rows j0-1 .. j0+tj-1.  Register queues: the same fields of the own row at columns
// i-2 .. i+3.  Own-column inputs (u at i+1, v at j+1, w, the M values) are loaded per lane.
enum { kTheta = 1, kVapour = 2, kRain = 4, kMoist = 7 };  // the fields a tile takes (kRain: qc and qr)
template <typename T, int PARTS>
struct ScalLds {
    static constexpr int TH = PARTS & kTheta ? 1 : 0, QV = PARTS & kVapour ? 1 : 0, QC = PARTS & kRain ? 1 : 0;
    static constexpr int NP = TH + QV + QC;       // pairs
    static constexpr int NFS = TH + QV + 2 * QC;  // face kinds
    __host__ __device__ static constexpr size_t s(int tj, int pitch) { return 2 * 2 * NP * (size_t)(tj + 6) * pitch; }  // [slot][pair][row][k][2]
    __host__ __device__ static constexpr size_t nf(int tj, int pitch) { return NFS * (size_t)(tj + 1) * pitch; }        // [row + 1][k][face]
    // packed rows, per wavefront: w, wbar and the fall speed of its first lane for the wavefront before it; top
    // faces and the rain face of its last lane for the one after it
    static constexpr size_t xw = 3 * 16, xb = (NFS + 1) * 16;
    static constexpr size_t bytes(int tj, int pitch) { return (s(tj, pitch) + nf(tj, pitch) + xw + xb) * sizeof(T); }
};

// TURB: apply_scalar_diffusion and apply_moisture_diffusion (turbulence.cpp:263-292) of the advected points,
// before zero_moisture as in the reference; the boundary epilogue adds them on the rows beside the box
template <typename T, int TJ, int PARTS, bool PACK, bool TURB = false>
__device__ __forceinline__ void adv_scalars_tile(const Geo &g, const Cols &c, const StageArgs &a, T step, int t, unsigned char *smem_raw) {
    using L = ScalLds<T, PARTS>;
    constexpr int NP = L::NP, NS = 2 * NP, NFS = L::NFS;
    constexpr bool TH = L::TH, QV = L::QV, QC = L::QC;
    constexpr int PV = L::TH, PC = L::TH + L::QV;  // pair (and face) of qv, pair of qc and qr, face of qc
    const RowMap<TJ, PACK> map(a.tj, g.NZ);
    const int tj = map.tj, KPW = map.pitch, k = map.k, r = map.r;
    const int R = tj + 6;
    constexpr int HH = halo_loads<TJ>();  // halo plane rows per lane
    T *spl = (T *)smem_raw;
    T *nface = spl + L::s(tj, KPW);
    T *xw = nface + L::nf(tj, KPW), *xb = xw + L::xw;

    const int j0 = a.jl + (t % a.nbj) * tj;
    const int i0 = a.il + (t / a.nbj) * a.ti;
    const int i1 = min(i0 + a.ti, a.ih);
    const int NZ = g.NZ, NY = g.NY;
    const unsigned NYNZ = (unsigned)g.NYNZ;
    const int j = j0 + r;
    const bool active = j < a.jh && k >= 1 && k <= NZ - 2;
    const int kc = min(k, NZ - 1), jc = min(j, NY - 1), jn = min(j + 1, NY - 1);
    const int km1 = max(kc - 1, 0), kp1 = min(kc + 1, NZ - 1), kp2 = min(kc + 2, NZ - 1);
    const unsigned rowoff = (unsigned)(jc * NZ + kc), rowoffn = (unsigned)(jn * NZ + kc);
    const unsigned topoff = (unsigned)(jc * NZ + NZ - 1);
    const int RO = r + 3;

    // pair pr of a plane row at level kk
    auto SP = [&](int slot, int pr, int row, int kk) -> T * { return spl + (((slot * NP + pr) * R + row) * KPW + kk) * 2; };
    const void *src[NS];
    if constexpr (TH) {
        src[0] = a.cur[3];
        src[1] = a.bar[3];
    }
    if constexpr (QV) {
        src[2 * PV] = a.cur[4];
        src[2 * PV + 1] = a.bar[4];
    }
    if constexpr (QC) {
        src[2 * PC] = a.cur[5];
        src[2 * PC + 1] = a.cur[6];
    }
    T q[NS][6], qs[NS];  // the own row at columns i-2 .. i+3 (i-3 .. i+2 in the prologue)

    // plane rows: the own row comes from the queue, the six halo rows j0-3..j0-1, j0+tj..j0+tj+2 are loaded
    auto halo_row = [&](int hh) { return hh < 3 ? hh : tj + hh; };
    T ss[HH][NS];
    auto fetch_plane = [&](int i) {
#pragma unroll
        for (int h = 0; h < HH; h++) {
            const int hh = r + h * tj;
            if (hh < 6) {
                const int jj = min(max(j0 - 3 + halo_row(hh), 0), NY - 1);
                const unsigned pp = (unsigned)i * NYNZ + (unsigned)(jj * NZ + kc);
#pragma unroll
                for (int f = 0; f < NS; f++) ss[h][f] = ld<T>(src[f], pp);
            }
        }
    };
    // qd: queue position of column i
    auto store_plane = [&](int i, int qd) {
        const int slot = i % 2;
#pragma unroll
        for (int f = 0; f < NP; f++) lds_st2(SP(slot, f, RO, k), q[2 * f][qd], q[2 * f + 1][qd]);
#pragma unroll
        for (int h = 0; h < HH; h++) {
            const int hh = r + h * tj;
            if (hh < 6) {
                const int rr = halo_row(hh);
#pragma unroll
                for (int f = 0; f < NP; f++) lds_st2(SP(slot, f, rr, k), ss[h][2 * f], ss[h][2 * f + 1]);
            }
        }
    };
    // Register budget: in FP32 the M values of theta and q and qbar travel with the column's prefetch, and
    // a column's results are stored after the end-of-column barrier (so no store is counted ahead of the
    // next column's loads).  In FP64 both would push the kernel further into scratch spills, whose
    // reloads wait on the memory counter too: there the M values are loaded when the column starts and
    // the results stored before the plane update (1.90 against 1.99 ms per moist 256x256x64 step).
    constexpr bool kLean = sizeof(T) == 8;
    // own-column inputs of column i: u, ubar at i+1; v, vbar at j+1 and j; w, wbar; VT at the top level;
    // the M values of theta and q and qbar (FP32)
    struct Col {
        T u1, ub1, vn, vbn, vs, vbs, w0, wb0, vtt, mth, mqv, mqc, mqr, qbp;
    };
    auto fetch_col = [&](int i, Col &o) {
        const unsigned p = (unsigned)i * NYNZ + rowoff, pe = (unsigned)(i + 1) * NYNZ + rowoff, pn = (unsigned)i * NYNZ + rowoffn;
        o.u1 = ld<T>(a.cur[0], pe);
        o.ub1 = ld<T>(a.bar[0], pe);
        o.vn = ld<T>(a.cur[1], pn);
        o.vbn = ld<T>(a.bar[1], pn);
        if (r == 0) {
            o.vs = ld<T>(a.cur[1], p);
            o.vbs = ld<T>(a.bar[1], p);
        }
        o.w0 = ld<T>(a.cur[2], p);
        o.wb0 = ld<T>(a.bar[2], p);
        if (QC) o.vtt = ld<T>(a.vt, (unsigned)i * NYNZ + topoff);
        if (!kLean) {
            if (TH) o.mth = ld<T>(a.mprev[3], p);
            if (QV) {
                o.mqv = ld<T>(a.mprev[4], p);
                o.qbp = ld<T>(a.bar[4], p);
            }
            if (QC) {
                o.mqc = ld<T>(a.mprev[5], p);
                o.mqr = ld<T>(a.mprev[6], p);
            }
        }
    };

#pragma unroll
    for (int f = 0; f < NS; f++)
#pragma unroll
        for (int d = 0; d < 6; d++) q[f][d] = ld<T>(src[f], (unsigned)(i0 - 3 + d) * NYNZ + rowoff);

    const T dtx = T(g.dtx), dty = T(g.dty);
    const T DTZ = T(g.dtz) * T(c.mu[kc]);
    const T rw1 = T(c.rhow[kp1]), rw0 = T(c.rhow[kc]), odr = T(c.one_d_rhou[kc]);
    const bool low = (k == 1 || k == NZ - 2);
    // The remaining column constants of this lane's level are read here, once.  A load inside the march
    // is waited for together with every load issued before it (the memory counter completes in order),
    // so one there would also wait for the next column's prefetch.  Indices are clamped for the lanes
    // outside the active levels, which never use the values.
    const T tbu = T(c.tb[kp1]) - T(c.tb[kc]), tbd = T(c.tb[kc]) - T(c.tb[km1]);
    T qbu = T(0), qbd = T(0), qbk = T(0), rk = T(1), vtden = T(0);
    if (QV) {
        qbu = T(c.qb[kp1]) - T(c.qb[kc]);
        qbd = T(c.qb[kc]) - T(c.qb[km1]);
        qbk = T(c.qb[kc]);
    }
    if (QC) {
        rk = T(c.rhou[kc]);
        vtden = sqrt(T(c.rhou[1]) / rk);
    }
    // fall speed of this level (kessler.cpp:222-252) from its rain; NZ-1 keeps the array's
    auto fall = [&](T qr, T top) -> T {
        T v = T(0);
        if (k >= 1 && k <= NZ - 2) {
            if (qr > T(1.0e-12)) {
                T qrr = fmax(qr * T(0.001) * rk, T(0));
                v = T(36.34) * (pow(qrr, T(0.1364))) * vtden;
            }
        } else if (k == NZ - 1) {
            v = top;
        }
        return v;
    };

    // east faces (s_east; fluxes.cpp:797-1032) of the queue's centre column with u, ubar at the column east of it
    auto east_faces = [&](T U1, T UB1, T *e) {
        const T ub = UB1 + U1;
        if constexpr (TH) {
            T se = i5(q[0][0], q[0][1], q[0][2], q[0][3], q[0][4], q[0][5], sgn(ub));
            T be = i5(q[1][0], q[1][1], q[1][2], q[1][3], q[1][4], q[1][5], sgn(U1));
            e[0] = U1 * be + ub * se;
        }
        if constexpr (QV) {
            constexpr int f = 2 * PV;
            T sv = i5(q[f][0], q[f][1], q[f][2], q[f][3], q[f][4], q[f][5], sgn(ub));
            T bv = i5(q[f + 1][0], q[f + 1][1], q[f + 1][2], q[f + 1][3], q[f + 1][4], q[f + 1][5], sgn(U1));
            e[PV] = U1 * bv + ub * sv;
        }
        if constexpr (QC) {
            constexpr int f = 2 * PC;
            e[PC] = ub * i5(q[f][0], q[f][1], q[f][2], q[f][3], q[f][4], q[f][5], sgn(ub));
            e[PC + 1] = ub * i5(q[f + 1][0], q[f + 1][1], q[f + 1][2], q[f + 1][3], q[f + 1][4], q[f + 1][5], sgn(ub));
        }
    };
    T west[NFS], east[NFS];
    {  // west faces of column i0: the east faces of column i0-1 (compute_west_scalar, fluxes.cpp:479-501)
        const unsigned pe = (unsigned)i0 * NYNZ + rowoff;
        east_faces(ld<T>(a.cur[0], pe), ld<T>(a.bar[0], pe), west);
    }
#pragma unroll
    for (int f = 0; f < NS; f++) {
#pragma unroll
        for (int d = 0; d < 5; d++) q[f][d] = q[f][d + 1];
        q[f][5] = ld<T>(src[f], (unsigned)(i0 + 3) * NYNZ + rowoff);
    }
    Col cc{}, cs{};
    fetch_col(i0, cc);
    // Packed rows: a wavefront's last lane reads w, wbar and the fall speed of the level above it, which
    // sit in the next wavefront's first lane, from LDS.  The fall speed of a column is therefore formed
    // before the barrier that ends the column before it.
    T vtk = T(0);
    auto publish_w = [&]() {
        if constexpr (PACK) {
            if (QC) vtk = fall(q[NS - 1][2], cc.vtt);
            if (map.lane == 0) {
                xw[3 * map.wave] = cc.w0;
                xw[3 * map.wave + 1] = cc.wb0;
                if (QC) xw[3 * map.wave + 2] = vtk;
            }
        }
    };
    publish_w();
    fetch_plane(i0);
    store_plane(i0, 2);
    __syncthreads();
    // Every prologue load has landed before the march starts.  Without this wait the waves that skip the
    // halo loads enter the loop with the own-column loads still counted as outstanding, and the compiler
    // then waits inside every iteration (at the first use of those registers) for most of the next
    // column's prefetch as well.
    __builtin_amdgcn_s_waitcnt(0);

    for (int i = i0; i < i1; i++) {
        const bool more = i + 1 < i1;
        const int c0 = i % 2;
        const unsigned p = (unsigned)i * NYNZ + rowoff;
        T td[NFS] = {};
        if (TURB) {
#pragma unroll
            for (int f = 0; f < NFS; f++) td[f] = ld<T>(a.tend[(TH ? 3 : QV ? 4 : 5) + f], p);
        }
        if (more) {
#pragma unroll
            for (int f = 0; f < NS; f++) qs[f] = ld<T>(src[f], (unsigned)(i + 4) * NYNZ + rowoff);
            fetch_col(i + 1, cs);
            fetch_plane(i + 1);
        }
        T mth = cc.mth, mqv = cc.mqv, mqc = cc.mqc, mqr = cc.mqr, qbp = cc.qbp;
        if (kLean) {
            if (TH) mth = ld<T>(a.mprev[3], p);
            if (QV) {
                mqv = ld<T>(a.mprev[4], p);
                qbp = ld<T>(a.bar[4], p);
            }
            if (QC) {
                mqc = ld<T>(a.mprev[5], p);
                mqr = ld<T>(a.mprev[6], p);
            }
        }

        east_faces(cc.u1, cc.ub1, east);
        // north faces (s_north) of row RR with v, vbar at the face
        auto north_faces = [&](int RR, T V1, T VB1, T *nf) {
            T x[6], y[6];
            auto rows = [&](int pr) {
#pragma unroll
                for (int d = 0; d < 6; d++) lds_ld2(SP(c0, pr, RR - 2 + d, k), x[d], y[d]);
            };
            const T vb = VB1 + V1;
            if constexpr (TH) {
                rows(0);
                T sn = i5(x[0], x[1], x[2], x[3], x[4], x[5], sgn(vb));
                T bn = i5(y[0], y[1], y[2], y[3], y[4], y[5], sgn(V1));
                nf[0] = V1 * bn + vb * sn;
            }
            if constexpr (QV) {
                rows(PV);
                T sv = i5(x[0], x[1], x[2], x[3], x[4], x[5], sgn(vb));
                T bv = i5(y[0], y[1], y[2], y[3], y[4], y[5], sgn(V1));
                nf[PV] = V1 * bv + vb * sv;
            }
            if constexpr (QC) {
                rows(PC);
                nf[PC] = vb * i5(x[0], x[1], x[2], x[3], x[4], x[5], sgn(vb));
                nf[PC + 1] = vb * i5(y[0], y[1], y[2], y[3], y[4], y[5], sgn(vb));
            }
        };
        auto put_faces = [&](int row, const T *nf) {
            T *o = nface + (row * KPW + k) * NFS;
            if constexpr (NFS == 1) {
                o[0] = nf[0];
            } else {
                lds_st2(o, nf[0], nf[1]);
                if constexpr (NFS == 4) lds_st2(o + 2, nf[2], nf[3]);
            }
        };
        T nf[NFS];
        north_faces(RO, cc.vn, cc.vbn, nf);
        put_faces(r + 1, nf);
        if (r == 0) {
            T sf[NFS];
            north_faces(RO - 1, cc.vs, cc.vbs, sf);
            put_faces(0, sf);
        }
        // top faces (s_top) of this level from the own column of the plane; w, wbar (and the fall speed) at
        // k+1 by lane exchange
        T W1 = lane_next(cc.w0), WB1 = lane_next(cc.wb0);
        if (QC && !PACK) vtk = fall(q[NS - 1][2], cc.vtt);
        T vk1 = QC ? lane_next(vtk) : T(0);
        if (PACK && map.lane == KP - 1) {  // (past the block's last wavefront: words no lane uses)
            W1 = xw[3 * map.wave + 3];
            WB1 = xw[3 * map.wave + 4];
            if (QC) vk1 = xw[3 * map.wave + 5];
        }
        // the pair's fields at levels k-1 .. k+2 of the own column
        T x[4], y[4];
        auto column = [&](int pr) {
            lds_ld2(SP(c0, pr, RO, km1), x[0], y[0]);
            lds_ld2(SP(c0, pr, RO, kc), x[1], y[1]);
            lds_ld2(SP(c0, pr, RO, kp1), x[2], y[2]);
            lds_ld2(SP(c0, pr, RO, kp2), x[3], y[3]);
        };
        auto s_top = [&](int pr) -> T {
            column(pr);
            T st_, bt;
            if (low) {
                st_ = i2(x[1], x[2]);
                bt = i2(y[1], y[2]);
            } else {
                st_ = i3(x[0], x[1], x[2], x[3], sgn(WB1 + W1));
                bt = i3(y[0], y[1], y[2], y[3], sgn(W1));
            }
            return W1 * bt + (WB1 + W1) * st_;
        };
        T tf[NFS];
        if constexpr (TH) tf[0] = s_top(0);
        if constexpr (QV) tf[PV] = s_top(PV);
        T qrt = T(0);
        if constexpr (QC) {
            column(PC);
            {
                T wb = WB1 + W1;
                T tq = low ? i2(x[1], x[2]) : i3(x[0], x[1], x[2], x[3], sgn(wb));
                tf[PC] = wb * tq;
            }
            // rain top face with the fall speed (fluxes.cpp:734, 780; 966-1030); level 0 falls as level 1 does
            if (k == 0) {
                T t0 = T(0.5) * (y[1] + y[2]);
                qrt = -T(0.5) * (vk1 + vk1) * t0;
            } else {
                T wb = WB1 + W1;
                T tq;
                if (kc == 1 || kc == NZ - 2) tq = i2(y[1], y[2]);
                else tq = i3(y[0], y[1], y[2], y[3], sgn(WB1 + W1 - T(0.5) * (vtk + vk1)));
                qrt = (wb - T(0.5) * (vk1 + vtk)) * tq;
            }
        }
        if (k == 0) {
#pragma unroll
            for (int f = 0; f < NFS; f++) tf[f] = T(0);
        }
        T bot[NFS];
        constexpr int NB = NP;  // top faces handed up (rain has its own)
#pragma unroll
        for (int f = 0; f < NB; f++) bot[f] = lane_prev(tf[f]);
        T qrb = QC ? lane_prev(qrt) : T(0);
        if (PACK && map.lane == KP - 1) {
#pragma unroll
            for (int f = 0; f < NB; f++) xb[(NFS + 1) * map.wave + f] = tf[f];
            xb[(NFS + 1) * map.wave + NFS] = qrt;
        }
        __syncthreads();
        if (PACK && map.lane == 0 && map.wave > 0) {
#pragma unroll
            for (int f = 0; f < NB; f++) bot[f] = xb[(NFS + 1) * (map.wave - 1) + f];
            if (QC) qrb = xb[(NFS + 1) * (map.wave - 1) + NFS];
        }
        const T vtk0 = vtk;  // this column's fall speed, stored below
        T oth = T(0), oqv = T(0), oqc = T(0), oqr = T(0);  // this level's final values (active levels)
        if (active) {
            T south[4];
            const T *so = nface + (r * KPW + k) * NFS;
            if constexpr (NFS == 1) {
                south[0] = so[0];
            } else {
                lds_ld2(so, south[0], south[1]);
                if constexpr (NFS == 4) lds_ld2(so + 2, south[2], south[3]);
            }
            // Z_ADVECT_BASE (advection.cpp:16-18) with the base-state differences du = b[k+1] - b[k],
            // dd = b[k] - b[k-1] of this level
            auto zbase = [&](T du, T dd) -> T { return (T(0.50) * (rw1 * W1 * du + rw0 * cc.w0 * dd) * odr); };
            if constexpr (TH) {  // theta (advection.cpp:152-168)
                T tend = -dtx * (east[0] - west[0]) - dty * (nf[0] - south[0]) - DTZ * (rw1 * tf[0] - rw0 * bot[0]) * odr -
                         DTZ * zbase(tbu, tbd);
                oth = mth + step * tend;
                if (TURB) oth += td[0] * step * T(g.dt);
            }
            const T tdt = step * T(g.dt);
            if constexpr (QV) {  // advection.cpp:197-253, then zero_moisture for the advected points (microphysics.cpp:677-698)
                T tq = -dtx * (east[PV] - west[PV]) - dty * (nf[PV] - south[PV]) - DTZ * (rw1 * tf[PV] - rw0 * bot[PV]) * odr -
                       DTZ * zbase(qbu, qbd);
                oqv = mqv + step * tq;
                if (TURB) oqv += td[PV] * tdt;
                if (oqv + qbp + qbk < T(0)) oqv = -(qbp + qbk);
            }
            if constexpr (QC) {
                T tc = -dtx * (east[PC] - west[PC]) - dty * (nf[PC] - south[PC]) - DTZ * (rw1 * tf[PC] - rw0 * bot[PC]) * odr;
                oqc = mqc + step * tc;
                T tr = -dtx * (east[PC + 1] - west[PC + 1]) - dty * (nf[PC + 1] - south[PC + 1]) - DTZ * (rw1 * qrt - rw0 * qrb) * odr;
                oqr = mqr + step * tr;
                if (TURB) {
                    oqc += td[PC] * tdt;
                    oqr += td[PC + 1] * tdt;
                }
                if (oqc < T(0)) oqc = T(0);
                if (oqr < T(0)) oqr = T(0);
            }
        }
        // With its own level, the lane of level 1 (NZ-2) writes the lid of upper_lower_boundaries
        // (boundaries.cpp:304-312): level 0 (NZ-1) takes its value.  These are the final values of an
        // interior column (no sponge or periodic copy touches it); the boundary epilogue redoes the columns
        // it rewrites whole.  The sources of the periodic copy are left to it: halo column 0 receives
        // column NX-6's values from before the lid.
        const bool lid = active && (k == 1 || k == NZ - 2) && i >= 6 && i < g.NX - 6;
        auto store_column = [&]() {
            if (active) {
                if (TH) st<T>(a.out[3], p, oth);
                if (QV) st<T>(a.out[4], p, oqv);
                if (QC) {
                    st<T>(a.out[5], p, oqc);
                    st<T>(a.out[6], p, oqr);
                    st<T>(a.vt, p, vtk0);
                    if (k == 1) st<T>(a.vt, p - 1, vtk0);
                }
            }
            if (lid) {
                const unsigned pl = k == 1 ? p - 1 : p + 1;
                if (TH) st<T>(a.out[3], pl, oth);
                if (QV) st<T>(a.out[4], pl, oqv);
                if (QC) {
                    st<T>(a.out[5], pl, oqc);
                    st<T>(a.out[6], pl, oqr);
                }
            }
        };
        if (kLean) store_column();
#pragma unroll
        for (int f = 0; f < NFS; f++) west[f] = east[f];
        if (more) {
            store_plane(i + 1, 3);
#pragma unroll
            for (int f = 0; f < NS; f++) {
#pragma unroll
                for (int d = 0; d < 5; d++) q[f][d] = q[f][d + 1];
                q[f][5] = qs[f];
            }
            cc = cs;
            publish_w();
        }
        // drained on every path (see the momentum kernel)
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        // FP32: this column's stores go out after the next column's planes are written.  The memory
        // counter completes loads and stores in order, so a store issued before that point would hold up
        // the wait for the next column's prefetched values; here it completes during the next column.
        if (!kLean) store_column();
    }
}

// threads of the largest block: TJ rows of one wavefront each, or kPackThreads lanes of packed rows
constexpr int kPackThreads = 512;
template <int TJ, bool PACK>
constexpr int stage_threads() { return PACK ? kPackThreads : KP * TJ; }

template <typename T, int TJ, bool MOIST, bool PACK, bool TURB>
__global__ void __launch_bounds__((stage_threads<TJ, PACK>())) k_adv_momentum(Geo g, Cols c, StageArgs a, T step) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    adv_momentum_tile<T, TJ, MOIST, PACK, TURB>(g, c, a, step, xcd_tile(blockIdx.x, gridDim.x), smem_raw);
}

// Blocks per tile of the scalar kernel.  Moist FP64 tiles go in two: theta and qv, qc and qr.  All four fields
// at once take more than the 256 registers that two wavefronts per SIMD leave each, and their scratch reloads wait
// behind the prefetch; halves need 199 and half the LDS, and read the winds twice (neighbouring blocks, so mostly
// from L2).  One block, two, three (theta, qv, qc with qr) at 256x256x64: 292, 222, 246 us; 150x126x50: 74, 58, 70;
// 160x120x90: 169, 116, 135.  FP32 keeps one: it fits, with three wavefronts per SIMD.
template <typename T, bool MOIST>
constexpr int scalar_parts() { return MOIST && sizeof(T) == 8 ? 2 : 1; }
template <typename T, bool MOIST>
constexpr size_t scalar_lds(int tj, int pitch) {
    if (!MOIST) return ScalLds<T, kTheta>::bytes(tj, pitch);
    return scalar_parts<T, MOIST>() == 1 ? ScalLds<T, kMoist>::bytes(tj, pitch) : ScalLds<T, (kTheta | kVapour)>::bytes(tj, pitch);
}
// tile t of the scalar half, counted over the parts
template <typename T, int TJ, bool MOIST, bool PACK, bool TURB>
__device__ __forceinline__ void adv_scalars_any(const Geo &g, const Cols &c, const StageArgs &a, T step, int t, unsigned char *smem_raw) {
    if constexpr (!MOIST) {
        adv_scalars_tile<T, TJ, kTheta, PACK, TURB>(g, c, a, step, t, smem_raw);
    } else if constexpr (scalar_parts<T, MOIST>() == 1) {
        adv_scalars_tile<T, TJ, kMoist, PACK, TURB>(g, c, a, step, t, smem_raw);
    } else {
        if (t % 2) adv_scalars_tile<T, TJ, kTheta | kVapour, PACK, TURB>(g, c, a, step, t / 2, smem_raw);
        else adv_scalars_tile<T, TJ, kRain, PACK, TURB>(g, c, a, step, t / 2, smem_raw);
    }
}
template <typename T, int TJ, bool MOIST, bool PACK, bool TURB>
__global__ void __launch_bounds__((stage_threads<TJ, PACK>())) k_adv_scalars(Geo g, Cols c, StageArgs a, T step) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    adv_scalars_any<T, TJ, MOIST, PACK, TURB>(g, c, a, step, xcd_tile(blockIdx.x, gridDim.x), smem_raw);
}

// Both halves of a stage in one launch, for grids whose blocks are all on the device at once: the momentum tiles
// (nm of them), then the scalar tiles with their march length.  Small grids' steps are a chain of launches of 5 to
// 20 us; a second stream beside it costs a fork and a join of about 8 us each.
template <typename T, int TJ, bool MOIST, bool PACK, bool TURB>
__global__ void __launch_bounds__((stage_threads<TJ, PACK>())) k_adv_stage(Geo g, Cols c, StageArgs a, T step, int nm, int ti_scal) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int b = blockIdx.x;
    if (b < nm) {
        adv_momentum_tile<T, TJ, MOIST, PACK, TURB>(g, c, a, step, xcd_tile(b, nm), smem_raw);
    } else {
        a.ti = ti_scal;
        adv_scalars_any<T, TJ, MOIST, PACK, TURB>(g, c, a, step, xcd_tile(b - nm, gridDim.x - nm), smem_raw);
    }
}

// zero_moisture outside the advected box (the fused kernel clips the points it writes)
template <typename T>
__global__ void k_zero_moisture_shell(Geo g, Cols c, T *__restrict__ QVP, T *__restrict__ QCP, T *__restrict__ QRP,
                                      const T *__restrict__ QB, long long n, int bil, int bih, int bjl, int bjh, int il, int ih, int jl,
                                      int jh) {
    long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    int k = (int)(p % g.NZ);
    long long rr = p / g.NZ;
    int j = (int)(rr % g.NY), i = (int)(rr / g.NY);
    bool inbox = i >= bil && i < bih && j >= bjl && j < bjh && k >= 1 && k < g.NZ - 1;
    if (inbox) return;
    if (QCP[p] < T(0)) QCP[p] = T(0);
    if (QRP[p] < T(0)) QRP[p] = T(0);
    if (i >= il && i < ih && j >= jl && j < jh && k >= 1 && k < g.NZ - 1) {
        if (QVP[p] + QB[p] + T(c.qb[k]) < T(0)) QVP[p] = -(QB[p] + T(c.qb[k]));
    }
}

// Lanes of packed rows (see RowMap) unless a 64-lane wavefront is nearly full: at 57 levels and more a row
// per wavefront wastes at most one lane in nine and needs no exchange at wavefront edges
bool stage_packs(const Ctx *c) { return c->g.nz < 57 || c->g.nz > KP; }

// shape: rows per block, march length and lane mapping of one launch
template <typename T, int TJ, bool MOIST, bool PACK, bool TURB>
int momentum_t(Ctx *c, const StageArgs &a0, T step, const StageShape &sh) {
    StageArgs a = a0;
    a.ti = sh.ti;
    a.tj = sh.tj;
    a.nbj = (a.jh - a.jl + sh.tj - 1) / sh.tj;
    const int nbi = (a.ih - a.il + sh.ti - 1) / sh.ti;
    const dim3 blk = PACK ? dim3((sh.tj * c->geo.NZ + KP - 1) / KP * KP) : dim3(KP, TJ);
    Timed _t(c, "adv_momentum", (double)(a.ih - a.il) * (a.jh - a.jl) * (c->geo.NZ - 2));
    hipLaunchKernelGGL((k_adv_momentum<T, TJ, MOIST, PACK, TURB>), dim3(a.nbj * nbi), blk, MomLds<T>::bytes(sh.tj, PACK ? c->geo.NZ : KP),
                       c->stream, c->geo, c->cols, a, step);
    DYN_LAUNCH_CHECK();
    return DYN_OK;
}

template <typename T, int TJ, bool MOIST, bool PACK, bool TURB>
int scalars_t(Ctx *c, const StageArgs &a0, T step, const StageShape &sh) {
    StageArgs a = a0;
    a.ti = sh.ti;
    a.tj = sh.tj;
    a.nbj = (a.jh - a.jl + sh.tj - 1) / sh.tj;
    const int nbi = (a.ih - a.il + sh.ti - 1) / sh.ti;
    const dim3 blk = PACK ? dim3((sh.tj * c->geo.NZ + KP - 1) / KP * KP) : dim3(KP, TJ);
    Timed _t(c, "adv_scalars", (double)(a.ih - a.il) * (a.jh - a.jl) * (c->geo.NZ - 2));
    hipLaunchKernelGGL((k_adv_scalars<T, TJ, MOIST, PACK, TURB>), dim3(a.nbj * nbi * scalar_parts<T, MOIST>()), blk,
                       (scalar_lds<T, MOIST>(sh.tj, PACK ? c->geo.NZ : KP)), c->stream, c->geo, c->cols, a, step);
    DYN_LAUNCH_CHECK();
    return DYN_OK;
}

template <typename T, int TJ, bool MOIST, bool PACK, bool TURB>
int stage_one_t(Ctx *c, const StageArgs &a0, T step, const StageOne &sh) {
    StageArgs a = a0;
    a.ti = sh.ti_mom;
    a.tj = sh.tj;
    a.nbj = (a.jh - a.jl + sh.tj - 1) / sh.tj;
    const int nm = a.nbj * ((a.ih - a.il + sh.ti_mom - 1) / sh.ti_mom);
    const int ns = a.nbj * ((a.ih - a.il + sh.ti_scal - 1) / sh.ti_scal) * scalar_parts<T, MOIST>();
    const int pitch = PACK ? c->geo.NZ : KP;
    const dim3 blk = PACK ? dim3((sh.tj * c->geo.NZ + KP - 1) / KP * KP) : dim3(KP, TJ);
    Timed _t(c, "adv_stage", (double)(a.ih - a.il) * (a.jh - a.jl) * (c->geo.NZ - 2));
    hipLaunchKernelGGL((k_adv_stage<T, TJ, MOIST, PACK, TURB>), dim3(nm + ns), blk,
                       (std::max(MomLds<T>::bytes(sh.tj, pitch), scalar_lds<T, MOIST>(sh.tj, pitch))), c->stream, c->geo, c->cols, a, step,
                       nm, sh.ti_scal);
    DYN_LAUNCH_CHECK();
    return DYN_OK;
}

template <typename T, bool MOIST, bool TURB>
int stage_t(Ctx *c, double step, int il, int ih, int jl, int jh, int parts) {
    StageArgs a{};
    for (int f = 0; f < 7; f++) {
        a.cur[f] = c->prog[f][DYN_ROLE_CUR];
        a.mprev[f] = c->prog[f][DYN_ROLE_M];
        a.out[f] = c->prog[f][DYN_ROLE_P];
    }
    for (int f = 0; f < 5; f++) a.bar[f] = c->bar[f];
    a.vt = c->vt;
    if (TURB) {
        for (int f = 0; f < 7; f++) a.tend[f] = turb_tendency(c, f);
        a.tdt = step * c->g.dt;
    }
    a.il = il;
    a.ih = ih;
    a.jl = jl;
    a.jh = jh;
    if (parts == (kStageMomentum | kStageScalars) && stage_in_one(c)) {
        const StageOne &m = c->auto_one;
        if (stage_packs(c)) {
            if (m.tj >= 6) return stage_one_t<T, 8, MOIST, true, TURB>(c, a, T(step), m);
            if (m.tj >= 3) return stage_one_t<T, 4, MOIST, true, TURB>(c, a, T(step), m);
            return stage_one_t<T, 2, MOIST, true, TURB>(c, a, T(step), m);
        }
        if (m.tj == 2) return stage_one_t<T, 2, MOIST, false, TURB>(c, a, T(step), m);
        if (m.tj == 4) return stage_one_t<T, 4, MOIST, false, TURB>(c, a, T(step), m);
        return stage_one_t<T, 8, MOIST, false, TURB>(c, a, T(step), m);
    }
    int rc = DYN_OK;
    if (parts & kStageMomentum) {
        const StageShape m = stage_shape(c, true);
        if (m.pack) {
            if (m.tj >= 6) rc = momentum_t<T, 8, MOIST, true, TURB>(c, a, T(step), m);
            else if (m.tj >= 3) rc = momentum_t<T, 4, MOIST, true, TURB>(c, a, T(step), m);
            else rc = momentum_t<T, 2, MOIST, true, TURB>(c, a, T(step), m);
        } else if (m.tj == 2) rc = momentum_t<T, 2, MOIST, false, TURB>(c, a, T(step), m);
        else if (m.tj == 4) rc = momentum_t<T, 4, MOIST, false, TURB>(c, a, T(step), m);
        else if (m.tj == 16) rc = momentum_t<T, 16, MOIST, false, TURB>(c, a, T(step), m);
        else rc = momentum_t<T, 8, MOIST, false, TURB>(c, a, T(step), m);
    }
    if (rc || !(parts & kStageScalars)) return rc;
    const StageShape m = stage_shape(c, false);
    if (m.pack) {
        if (m.tj >= 6) return scalars_t<T, 8, MOIST, true, TURB>(c, a, T(step), m);
        if (m.tj >= 3) return scalars_t<T, 4, MOIST, true, TURB>(c, a, T(step), m);
        return scalars_t<T, 2, MOIST, true, TURB>(c, a, T(step), m);
    }
    if (m.tj == 2) return scalars_t<T, 2, MOIST, false, TURB>(c, a, T(step), m);
    if (m.tj == 4) return scalars_t<T, 4, MOIST, false, TURB>(c, a, T(step), m);
    if (m.tj == 12) return scalars_t<T, 12, MOIST, false, TURB>(c, a, T(step), m);
    return scalars_t<T, 8, MOIST, false, TURB>(c, a, T(step), m);
}

template <typename T>
int shell_t(Ctx *c, int il, int ih, int jl, int jh) {
    long long n = (long long)c->npts;
    Timed _t(c, "zero_moisture_shell", (double)n);
    hipLaunchKernelGGL(k_zero_moisture_shell<T>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream, c->geo, c->cols,
                       (T *)c->prog[DYN_QV][2], (T *)c->prog[DYN_QC][2], (T *)c->prog[DYN_QR][2], (const T *)c->bar[4], n, 3,
                       c->g.nx - 3, 3, c->g.ny - 3, il, ih, jl, jh);
    DYN_LAUNCH_CHECK();
    return DYN_OK;
}


// ---- boundary epilogues of a stage (PGF + apply_boundary_condition(_microphysics)) ------------------
// A wavefront owns one source column isrc in [3, NX-3) (lane = k) and writes that column's final values
// and, for the six columns the periodic copy feeds (boundaries.cpp:562-574), the halo column's values.
// Per field the reference's order is kept: sponge rows (boundaries.cpp:466-475), periodic copy, then the
// lid from i = 1, j = 1 (boundaries.cpp:304-326); column 0 therefore keeps the pre-lid values.  Lid
// values come from lanes 1 and NZ-2 through cross-lane reads, so no wavefront reads another's output.
struct PostArgs {
    void *f[7];          // UP VP WP THP QVP QCP QRP (forecast buffers)
    const void *pi, *qb;  // PI, QBAR
    const double *cs, *cn;
    int js, jn;
    int zl, zh, zjl, zjh;  // zero_moisture bounds (qv clip)
    // Rayleigh damping after the boundary update (end of a step): levels >= ray_level, coefficients
    // [u v theta][k] then [w][k]; ray_level >= NZ: none
    const double *ray = nullptr;
    int ray_level = 1 << 30;
    // turbulence tendencies of TH QV QC QR (nullptr: none) for the rows beside the advected box that the
    // diffusion's box [1, NY-1) still holds, in a stage (step, dt)
    const void *tend[4] = {};
    double step = 0.0;
};

template <typename T>
__device__ __forceinline__ T sponge_coef(const Geo &g, const PostArgs &a, int j) {
    if (j < a.js) return T(a.cs[j]);
    if (j >= g.NY - a.jn) return T(a.cn[j - (g.NY - a.jn)]);
    return T(-1);  // no sponge
}

template <typename T>
// damp: rayleigh_damping (damping.cpp:1148-1177) of the written values with coefficient cd on the
// columns it covers, i in [1, NX-1) (the caller checks j and k)
__device__ __forceinline__ void write_col(const Geo &g, T *A, int isrc, int j, int k, T fin, T prelid, bool damp = false,
                                          T cd = T(0)) {
    long long s = g.NYNZ;
    long long p = (long long)isrc * s + (long long)j * g.NZ + k;
    auto dv = [&](int i, T v) { return damp && i >= 1 && i < g.NX - 1 ? v - cd * v : v; };
    A[p] = dv(isrc, fin);
    const int shift = g.NX - 6;
    if (isrc >= shift && isrc < shift + 3) {
        int ih = isrc - shift;  // halo 0, 1, 2
        A[p - (long long)shift * s] = dv(ih, ih == 0 ? prelid : fin);
    }
    if (isrc >= 3 && isrc < 6) A[p + (long long)shift * s] = dv(isrc + shift, fin);
}

// PGF (solver.cpp:123-135) + sponge/periodic/lid for UP, VP and WP
template <typename T>
__device__ __forceinline__ void post_uvw_col(const Geo &g, const Cols &c, const PostArgs &a, T step, bool pgf, int jb, int isrc) {
    const int k = threadIdx.x;
    const int j = jb * blockDim.y + threadIdx.y;
    if (j >= g.NY) return;
    const int NZ = g.NZ;
    const int kc = k < NZ ? k : NZ - 1;
    const long long p = (long long)isrc * g.NYNZ + (long long)j * NZ + kc;
    T *UP = (T *)a.f[0], *VP = (T *)a.f[1], *WP = (T *)a.f[2];
    const T *PI = (const T *)a.pi;
    T u = UP[p], v = VP[p], w = WP[p];
    // every load of the column goes out before the arithmetic: the neighbours p - NYNZ, p - NZ, p - 1
    // lie inside the array for every source column (isrc >= 3), used or not
    const T pc = PI[p], pw = PI[p - g.NYNZ], psn = PI[p - NZ], pb = PI[p - 1];
    const double mwk = c.mw[kc];
    if (pgf && j >= 1 && j <= g.NY - 2 && kc >= 1 && kc <= NZ - 2) {
        u -= step * (T(g.dtx) * (pc - pw));
        v -= step * (T(g.dty) * (pc - psn));
        if (kc >= 2) w -= step * ((T(g.dtz) * T(mwk)) * (pc - pb));
    }
    T coef = sponge_coef<T>(g, a, j);
    if (coef >= T(0) && kc >= 1) {
        u -= coef * u;
        v -= coef * v;
        w -= coef * w;
    }
    // lid from lanes 1 and NZ-2 (j >= 1; every source column has i >= 1)
    const int lz = (NZ - 2) & (KP - 1);  // lane of level NZ-2 in its wavefront
    T u1 = lane_read(u, 1), uz = lane_read(u, lz), v1 = lane_read(v, 1), vz = lane_read(v, lz);
    if (k >= NZ) return;
    T uf = u, vf = v, wf = w;
    if (j >= 1) {
        if (k == 0) { uf = u1; vf = v1; }
        if (k == NZ - 1) { uf = uz; vf = vz; }
        if (k == 0 || k == 1 || k == NZ - 1) wf = T(0);
    }
    // Rayleigh damping after the boundary update (j in [1, NY-1), k >= level)
    const bool dm = k >= a.ray_level && j >= 1 && j < g.NY - 1;
    const T cu = dm ? T(a.ray[k]) : T(0), cw = dm ? T(a.ray[NZ + k]) : T(0);
    write_col(g, UP, isrc, j, k, uf, u, dm, cu);
    write_col(g, VP, isrc, j, k, vf, v, dm, cu);
    write_col(g, WP, isrc, j, k, wf, w, dm, cw);
}

// sponge/periodic/lid for THP (and QVP, QCP, QRP with zero_moisture outside the advected box); only the
// columns a sponge row, a ghost row or the periodic copy touches are rewritten whole, the others get the
// two lid levels
// lid_interior: also set the lid of the interior columns (the stage advection already did after a stage;
// after Kessler it must be redone)
template <typename T, bool MOIST>
__device__ __forceinline__ void post_scalars_col(const Geo &g, const Cols &c, const PostArgs &a, bool clip, bool lid_interior, int j,
                                                 int isrc) {
    const int k = threadIdx.x;
    if (j >= g.NY) return;
    const int NZ = g.NZ;
    const int kc = k < NZ ? k : NZ - 1;
    const long long col = (long long)isrc * g.NYNZ + (long long)j * NZ;
    const T coef = sponge_coef<T>(g, a, j);
    const bool full = coef >= T(0) || j < 3 || j >= g.NY - 3 || isrc < 6 || isrc >= g.NX - 6;
    constexpr int NFLD = MOIST ? 4 : 1;
    if (!full) {  // interior column: lid only (values at 1 and NZ-2 are final already)
        // with Rayleigh damping (end of a step) theta is rewritten from level ray_level up as well: the
        // lid from the undamped levels 1 and NZ-2, then the damping (j in [3, NY-3) here)
        const bool ray = a.ray_level < NZ;
        if (lid_interior && j >= 1 && (k == 0 || k == NZ - 1)) {
            int ks = k == 0 ? 1 : NZ - 2;
#pragma unroll
            for (int f = ray ? 1 : 0; f < NFLD; f++) {
                T *A = (T *)a.f[3 + f];
                A[col + k] = A[col + ks];
            }
        }
        if (ray) {
            T *A = (T *)a.f[3];
            const T x = A[col + kc];
            const T x1 = lane_read(x, 1), xz = lane_read(x, (NZ - 2) & (KP - 1));
            const bool lid = lid_interior && (k == 0 || k == NZ - 1);
            if (k < NZ && (lid || k >= a.ray_level)) {
                T fin = k == 0 && lid ? x1 : (k == NZ - 1 && lid ? xz : x);
                if (k >= a.ray_level) fin = fin - T(a.ray[k]) * fin;
                A[col + k] = fin;
            }
        }
        return;
    }
    const bool edge = a.tend[0] && j >= 1 && j < g.NY - 1 && (j < 3 || j >= g.NY - 3);
#pragma unroll
    for (int f = 0; f < NFLD; f++) {
        T *A = (T *)a.f[3 + f];
        T x = A[col + kc];
        if (edge && kc >= 1 && kc <= NZ - 2) {
            const T d = ((const T *)a.tend[f])[col + kc];
            if (f == 0) x += d * T(a.step) * T(g.dt);
            else x += d * (T(a.step) * T(g.dt));
        }
        if (MOIST && clip && f == 2 && x < T(0)) x = T(0);  // qc
        if (MOIST && clip && f == 3 && x < T(0)) x = T(0);  // qr
        if (MOIST && clip && f == 1 && isrc >= a.zl && isrc < a.zh && j >= a.zjl && j < a.zjh && kc >= 1 && kc <= NZ - 2) {
            T qbp = ((const T *)a.qb)[col + kc];
            if (x + qbp + T(c.qb[kc]) < T(0)) x = -(qbp + T(c.qb[kc]));
        }
        if (coef >= T(0) && kc >= 1) x -= coef * x;
        T x1 = lane_read(x, 1), xz = lane_read(x, (NZ - 2) & (KP - 1));
        if (k < NZ) {
            T fin = x;
            if (j >= 1) {
                if (k == 0) fin = x1;
                if (k == NZ - 1) fin = xz;
            }
            // Rayleigh damping of theta after its boundary update (j in [1, NY-1), k >= level)
            const bool dm = f == 0 && k >= a.ray_level && j >= 1 && j < g.NY - 1;
            write_col(g, A, isrc, j, k, fin, x, dm, dm ? T(a.ray[k]) : T(0));
        }
    }
}

template <typename T>
__global__ void __launch_bounds__(256) k_post_uvw(Geo g, Cols c, PostArgs a, T step, bool pgf) {
    post_uvw_col<T>(g, c, a, step, pgf, blockIdx.x, blockIdx.y + 3);
}
template <typename T, bool MOIST>
__global__ void __launch_bounds__(256) k_post_scalars(Geo g, Cols c, PostArgs a, bool clip, bool lid_interior) {
    post_scalars_col<T, MOIST>(g, c, a, clip, lid_interior, blockIdx.x * blockDim.y + threadIdx.y, blockIdx.y + 3);
}

// Source columns post_scalars_col rewrites whole when the interior lids are already set (after a
// stage): rows j < rl and j >= NY - rh (sponge and ghost rows) for every isrc in [3, NX-3), then, on the
// other rows, the six periodic source columns.  One wavefront per column, item = its index in that list.
struct ShellCols {
    int rl, rh, nb, ni;  // low rows, high rows, rows between, source columns (NX - 6)
    int ncb;             // periodic source columns (6, or every column on a narrow grid)
    int total;
};
inline ShellCols shell_cols(const Ctx *c) {
    ShellCols s;
    const int NY = c->g.ny, ni = c->g.nx - 6;
    s.rl = std::min(NY, std::max(c->g.sponge_south, 3));
    s.rh = std::min(NY - s.rl, std::max(c->g.sponge_north, 3));
    s.nb = NY - s.rl - s.rh;
    s.ni = ni;
    s.ncb = ni <= 6 ? ni : 6;
    s.total = (s.rl + s.rh) * ni + s.ncb * s.nb;
    return s;
}
__device__ __forceinline__ bool shell_item(const Geo &g, const ShellCols &s, int item, int &j, int &isrc) {
    if (item >= s.total) return false;
    const int na = (s.rl + s.rh) * s.ni;
    if (item < na) {
        const int r = item / s.ni;
        isrc = 3 + item % s.ni;
        j = r < s.rl ? r : g.NY - s.rh + (r - s.rl);
    } else {
        const int q = item - na, cb = q / s.nb;
        j = s.rl + q % s.nb;
        isrc = s.ni <= 6 ? 3 + cb : (cb < 3 ? 3 + cb : g.NX - 6 + (cb - 3));
    }
    return true;
}
template <typename T, bool MOIST>
__global__ void __launch_bounds__(256) k_post_scalars_shell(Geo g, Cols c, PostArgs a, bool clip, ShellCols s) {
    int j, isrc;
    if (shell_item(g, s, blockIdx.x * blockDim.y + threadIdx.y, j, isrc)) post_scalars_col<T, MOIST>(g, c, a, clip, false, j, isrc);
}

// Both in one launch: nu blocks of u, v, w, then the scalars' shell (shell: the items of s) or every column
template <typename T, bool MOIST>
__global__ void __launch_bounds__(256) k_post_all(Geo g, Cols c, PostArgs a, T step, bool pgf, int nu, bool clip, bool shell, ShellCols s) {
    const int nbj = (g.NY + blockDim.y - 1) / blockDim.y;
    int b = blockIdx.x;
    if (b < nu) {
        post_uvw_col<T>(g, c, a, step, pgf, b % nbj, b / nbj + 3);
        return;
    }
    b -= nu;
    int j, isrc;
    if (!shell) post_scalars_col<T, MOIST>(g, c, a, clip, true, b % nbj * blockDim.y + threadIdx.y, b / nbj + 3);
    else if (shell_item(g, s, b * blockDim.y + threadIdx.y, j, isrc)) post_scalars_col<T, MOIST>(g, c, a, clip, false, j, isrc);
}

// ---- batched over the members of an ensemble: one block per work item of the concatenated work list ----
__device__ __forceinline__ StageArgs ens_stage_args(const EnsMember &e, const EnsRoles &ro, int tj, int ti, int nbj) {
    StageArgs a;
    a.tj = tj;
    for (int f = 0; f < 7; f++) {
        a.cur[f] = e.buf[f][ro.r[f][DYN_ROLE_CUR]];
        a.mprev[f] = e.buf[f][ro.r[f][DYN_ROLE_M]];
        a.out[f] = e.buf[f][ro.r[f][DYN_ROLE_P]];
    }
    for (int f = 0; f < 5; f++) a.bar[f] = e.bar[f];
    a.vt = e.vt;
    a.il = 3;
    a.ih = e.g.NX - 3;
    a.jl = 3;
    a.jh = e.g.NY - 3;
    a.ti = ti;
    a.nbj = nbj;
    return a;
}
__device__ __forceinline__ PostArgs ens_post_args(const EnsMember &e, const EnsRoles &ro) {
    PostArgs a;
    for (int f = 0; f < 7; f++) a.f[f] = e.buf[f][ro.r[f][DYN_ROLE_P]];
    a.pi = e.pi;
    a.qb = e.bar[4];
    a.cs = e.sponge_s;
    a.cn = e.sponge_n;
    a.js = e.js;
    a.jn = e.jn;
    a.zl = 1;
    a.zh = e.g.NX - 1;
    a.zjl = 1;
    a.zjh = e.g.NY - 1;
    return a;
}

template <typename T, int TJ, bool MOIST, bool PACK>
__global__ void __launch_bounds__((stage_threads<TJ, PACK>())) k_ens_momentum(const EnsMember *mem, int nmem, EnsRoles ro, T step,
                                                                                   int tj, int ti, int total) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int item = xcd_tile(blockIdx.x, gridDim.x);
    const EnsMember &e = mem[ens_member(mem, nmem, item, &EnsMember::mom0)];
    const StageArgs a = ens_stage_args(e, ro, tj, ti, e.nbj_mom);
    adv_momentum_tile<T, TJ, MOIST, PACK>(e.g, e.c, a, step, item - e.mom0, smem_raw);
}

template <typename T, int TJ, bool MOIST, bool PACK>
__global__ void __launch_bounds__((stage_threads<TJ, PACK>())) k_ens_scalars(const EnsMember *mem, int nmem, EnsRoles ro, T step,
                                                                                   int tj, int ti, int total) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int item = xcd_tile(blockIdx.x, gridDim.x);
    const EnsMember &e = mem[ens_member(mem, nmem, item, &EnsMember::scal0)];
    const StageArgs a = ens_stage_args(e, ro, tj, ti, e.nbj_scal);
    adv_scalars_tile<T, TJ, kTheta, PACK>(e.g, e.c, a, step, item - e.scal0, smem_raw);
}

template <typename T>
__global__ void __launch_bounds__(256) k_ens_post(const EnsMember *mem, int nmem, EnsRoles ro, T step, bool pgf, bool scalars, int total) {
    const int item = xcd_tile(blockIdx.x, gridDim.x);
    const EnsMember &e = mem[ens_member(mem, nmem, item, &EnsMember::post0)];
    const PostArgs a = ens_post_args(e, ro);
    const int local = item - e.post0, nb = (e.g.NY + 3) / 4;
    post_uvw_col<T>(e.g, e.c, a, step, pgf, local % nb, local / nb + 3);
    if (scalars) post_scalars_col<T, false>(e.g, e.c, a, false, !pgf, (local % nb) * blockDim.y + threadIdx.y, local / nb + 3);
}

// advance_outer's memcpy(M <- P) for u, v, w, theta of every member; work items are 1024-element chunks
template <typename T>
__global__ void __launch_bounds__(256) k_ens_copy(const EnsMember *mem, int nmem, EnsRoles ro, int total) {
    {
        const int item = blockIdx.x;
        const EnsMember &e = mem[ens_member(mem, nmem, item, &EnsMember::cp0)];
        const long long n = (long long)e.g.NX * e.g.NYNZ;
        const long long per = (n + 1023) / 1024;
        const int local = item - e.cp0;
        const int fi = local / (int)per;
        const int f = fi == 0 ? DYN_U : fi == 1 ? DYN_V : fi == 2 ? DYN_W : DYN_TH;
        T *dst = (T *)e.buf[f][ro.r[f][DYN_ROLE_M]];
        const T *src = (const T *)e.buf[f][ro.r[f][DYN_ROLE_P]];
        const long long base = (long long)(local % (int)per) * 1024;
        for (long long p = base + threadIdx.x; p < base + 1024 && p < n; p += blockDim.x) dst[p] = src[p];
    }
}

template <typename T>
int post_t(Ctx *c, double step, bool pgf, bool scalars, bool clip, bool uvw, int ray_level, bool interior_done) {
    PostArgs a{};
    if (ray_level >= 0 && ray_level < c->g.nz) {
        a.ray = c->raycoef;
        a.ray_level = ray_level;
    }
    for (int f = 0; f < 7; f++) a.f[f] = c->prog[f][DYN_ROLE_P];
    a.pi = c->pi;
    a.qb = c->bar[4];
    a.cs = c->sponge_s;
    a.cn = c->sponge_n;
    a.js = c->g.sponge_south;
    a.jn = c->g.sponge_north;
    a.zl = 1;
    a.zh = c->g.nx - 1;
    a.zjl = 1;
    a.zjh = c->g.ny - 1;
    if (c->turb.on && pgf) {
        for (int f = 0; f < 4; f++) a.tend[f] = turb_tendency(c, DYN_TH + f);
        a.step = step;
    }
    // one wavefront per column, two when NZ > 64; 256 threads per block
    const int kw = c->g.nz > KP ? 2 : 1, rows = 4 / kw;
    dim3 blk(KP * kw, rows), grd((c->g.ny + rows - 1) / rows, c->g.nx - 6);
    if (uvw && scalars && stage_in_one(c)) {
        Timed _t(c, "post_all", (double)c->npts);
        const bool shell = pgf || interior_done;
        const ShellCols sc = shell_cols(c);
        const int nu = grd.x * grd.y, ns = shell ? (sc.total + rows - 1) / rows : nu;
        if (c->g.microphysics)
            hipLaunchKernelGGL((k_post_all<T, true>), dim3(nu + ns), blk, 0, c->stream, c->geo, c->cols, a, T(step), pgf, nu, clip, shell, sc);
        else
            hipLaunchKernelGGL((k_post_all<T, false>), dim3(nu + ns), blk, 0, c->stream, c->geo, c->cols, a, T(step), pgf, nu, clip, shell, sc);
        DYN_LAUNCH_CHECK();
        return DYN_OK;
    }
    if (uvw) {
        Timed _t(c, "post_uvw", (double)c->npts);
        hipLaunchKernelGGL(k_post_uvw<T>, grd, blk, 0, c->stream, c->geo, c->cols, a, T(step), pgf);
        DYN_LAUNCH_CHECK();
    }
    if (scalars) {
        Timed _t(c, "post_scalars", (double)c->npts);
        // after a stage the advection kernel has set the interior lids; at the end of the step (no
        // gradient force) Kessler has changed the interior, so they are redone
        const bool lid_interior = !pgf;
        if (!lid_interior || interior_done) {  // only the sponge rows, ghost rows and periodic source columns change
            const ShellCols sc = shell_cols(c);
            const dim3 gs((unsigned)std::max(1, (sc.total + rows - 1) / rows));
            if (c->g.microphysics)
                hipLaunchKernelGGL((k_post_scalars_shell<T, true>), gs, blk, 0, c->stream, c->geo, c->cols, a, clip, sc);
            else hipLaunchKernelGGL((k_post_scalars_shell<T, false>), gs, blk, 0, c->stream, c->geo, c->cols, a, clip, sc);
        } else if (c->g.microphysics) {
            hipLaunchKernelGGL((k_post_scalars<T, true>), grd, blk, 0, c->stream, c->geo, c->cols, a, clip, lid_interior);
        } else {
            hipLaunchKernelGGL((k_post_scalars<T, false>), grd, blk, 0, c->stream, c->geo, c->cols, a, clip, lid_interior);
        }
        DYN_LAUNCH_CHECK();
    }
    return DYN_OK;
}

}  // namespace

// Wavefronts per column of the boundary kernels: one up to NZ = 64; two for NZ in [66, 128], where the lid's
// source levels 1 and NZ-2 sit in the wavefronts of the levels they feed (0 and NZ-1); 0 otherwise: the
// fused step is not offered
int fused_waves(const Ctx *c) {
    const int nz = c->g.nz;
    return nz <= KP ? 1 : (nz >= KP + 2 && nz <= 2 * KP ? 2 : 0);
}

// ... and 32-bit byte offsets into every field
bool fused_supported(const Ctx *c) {
    return fused_waves(c) > 0 && (double)c->npts * (double)c->elt < 4294967296.0;
}

namespace {
// LDS bytes per block of a stage kernel with tj rows of `pitch` lanes
size_t stage_lds(const Ctx *c, bool momentum, int tj, int pitch) {
    const bool moist = c->g.microphysics != 0;
    if (c->prec == DYN_FP32)
        return momentum ? MomLds<float>::bytes(tj, pitch) : moist ? scalar_lds<float, true>(tj, pitch) : scalar_lds<float, false>(tj, pitch);
    return momentum ? MomLds<double>::bytes(tj, pitch) : moist ? scalar_lds<double, true>(tj, pitch) : scalar_lds<double, false>(tj, pitch);
}
}  // namespace

// launch-shape knobs of the stage kernels: rows per block (2, 4 and 8 up to 64 levels, and 16 for the
// momentum kernel, 12 for the scalar kernel; 2 and 4 above; within the LDS that rows of whole wavefronts
// take) and march length
bool fused_shape_ok(const Ctx *c, int param, int value) {
    if (param == DYN_TUNE_MOMENTUM_TJ || param == DYN_TUNE_SCALAR_TJ) {
        const bool one = fused_waves(c) != 2, mom = param == DYN_TUNE_MOMENTUM_TJ;
        const bool inst = value == 2 || value == 4 || (one && (value == 8 || value == (mom ? 16 : 12)));
        return inst && stage_lds(c, mom, value, KP * (one ? 1 : 2)) <= c->pp.lds_max;
    }
    if (param == DYN_TUNE_MOMENTUM_TI || param == DYN_TUNE_SCALAR_TI) return value >= 2 && value <= 512;
    if (param == DYN_TUNE_PRESSURE_JPASS) return value == 2 || (value == 1 && c->pp.fused_y) || (value == 3 && c->pp.half_y);
    if (param == DYN_TUNE_STAGE_STREAMS) return value >= 1 && value <= 4;
    return false;
}

namespace {
// The FP32 scalar kernel on one stream (no pressure pass beside it): 12 rows per block (three waves per
// SIMD at its register count, one block per CU) and march lengths that make one round of blocks fill the
// device.  Measured at 256x256x64 moist: 92.7 us against 104.2 us for 8 rows x 16 columns, one-stream
// step 0.956 against 0.990 ms.  Beside the pressure solve 8 rows stay faster (the scalar blocks must
// leave room for the solve's).
bool scalar_one_round(const Ctx *c) {
    if (c->prec != DYN_FP32 || fused_waves(c) != 1 || c->pp.cus <= 0) return false;
    if (c->tune[DYN_TUNE_STAGE_STREAMS] != 1) return false;  // one stream only when asked for
    return fused_shape_ok(c, DYN_TUNE_SCALAR_TJ, 12);
}
}  // namespace

int fused_shape(const Ctx *c, int param) {
    if (c->tune[param]) return c->tune[param];
    const bool f32 = c->prec == DYN_FP32;
    // FP64: 8 rows per block when that still gives two blocks per CU at 16 columns per block (measured
    // 8 % faster at 256x256x64), else 4
    const int rows8 = ((c->g.ny - 6 + 7) / 8) * ((c->g.nx - 6 + 15) / 16);
    const int tj = f32 || rows8 >= 512 ? 8 : 4;
    switch (param) {
    case DYN_TUNE_MOMENTUM_TJ:
    case DYN_TUNE_SCALAR_TJ:
        // two wavefronts per column: blocks of 512 threads (4 rows) where the LDS allows and the moist
        // FP64 scalar kernel keeps its registers (at 4 rows it spills), else 2 rows
        if (fused_waves(c) == 2) {
            if (!f32 && param == DYN_TUNE_SCALAR_TJ && c->g.microphysics) return 2;
            return fused_shape_ok(c, param, 4) ? 4 : 2;
        }
        if (param == DYN_TUNE_SCALAR_TJ && scalar_one_round(c)) return 12;
        return tj;
    case DYN_TUNE_MOMENTUM_TI: return fused_waves(c) == 2 ? 32 : 16;  // 512x512x80: 32 measured 3 % faster
    // (Nominal values; while the knobs are unset stage_streams and stage_shape decide.)
    // The scalar kernel beside the pressure solve (fork after the momentum kernel): 24 columns, about 2 %
    // faster per step than 16 (FP32 at 256x256x64 moist and 192x192x40 dry, FP64 at 192x192x40 dry).
    // Its 352 blocks at 256x256 leave most CUs one block, beside which a j-pass block still fits; alone
    // the kernel is slower that way (165 against 120 us), so the one-stream step keeps 16, and so does
    // the later fork, where 16 measured best.
    case DYN_TUNE_SCALAR_TI:
        if (fused_waves(c) == 2) return 32;
        if (scalar_one_round(c)) {  // as many i-chunks per 12-row band as leave every block one CU, at
                                    // least 16 columns each (shorter marches spend more on the queue fill)
            const int nbj = (c->g.ny - 6 + 11) / 12, per = std::max(1, c->pp.cus / nbj);
            return std::min(512, std::max(16, (c->g.nx + per - 1) / per));
        }
        {
            const int streams = fused_shape(c, DYN_TUNE_STAGE_STREAMS);
            return streams == 2 || streams == 4 ? 24 : 16;
        }
    case DYN_TUNE_PRESSURE_JPASS: return c->pp.fused_y ? 1 : (c->pp.half_y ? 3 : 2);
    // the scalar half forked after the pressure solve's first pass where the j pass runs on half slabs
    // (FP64 256x256x64: 4 % faster); after the momentum kernel elsewhere (FP32 there: 7 % faster), in
    // FP64 with its launches queued after the first pass (192x192x40: 5 % faster)
    case DYN_TUNE_STAGE_STREAMS: return fused_shape(c, DYN_TUNE_PRESSURE_JPASS) == 3 ? 3 : (f32 ? 2 : 4);
    default: return DYN_E_ARG;
    }
}

namespace {
// Modelled microseconds of a stage kernel's launch with tj rows and ti columns per block.  A block marches
// ti columns after a prologue worth about one more; a column takes `lat` while few wavefronts share a SIMD
// (the march is a chain of barriers and loads) and `issue` for each wavefront on the fullest SIMD once
// they are many; blocks beyond what fits on a CU wait for a round of their own, and each block loads six
// halo rows beside its own.  Blocks whose wavefronts do not fill the four SIMDs evenly run at the pace of
// the fullest one: at 192x192x40 (FP32 moist) the momentum kernel takes 26.7 us with 6 rows (4 wavefronts),
// 36.6 with 8 (5 wavefronts) and 27.6 with 12 (8 wavefronts).  The constants are fitted to timings of
// 32x32x20 to 512x512x80 grids in every form, 2 to 25 rows and 2 to 32 columns (one kernel on the device);
// the shape the model picks is within 10 % of the fastest of them in all but the smallest launches.
struct StageCost {
    double lat, issue;
    int simd;  // wavefronts per SIMD that the kernel's registers allow
};
StageCost stage_cost(const Ctx *c, bool momentum) {
    const bool f32 = c->prec == DYN_FP32, moist = c->g.microphysics != 0;
    if (momentum) return f32 ? StageCost{1.65, 0.70, 4} : StageCost{2.15, 1.40, 2};
    if (moist) return f32 ? StageCost{2.70, 1.00, 3} : StageCost{1.60, 1.20, 2};
    return f32 ? StageCost{1.00, 0.38, 5} : StageCost{1.40, 0.65, 3};
}
double stage_model(const Ctx *c, bool momentum, bool pack, int tj, int ti, long long blocks) {
    const StageCost k = stage_cost(c, momentum);
    const int waves = pack ? (tj * c->g.nz + KP - 1) / KP : tj, per_simd = (waves + 3) / 4, cus = std::max(1, c->pp.cus);
    const int fit = std::max(1, std::min(k.simd / per_simd, (int)(c->pp.lds_max / stage_lds(c, momentum, tj, pack ? c->g.nz : KP))));
    const int per_cu = (int)((blocks + cus - 1) / cus);
    auto column = [&](int n) { return n ? std::max(k.lat, k.issue * n * per_simd) : 0.0; };
    return (ti + 1) * (per_cu / fit * column(fit) + column(per_cu % fit)) * (1.0 + 0.3 / tj);
}
}  // namespace

// The launch of a stage kernel.  With a knob of its own set, or on grids of 57 to 64 levels whose nominal
// blocks (fused_shape) number one per CU or more, the nominal shape; else the one the model above takes to
// be fastest: small grids get short marches (64x64x40 FP32: momentum 34.3 us in 32 blocks of 16 columns,
// 10.0 in 256 of 2), and packed rows the row count that fills whole groups of four wavefronts.
StageShape stage_shape(const Ctx *c, bool momentum) {
    const int ptj = momentum ? DYN_TUNE_MOMENTUM_TJ : DYN_TUNE_SCALAR_TJ, pti = momentum ? DYN_TUNE_MOMENTUM_TI : DYN_TUNE_SCALAR_TI;
    if (!c->tune[ptj] && !c->tune[pti] && c->auto_shape[momentum].tj) return c->auto_shape[momentum];
    StageShape s{fused_shape(c, ptj), fused_shape(c, pti), stage_packs(c)};
    if (s.pack && s.tj * c->g.nz > kPackThreads) s.pack = false;  // 12 or 16 rows asked for
    return s;
}

bool stage_in_one(const Ctx *c) {
    for (int p : {DYN_TUNE_MOMENTUM_TJ, DYN_TUNE_MOMENTUM_TI, DYN_TUNE_SCALAR_TJ, DYN_TUNE_SCALAR_TI, DYN_TUNE_STAGE_STREAMS})
        if (c->tune[p]) return false;
    return c->auto_one.tj > 0;
}

// How a step's stages use the second stream (the values of DYN_TUNE_STAGE_STREAMS) while the knob is unset.
// With short marches the scalar kernel no longer delays the divergence pass it is queued behind, so the late
// queueing (4) is the faster form nearly everywhere (us per step, nominal form against 4: FP32 moist 344 and
// 319 at 128x128x64, 679 and 655 at 256x256x40; FP64 579 and 522 moist at 128x128x64, 1314 and 1239 dry at
// 256x256x64); the largest moist FP32 grids keep the nominal form (256x256x64: 833 against 874).  FP64 moist on
// half slabs at 256x256x64, us per step by form and scalar march: 2 1742 (16 columns) and 1785 (24), 3 1820 and 1804,
// 4 1805 and 1737; 16 columns is the march in force.
int stage_streams(const Ctx *c) {
    const int nominal = fused_shape(c, DYN_TUNE_STAGE_STREAMS);
    if (c->tune[DYN_TUNE_STAGE_STREAMS]) return nominal;
    return nominal == 2 && c->g.microphysics && c->npts >= 3000000u ? nominal : 4;
}

int tune_in_force(const Ctx *c, int param) {
    const bool one = stage_in_one(c);
    switch (param) {
    case DYN_TUNE_MOMENTUM_TJ: return one ? c->auto_one.tj : stage_shape(c, true).tj;
    case DYN_TUNE_MOMENTUM_TI: return one ? c->auto_one.ti_mom : stage_shape(c, true).ti;
    case DYN_TUNE_SCALAR_TJ: return one ? c->auto_one.tj : stage_shape(c, false).tj;
    case DYN_TUNE_SCALAR_TI: return one ? c->auto_one.ti_scal : stage_shape(c, false).ti;
    case DYN_TUNE_PRESSURE_JPASS: return pressure_jpass(c);
    case DYN_TUNE_STAGE_STREAMS: return one ? 1 : stage_streams(c);
    default: return DYN_E_ARG;
    }
}

namespace {
// auto_shape of both kernels; left empty (tj = 0) where the nominal shape is kept
void choose_stage_shapes(Ctx *c) {
    const bool pack = stage_packs(c), two = c->g.microphysics && c->prec == DYN_FP64;  // scalar_parts
    const int nx = c->g.nx - 6, ny = c->g.ny - 6;
    for (int m = 0; m < 2; m++) {
        const bool momentum = m == 1;
        c->auto_shape[m] = StageShape{0, 0, pack};
        if (!pack) {
            const int tj = fused_shape(c, momentum ? DYN_TUNE_MOMENTUM_TJ : DYN_TUNE_SCALAR_TJ);
            const int ti = fused_shape(c, momentum ? DYN_TUNE_MOMENTUM_TI : DYN_TUNE_SCALAR_TI);
            if ((long long)((ny + tj - 1) / tj) * ((nx + ti - 1) / ti) >= c->pp.cus) continue;
        }
        double best = 0.0;
        for (int tj = 2; tj * (pack ? c->g.nz : KP) <= kPackThreads; tj++) {
            if (!pack && tj != 2 && tj != 4 && tj != 8) continue;
            if (stage_lds(c, momentum, tj, pack ? c->g.nz : KP) > c->pp.lds_max) continue;
            for (int ti = 2; ti <= 48; ti++) {
                const long long n = (long long)((ny + tj - 1) / tj) * ((nx + ti - 1) / ti) * (!momentum && two ? 2 : 1);
                const double t = stage_model(c, momentum, pack, tj, ti, n);
                if (c->auto_shape[m].tj == 0 || t < best) {
                    best = t;
                    c->auto_shape[m] = StageShape{tj, ti, pack};
                }
            }
        }
    }
}

// One launch for both halves of a stage: the shape with the shortest longest march among those whose blocks all run
// at once (the registers and LDS of the heavier half count for every block), where the model gives it 12 us or
// less, 15 with the scalar half in two parts.  Past that the halves are worth two streams (us per step, two streams
// against one launch, with the model's figure: dry FP32 159 and 142 at 64x64x40 (5.1), 230 and 221 at 128x96x40
// (11.0), 268 and 277 at 150x126x50 (19.3); dry FP64 122 and 96 at 32x32x20 (6.6), 195 and 191 at 64x64x64 (11.6),
// 247 and 257 at 128x96x40 (20.1); moist FP32 194 and 184 at 64x64x64 (11.3), 218 and 225 at 64x64x80 (13.2);
// moist FP64 213 and 201 at 64x64x40 (14.3), 225 and 241 at 64x64x64 (20.3)).
void choose_stage_one(Ctx *c) {
    c->auto_one = StageOne{};
    const bool pack = stage_packs(c);
    const int nx = c->g.nx - 6, ny = c->g.ny - 6, pitch = pack ? c->g.nz : KP, cus = std::max(1, c->pp.cus);
    const StageCost km = stage_cost(c, true), ks = stage_cost(c, false);
    const int simd = std::min(km.simd, ks.simd), parts = c->g.microphysics && c->prec == DYN_FP64 ? 2 : 1;
    double best = 0.0;
    for (int tj = 2; tj * pitch <= kPackThreads; tj++) {
        if (!pack && tj != 2 && tj != 4 && tj != 8) continue;
        const size_t lds = std::max(stage_lds(c, true, tj, pitch), stage_lds(c, false, tj, pitch));
        if (lds > c->pp.lds_max) continue;
        const int waves = pack ? (tj * c->g.nz + KP - 1) / KP : tj, per_simd = (waves + 3) / 4;
        const int fit = std::min(simd / per_simd, (int)(c->pp.lds_max / lds)), nbj = (ny + tj - 1) / tj;
        for (int tm = 2; tm <= 32; tm++)
            for (int ts = 2; ts <= 32; ts++) {
                const int n = nbj * ((nx + tm - 1) / tm + parts * ((nx + ts - 1) / ts)), per_cu = (n + cus - 1) / cus;
                if (per_cu > fit) continue;
                const double t = std::max((tm + 1) * std::max(km.lat, km.issue * per_cu * per_simd),
                                          (ts + 1) * std::max(ks.lat, ks.issue * per_cu * per_simd)) * (1.0 + 0.3 / tj);
                if (c->auto_one.tj == 0 || t < best) {
                    best = t;
                    c->auto_one = StageOne{tj, tm, ts};
                }
            }
    }
    if (best > (parts == 2 ? 15.0 : 12.0)) c->auto_one = StageOne{};
}

template <typename T, int TJ, bool MOIST, bool PACK, bool TURB>
int set_lds_limits(const Ctx *c) {
    const int most = (int)c->pp.lds_max;
    const void *k[] = {(const void *)k_adv_stage<T, TJ, MOIST, PACK, TURB>, (const void *)k_adv_momentum<T, TJ, MOIST, PACK, TURB>,
                       (const void *)k_adv_scalars<T, TJ, MOIST, PACK, TURB>};
    for (const void *f : k) DYN_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, most));
    return DYN_OK;
}

template <typename T, bool MOIST, bool TURB>
int set_lds_limits_all(const Ctx *c) {
    int rc = set_lds_limits<T, 2, MOIST, true, TURB>(c);
    if (!rc) rc = set_lds_limits<T, 4, MOIST, true, TURB>(c);
    if (!rc) rc = set_lds_limits<T, 8, MOIST, true, TURB>(c);
    if (!rc) rc = set_lds_limits<T, 2, MOIST, false, TURB>(c);
    if (!rc) rc = set_lds_limits<T, 4, MOIST, false, TURB>(c);
    if (!rc) rc = set_lds_limits<T, 8, MOIST, false, TURB>(c);
    if (rc) return rc;
    const int most = (int)c->pp.lds_max;
    const void *k[] = {(const void *)k_adv_momentum<T, 16, MOIST, false, TURB>, (const void *)k_adv_scalars<T, 12, MOIST, false, TURB>};
    for (const void *f : k) DYN_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, most));
    return DYN_OK;
}
}  // namespace

// the stage kernels may use more than 64 KiB of LDS: raise the per-launch limit once, outside any capture
int fused_lds_limits(Ctx *c, bool turbulence) {
    auto run = [&](auto turb) {
        constexpr bool TURB = decltype(turb)::value;
        if (c->prec == DYN_FP32)
            return c->g.microphysics ? set_lds_limits_all<float, true, TURB>(c) : set_lds_limits_all<float, false, TURB>(c);
        return c->g.microphysics ? set_lds_limits_all<double, true, TURB>(c) : set_lds_limits_all<double, false, TURB>(c);
    };
    return turbulence ? run(std::true_type{}) : run(std::false_type{});
}

// rows per block that a batch's stage kernels take: any number of packed rows that fit, else the instances' own
bool ens_rows_ok(const Ctx *c0, bool momentum, int tj) {
    if (!stage_packs(c0)) return tj == 2 || tj == 4 || tj == 8;
    return tj >= 2 && tj <= kPackThreads / c0->g.nz && stage_lds(c0, momentum, tj, c0->g.nz) <= c0->pp.lds_max;
}

// The model's shape for a batch's blocks; without packed rows the nominal one.  Most batches fill the chip many times
// over, so what counts is whole groups of four wavefronts and long marches (32 FP32 members of 96 to 192 points a
// side and 40 levels, in two batches: momentum 265 us a launch in blocks of 8 rows and 16 columns, 200 in the model's;
// scalars 142 and 130).
void choose_ens_shape(const Ctx *c0, const std::vector<std::pair<int, int>> &sides, int *shape) {
    const int nominal = c0->prec == DYN_FP32 ? 8 : 4;
    for (int m = 0; m < 2; m++) {
        shape[2 * m] = nominal;
        shape[2 * m + 1] = 16;
        if (!stage_packs(c0)) continue;
        double best = 0.0;
        for (int tj = 2; tj * c0->g.nz <= kPackThreads; tj++) {
            if (!ens_rows_ok(c0, m == 0, tj)) continue;
            for (int ti = 2; ti <= 48; ti++) {
                long long n = 0;
                for (const auto &p : sides) n += (long long)((p.second + tj - 1) / tj) * ((p.first + ti - 1) / ti);
                const double t = stage_model(c0, m == 0, true, tj, ti, n);
                if (best == 0.0 || t < best) {
                    best = t;
                    shape[2 * m] = tj;
                    shape[2 * m + 1] = ti;
                }
            }
        }
    }
}

int fused_prepare(Ctx *c) {
    choose_stage_shapes(c);
    choose_stage_one(c);
    return fused_lds_limits(c, false);
}

// advect_uvw_velocity + advect_theta (+ advect_microphysics_cell and the interior zero_moisture)
// over the box [il,ih) x [jl,jh)
int launch_fused_advect(Ctx *c, double step, int il, int ih, int jl, int jh, int parts) {
    // the i-queues reach columns il-3 .. ih+2 and the planes rows jl-3 .. jh+2
    if (il < 3 || ih > c->g.nx - 3 || jl < 3 || jh > c->g.ny - 3 || il >= ih || jl >= jh) {
        set_error("fused stage: box outside [3, NX-3) x [3, NY-3)");
        return DYN_E_ARG;
    }
    const bool moist = c->g.microphysics != 0;
    auto run = [&](auto turb) {
        constexpr bool TURB = decltype(turb)::value;
        if (c->prec == DYN_FP32)
            return moist ? stage_t<float, true, TURB>(c, step, il, ih, jl, jh, parts) : stage_t<float, false, TURB>(c, step, il, ih, jl, jh, parts);
        return moist ? stage_t<double, true, TURB>(c, step, il, ih, jl, jh, parts) : stage_t<double, false, TURB>(c, step, il, ih, jl, jh, parts);
    };
    return c->turb.on ? run(std::true_type{}) : run(std::false_type{});
}

// PGF (optional) and the boundary update of every prognostic after launch_fused_advect; stands for
// dyn_pgf + zero_moisture's remainder + dyn_apply_bc + dyn_apply_bc_micro of one stage
int launch_post_stage(Ctx *c, double step, bool pgf, bool scalars, bool clip, bool uvw, int ray_level, bool interior_done) {
    if (c->prec == DYN_FP32) return post_t<float>(c, step, pgf, scalars, clip, uvw, ray_level, interior_done);
    return post_t<double>(c, step, pgf, scalars, clip, uvw, ray_level, interior_done);
}

// the rest of zero_moisture(il,ih,jl,jh) after launch_fused_advect on the box [3,NX-3) x [3,NY-3)
int launch_zero_moisture_shell(Ctx *c, int il, int ih, int jl, int jh) {
    if (c->prec == DYN_FP32) return shell_t<float>(c, il, ih, jl, jh);
    return shell_t<double>(c, il, ih, jl, jh);
}


// ---- ensemble launchers ----------------------------------------------------------------------------
namespace {
// packed rows in the ensemble's batches too (every member has the same level count; at most 8 rows of 64)
template <typename T, int TJ, bool PACK>
int ens_momentum_t(Ctx *c0, const EnsMember *d, int nmem, const EnsRoles &ro, T step, int tj, int ti, int total) {
    const dim3 blk = PACK ? dim3((tj * c0->geo.NZ + KP - 1) / KP * KP) : dim3(KP, TJ);
    Timed _t(c0, "ens_momentum", 0.0);
    hipLaunchKernelGGL((k_ens_momentum<T, TJ, false, PACK>), dim3(total), blk, MomLds<T>::bytes(tj, PACK ? c0->geo.NZ : KP), c0->stream,
                       d, nmem, ro, step, tj, ti, total);
    DYN_LAUNCH_CHECK();
    return DYN_OK;
}
template <typename T, int TJ, bool PACK>
int ens_scalars_t(Ctx *c0, const EnsMember *d, int nmem, const EnsRoles &ro, T step, int tj, int ti, int total) {
    const dim3 blk = PACK ? dim3((tj * c0->geo.NZ + KP - 1) / KP * KP) : dim3(KP, TJ);
    Timed _t(c0, "ens_scalars", 0.0);
    hipLaunchKernelGGL((k_ens_scalars<T, TJ, false, PACK>), dim3(total), blk, (scalar_lds<T, false>(tj, PACK ? c0->geo.NZ : KP)),
                       c0->stream, d, nmem, ro, step, tj, ti, total);
    DYN_LAUNCH_CHECK();
    return DYN_OK;
}
template <typename T, bool PACK>
int ens_stage_t(Ctx *c0, const EnsMember *d, int nmem, const EnsRoles &ro, double step, const int *shape, int tot_mom, int tot_scal) {
    int rc;
    if (shape[0] <= 2) rc = ens_momentum_t<T, 2, PACK>(c0, d, nmem, ro, T(step), shape[0], shape[1], tot_mom);
    else if (shape[0] <= 5) rc = ens_momentum_t<T, 4, PACK>(c0, d, nmem, ro, T(step), shape[0], shape[1], tot_mom);
    else rc = ens_momentum_t<T, 8, PACK>(c0, d, nmem, ro, T(step), shape[0], shape[1], tot_mom);
    if (rc) return rc;
    if (shape[2] <= 2) return ens_scalars_t<T, 2, PACK>(c0, d, nmem, ro, T(step), shape[2], shape[3], tot_scal);
    if (shape[2] <= 5) return ens_scalars_t<T, 4, PACK>(c0, d, nmem, ro, T(step), shape[2], shape[3], tot_scal);
    return ens_scalars_t<T, 8, PACK>(c0, d, nmem, ro, T(step), shape[2], shape[3], tot_scal);
}
template <typename T>
int ens_post_t(Ctx *c0, const EnsMember *d, int nmem, const EnsRoles &ro, double step, bool pgf, int total) {
    const int grid = total;
    Timed _t(c0, "ens_post", 0.0);
    hipLaunchKernelGGL(k_ens_post<T>, dim3(grid), dim3(KP, 4), 0, c0->stream, d, nmem, ro, T(step), pgf, true, total);
    DYN_LAUNCH_CHECK();
    return DYN_OK;
}
template <typename T>
int ens_copy_t(Ctx *c0, const EnsMember *d, int nmem, const EnsRoles &ro, int total) {
    const int grid = total;
    Timed _t(c0, "ens_advance_copy", 0.0);
    hipLaunchKernelGGL(k_ens_copy<T>, dim3(grid), dim3(256), 0, c0->stream, d, nmem, ro, total);
    DYN_LAUNCH_CHECK();
    return DYN_OK;
}
template <typename T, int TJ, bool PACK>
int ens_lds_limits() {
    int dev = 0, most = 0;
    DYN_HIP(hipGetDevice(&dev));
    DYN_HIP(hipDeviceGetAttribute(&most, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
    const void *k[] = {(const void *)k_ens_momentum<T, TJ, false, PACK>, (const void *)k_ens_scalars<T, TJ, false, PACK>};
    for (const void *f : k) DYN_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, most));
    return DYN_OK;
}
template <typename T>
int ens_lds_limits_all() {
    int rc = ens_lds_limits<T, 2, true>();
    if (!rc) rc = ens_lds_limits<T, 4, true>();
    if (!rc) rc = ens_lds_limits<T, 8, true>();
    if (!rc) rc = ens_lds_limits<T, 2, false>();
    if (!rc) rc = ens_lds_limits<T, 4, false>();
    if (!rc) rc = ens_lds_limits<T, 8, false>();
    return rc;
}
}  // namespace

int ens_prepare(bool fp32) { return fp32 ? ens_lds_limits_all<float>() : ens_lds_limits_all<double>(); }
// the stage advection of every member (one momentum and one scalar launch); shape = {mom TJ, mom TI, scal TJ, scal TI}
int launch_ens_stage(Ctx *c0, const EnsMember *d, int nmem, const EnsRoles &ro, double step, const int *shape, int tot_mom, int tot_scal) {
    if (stage_packs(c0))
        return c0->prec == DYN_FP32 ? ens_stage_t<float, true>(c0, d, nmem, ro, step, shape, tot_mom, tot_scal)
                                    : ens_stage_t<double, true>(c0, d, nmem, ro, step, shape, tot_mom, tot_scal);
    return c0->prec == DYN_FP32 ? ens_stage_t<float, false>(c0, d, nmem, ro, step, shape, tot_mom, tot_scal)
                                : ens_stage_t<double, false>(c0, d, nmem, ro, step, shape, tot_mom, tot_scal);
}
int launch_ens_post(Ctx *c0, const EnsMember *d, int nmem, const EnsRoles &ro, double step, bool pgf, int total) {
    return c0->prec == DYN_FP32 ? ens_post_t<float>(c0, d, nmem, ro, step, pgf, total) : ens_post_t<double>(c0, d, nmem, ro, step, pgf, total);
}
int launch_ens_copy(Ctx *c0, const EnsMember *d, int nmem, const EnsRoles &ro, int total) {
    return c0->prec == DYN_FP32 ? ens_copy_t<float>(c0, d, nmem, ro, total) : ens_copy_t<double>(c0, d, nmem, ro, total);
}

}  // namespace dyn
