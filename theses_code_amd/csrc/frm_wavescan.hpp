// Wavefront-level building blocks for tridiagonal (Thomas) sweeps.
//
// A line of n unknowns is split into 64 contiguous chunks of CM elements,
// one chunk per lane.  The Thomas forward and back-substitution recurrences
// are first-order affine maps, so each lane composes the maps of its chunk,
// a 6-level scan over the wavefront gives every lane the value
// entering its chunk, and the lane then replays the exact sequential Thomas
// formulas over its chunk (method: Stone 1973 recurrence scan; the in-chunk
// arithmetic is the reference's progonka, mt_minimal.cpp:942-1024).
#pragma once
#include <hip/hip_runtime.h>

namespace frm {

// Lane i's value of x moved by a DPP control (row_shr/row_shl within the rows of
// 16 lanes, row_bcast across them, wave_shr/wave_shl by one lane); lanes the
// control gives no source, and rows outside RMASK, take `old`.  A scan level
// through DPP is a few register moves, one through __shfl two LDS round trips.
template <int CTRL, int RMASK = 0xf>
__device__ __forceinline__ double dpp_move(double old, double x) {
    const int lo = __builtin_amdgcn_update_dpp(__double2loint(old), __double2loint(x), CTRL, RMASK, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(old), __double2hiint(x), CTRL, RMASK, 0xf, false);
    return __hiloint2double(hi, lo);
}
constexpr int kDppRowShr = 0x110, kDppRowShl = 0x100, kDppWaveShr1 = 0x138, kDppWaveShl1 = 0x130,
              kDppRowBcast15 = 0x142, kDppRowBcast31 = 0x143;

__device__ __forceinline__ double lane_value(double x, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), lane),
                            __builtin_amdgcn_readlane(__double2loint(x), lane));
}

// The same with 0 where there is no source (the control's own zero: no moves to
// set it up).
template <int CTRL>
__device__ __forceinline__ double dpp_zero(double x) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

// One scan level: (P, Q) after the map that the control brings (the identity
// where it brings none).
template <int CTRL, int RMASK = 0xf>
__device__ __forceinline__ void affine_level(double& P, double& Q) {
    const double Po = dpp_move<CTRL, RMASK>(1.0, P);
    double Qo;
    if constexpr (RMASK == 0xf) Qo = dpp_zero<CTRL>(Q);
    else Qo = dpp_move<CTRL, RMASK>(0.0, Q);
    Q = P * Qo + Q;
    P = P * Po;
}

// Exclusive composition of affine maps x -> P x + Q over lanes 0..lane-1
// (forward: earlier lanes first), and the whole wavefront's map (Pt, Qt).
__device__ inline void scan_affine_up_total(double& P, double& Q, int lane, double& Pt, double& Qt) {
    affine_level<kDppRowShr + 1>(P, Q);
    affine_level<kDppRowShr + 2>(P, Q);
    affine_level<kDppRowShr + 4>(P, Q);
    affine_level<kDppRowShr + 8>(P, Q);
    affine_level<kDppRowBcast15, 0xa>(P, Q);  // rows 1 and 3 after rows 0 and 2
    affine_level<kDppRowBcast31, 0xc>(P, Q);  // rows 2 and 3 after row 1
    Pt = lane_value(P, 63);
    Qt = lane_value(Q, 63);
    P = dpp_move<kDppWaveShr1>(1.0, P);
    Q = dpp_move<kDppWaveShr1>(0.0, Q);
}

// Exclusive composition over lanes lane+1..63 (backward: later lanes first),
// and the whole wavefront's map.
__device__ inline void scan_affine_down_total(double& P, double& Q, int lane, double& Pt,
                                              double& Qt) {
    affine_level<kDppRowShl + 1>(P, Q);
    affine_level<kDppRowShl + 2>(P, Q);
    affine_level<kDppRowShl + 4>(P, Q);
    affine_level<kDppRowShl + 8>(P, Q);
    // rows 0 and 2 after rows 1 and 3, then rows 0 and 1 after row 2 (DPP
    // broadcasts upwards only)
    {
        const double P1 = lane_value(P, 16), Q1 = lane_value(Q, 16);
        const double P3 = lane_value(P, 48), Q3 = lane_value(Q, 48);
        const double Po = lane < 32 ? P1 : P3, Qo = lane < 32 ? Q1 : Q3;
        if (!(lane & 16)) {
            Q = P * Qo + Q;
            P = P * Po;
        }
    }
    {
        const double Po = lane_value(P, 32), Qo = lane_value(Q, 32);
        if (lane < 32) {
            Q = P * Qo + Q;
            P = P * Po;
        }
    }
    Pt = lane_value(P, 0);
    Qt = lane_value(Q, 0);
    P = dpp_move<kDppWaveShl1>(1.0, P);
    Q = dpp_move<kDppWaveShl1>(0.0, Q);
}

__device__ inline void scan_affine_up(double& P, double& Q, int lane) {
    double Pt, Qt;
    scan_affine_up_total(P, Q, lane, Pt, Qt);
}

__device__ inline void scan_affine_down(double& P, double& Q, int lane) {
    double Pt, Qt;
    scan_affine_down_total(P, Q, lane, Pt, Qt);
}

// Scratch in LDS for one line that spans W wavefronts.
template <int W>
struct LineShare {
    double fP[W], fQ[W];  // forward wave totals
    double bP[W], bQ[W];  // backward wave totals
    double un;
};

// line_solve for a line spread over W wavefronts of one workgroup: lane
// `lane` of wavefront `wl` (0..W-1) owns elements e0 = (64 wl + lane) CM ..
// + CM - 1.  The wavefront totals meet in `sh`; every wavefront of the
// workgroup must call this (it contains workgroup barriers), `active`
// false for wavefronts without a line.
template <int CM, int W>
__device__ inline double line_solve_mw(const double (&a)[CM], const double (&f)[CM],
                                       const double (&al)[CM], double (&v)[CM], int e0, int n,
                                       double b0, int lane, int wl, LineShare<W>* sh, bool active,
                                       const double* un_fixed = nullptr) {
    return line_solve_mw(a, f, al, v, e0, n, b0, lane, wl, sh, active, un_fixed, [] {});
}

// mid() runs between the passes, where a and f are no longer needed: loads for
// after the solve can go out there into their registers.
template <int CM, int W, typename Mid>
__device__ inline double line_solve_mw(const double (&a)[CM], const double (&f)[CM],
                                       const double (&al)[CM], double (&v)[CM], int e0, int n,
                                       double b0, int lane, int wl, LineShare<W>* sh, bool active,
                                       const double* un_fixed, Mid mid) {
    // ---- forward
    double P = 1.0, Q = 0.0, Pt = 1.0, Qt = 0.0;
#pragma unroll
    for (int k = 0; k < CM; ++k) {
        if (e0 + k < n) {
            const double p = f[k] * a[k];
            const double q = -f[k] * v[k];
            Q = p * Q + q;
            P = p * P;
        }
    }
    if (active) {
        scan_affine_up_total(P, Q, lane, Pt, Qt);
        if (lane == 0) {
            sh->fP[wl] = Pt;
            sh->fQ[wl] = Qt;
        }
    }
    __syncthreads();
    double x = 0.0;
    if (active) {
        double y = b0;  // value entering this wavefront's part of the line
        for (int w = 0; w < wl; ++w) y = sh->fP[w] * y + sh->fQ[w];
        x = P * y + Q;
#pragma unroll
        for (int k = 0; k < CM; ++k) {
            if (e0 + k < n) {
                x = f[k] * (a[k] * x - v[k]);
                v[k] = x;
            }
        }
#pragma unroll
        for (int k = 0; k < CM; ++k)
            if (e0 + k == n - 1) sh->un = un_fixed ? *un_fixed : v[k] / (1.0 - al[k]);
    }
    mid();
    __syncthreads();
    const double un = active ? sh->un : 0.0;
    // ---- backward
    P = 1.0;
    Q = 0.0;
#pragma unroll
    for (int k = CM - 1; k >= 0; --k) {
        if (e0 + k < n) {
            Q = al[k] * Q + v[k];
            P = al[k] * P;
        }
    }
    if (active) {
        scan_affine_down_total(P, Q, lane, Pt, Qt);
        if (lane == 0) {
            sh->bP[wl] = Pt;
            sh->bQ[wl] = Qt;
        }
    }
    __syncthreads();
    if (active) {
        double y = un;  // value just above this wavefront's part of the line
        for (int w = W - 1; w > wl; --w) y = sh->bP[w] * y + sh->bQ[w];
        y = P * y + Q;
#pragma unroll
        for (int k = CM - 1; k >= 0; --k) {
            if (e0 + k < n) {
                y = al[k] * y + v[k];
                v[k] = y;
            }
        }
    }
    return un;
}

// Solve one line whose Thomas alpha coefficients are known.
//   forward : bt_e = f_e * (a_e * bt_{e-1} - om_e),  bt_{-1} = b0
//   backward: u_e  = al_e * u_{e+1} + bt_e,           u_n = bt_{n-1} / (1 - al_{n-1})
// (fr_d_t_g_2d.cpp:3494-3553 and 2548-2550 with f_e = Al[i+1]/B(i)).
// On entry v[] holds om for the lane's chunk; on exit it holds u.
// Returns u_n (the value at i = N) to every lane; with un_fixed the caller
// gives u_n (a Dirichlet end) instead.
template <int CM>
__device__ inline double line_solve(const double (&a)[CM], const double (&f)[CM],
                                    const double (&al)[CM], double (&v)[CM], int e0, int n,
                                    double b0, int lane, const double* un_fixed = nullptr) {
    // ---- forward: compose chunk maps x -> p x + q, p = f a, q = -f om
    double P = 1.0, Q = 0.0;
#pragma unroll
    for (int k = 0; k < CM; ++k) {
        if (e0 + k < n) {
            const double p = f[k] * a[k];
            const double q = -f[k] * v[k];
            Q = p * Q + q;
            P = p * P;
        }
    }
    scan_affine_up(P, Q, lane);
    double x = P * b0 + Q;  // bt entering the chunk
#pragma unroll
    for (int k = 0; k < CM; ++k) {
        if (e0 + k < n) {
            x = f[k] * (a[k] * x - v[k]);
            v[k] = x;  // v now holds bt
        }
    }
    // ---- u_n from the lane holding element n-1
    const int last = (n - 1) / CM;
    double un_local = 0.0;
#pragma unroll
    for (int k = 0; k < CM; ++k)
        if (e0 + k == n - 1) un_local = v[k] / (1.0 - al[k]);
    const double un = un_fixed ? *un_fixed : __shfl(un_local, last);
    // ---- backward: compose y -> al y + bt from the top of the chunk down
    P = 1.0;
    Q = 0.0;
#pragma unroll
    for (int k = CM - 1; k >= 0; --k) {
        if (e0 + k < n) {
            Q = al[k] * Q + v[k];
            P = al[k] * P;
        }
    }
    scan_affine_down(P, Q, lane);
    double y = P * un + Q;  // u just above the chunk
#pragma unroll
    for (int k = CM - 1; k >= 0; --k) {
        if (e0 + k < n) {
            y = al[k] * y + v[k];
            v[k] = y;  // v now holds u
        }
    }
    return un;
}

}  // namespace frm

namespace frm {

// 2x2 matrix [[m00, m01], [m10, m11]] acting on homogeneous (y, z); used for
// the Thomas alpha recurrence c'_k = c_k / (b_k - a_k c'_{k-1}), a Moebius
// map.  Products are rescaled by an exact power of two to stay in range.
struct Mob {
    double m00, m01, m10, m11;
};

__device__ inline Mob mob_scale(Mob r) {
    const double mx = fmax(fmax(fabs(r.m00), fabs(r.m01)), fmax(fabs(r.m10), fabs(r.m11)));
    if (mx > 0.0 && isfinite(mx)) {
        int ex;
        frexp(mx, &ex);
        r.m00 = ldexp(r.m00, -ex);
        r.m01 = ldexp(r.m01, -ex);
        r.m10 = ldexp(r.m10, -ex);
        r.m11 = ldexp(r.m11, -ex);
    }
    return r;
}

__device__ inline Mob mob_mul(const Mob& x, const Mob& y) {  // x * y (apply y first)
    Mob r;
    r.m00 = x.m00 * y.m00 + x.m01 * y.m10;
    r.m01 = x.m00 * y.m01 + x.m01 * y.m11;
    r.m10 = x.m10 * y.m00 + x.m11 * y.m10;
    r.m11 = x.m10 * y.m01 + x.m11 * y.m11;
    return r;
}

template <int CTRL, int RMASK = 0xf>
__device__ __forceinline__ Mob dpp_mob(const Mob& m) {  // the identity where there is no source
    return Mob{dpp_move<CTRL, RMASK>(1.0, m.m00), dpp_move<CTRL, RMASK>(0.0, m.m01),
               dpp_move<CTRL, RMASK>(0.0, m.m10), dpp_move<CTRL, RMASK>(1.0, m.m11)};
}

template <int CTRL, int RMASK, bool SCALE>
__device__ __forceinline__ void mob_level(Mob& m) {
    m = mob_mul(m, dpp_mob<CTRL, RMASK>(m));
    if (SCALE) m = mob_scale(m);
}

// Exclusive forward scan of Moebius maps (earlier lanes applied first), and the
// whole wavefront's map.  The maps come scaled (mob_scale).  SCALE: rescaled on
// every level, for any matrix; without, once at the end: for rows with diagonal
// R > A + B >= 0, whose elimination divides by at least about R/2, 64 scaled
// maps stay far inside the range.
template <bool SCALE>
__device__ inline Mob scan_mob_up_total(Mob m, int lane, Mob& tot) {
    mob_level<kDppRowShr + 1, 0xf, SCALE>(m);
    mob_level<kDppRowShr + 2, 0xf, SCALE>(m);
    mob_level<kDppRowShr + 4, 0xf, SCALE>(m);
    mob_level<kDppRowShr + 8, 0xf, SCALE>(m);
    mob_level<kDppRowBcast15, 0xa, SCALE>(m);
    mob_level<kDppRowBcast31, 0xc, true>(m);
    tot = Mob{lane_value(m.m00, 63), lane_value(m.m01, 63), lane_value(m.m10, 63),
              lane_value(m.m11, 63)};
    return dpp_mob<kDppWaveShr1>(m);
}

__device__ inline Mob scan_mob_up(const Mob& m, int lane) {
    Mob tot;
    return scan_mob_up_total<true>(m, lane, tot);
}

}  // namespace frm
