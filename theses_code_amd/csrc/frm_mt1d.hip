// Batched 1D time-fractional moisture solver: the hot path of
// H_solver::calc_step of mt_minimal.cpp (Caputo L1 weights) and
// mt_psi_caputo.cpp (psi-Caputo weights, psi(t) = t^beta), gamma = 1.
//
// The reference steps one problem at a time on the CPU: coefficient calls
// per node (al1 829-858, bt1 942-980), the history loop of Om1 (906-939 /
// 1315-1342) over heap snapshots, the progonka back-substitution (1021-1022)
// and, for psi, a full rebuild of kb_time with series integrals every step
// (mt_psi_caputo.cpp:1481-1489).  Here a whole batch of problems of uneven
// size advances together, a block of kHistBlock steps at a time:
//   1. (psi only) weights of the block's steps, which do not depend on the
//      state: one lane per (problem, interval, step), FP64 series, formed on
//      a second stream while the block before runs;
//   2. far sums: the history of the block's steps up to its start, one pass
//      over the stored increments for all of them (FP64 matrix cores);
//   3. steps: one wavefront per problem runs the block's steps one after
//      another -- the block's own increments, coefficients from the current
//      iterate (held in LDS), Thomas alpha/beta/back-substitution with
//      wavefront-scan chunk seeds, boundary rules, Picard iterations, and the
//      push of the new increment.  Problems are independent, so nothing else
//      has to be waited for between steps.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <tuple>
#include <type_traits>
#include <vector>

#include "frm_blockhist.hpp"
#include "frm_diag.h"
#include "frm_history.hpp"
#include "frm_wavescan.hpp"
#include "frm_weights.hpp"

namespace frm {

constexpr int kGroup = 128;       // nodes per memory-term wavefront
// The step kernels run a problem on up to kMtMaxW wavefronts of one workgroup,
// kMtCM unknowns per lane (N - 1 <= 1024).  Measured per step at 4 / 8 / 16
// unknowns per lane: 4096 uneven psi problems 84 / 81 / 97 us, 1024 AB problems
// 11.3 / 11.6 us, one 200-node problem 2.8 / 3.7 us; one wavefront per problem
// of up to 16 per lane ran the psi problems in 215 us and spilled.
constexpr int kMtCM = 4;
constexpr int kMtMaxW = 4;
constexpr int kMtMaxN = 64 * kMtCM * kMtMaxW + 1;

struct MtProbDev {
    int N, form, top, bottom_cond, src;
    int64_t uoff, hoff;
    double dL, Dg, Da, alpha, beta, D, k, k0, b, top_val, Ev, Hbottom;
    // kind AB with the series history: series length, offsets of the
    // problem's per-step coefficient rows and phase choices
    int ser, ser_maxl;
    int64_t ser_off, ser_coff;
};

// ---------------------------------------------------------------- physics
// KK(i) and inv_dw_dh(i) of H_solver at state value x (mt_minimal.cpp:481-562
// for cv_form 2 and k_form 0; CONST and KEXP are this build's forms).
__device__ inline double mt_KK(const MtProbDev& P, double x) {
    if (P.form == FRM_FORM_CV2) return 1.0 * P.k;
    if (P.form == FRM_FORM_KEXP) return P.k0 * exp(P.b * x);
    return P.D;
}
__device__ inline double mt_inv(const MtProbDev& P, double x) {
    if (P.form != FRM_FORM_CV2) return 1.0;
    const double Pr = -x;
    double Ch = 0.0;
    if (Pr >= 10) Ch = 0.05;
    if ((Pr < 10) && (Pr >= 0.0)) Ch = 0.5 - Pr * (0.5 - 0.05) / 10.0;
    return Ch != 0.0 ? 1.0 / Ch : 1e20;
}

// ---------------------------------------------------------------- far sums
// G[j*ldh + i] = sum_{s < N0} w(N0 + j, s) Delta_s[i], j < J = kHistBlock, for
// the node i of its problem p: the settled part of the history sums of the J
// steps N0 .. N0 + J - 1 (history index: the number of increments before the
// step).  One FP64 product per problem on v_mfma_f64_16x16x4_f64: the J steps
// are its 16 rows, 16 NC nodes a wavefront's columns, four slots per
// instruction (A[l%16][l/16] = w(N0 + l%16, s0 + l/16), B[l/16][l%16] =
// Delta_{s0 + l/16}, D row 4 r + l/16).  The history is read once per J steps
// instead of every step: 223 -> 16 us per step on 1024 uneven FP64 problems at
// 300 slots, 302 -> 29 us on 4096 psi problems with FP32 increments at 200.
//
// Weights: lag-indexed per problem (w[p*ldw + lag - 1]), or (TAB) the psi
// table w[(p*ldw + s)*J + j], whose four slots x 16 steps are one contiguous
// load per instruction.  gprob/gvalid give each 128-node group's problem (-1:
// none) and its count of real nodes; tiles past it are skipped, and a partial
// tile's lanes repeat its last nodes, so the stream carries the problems' own
// nodes only.  SPLIT: the wavefronts of a workgroup share a tile's slots and
// add their sums through LDS in wavefront order, for batches with too few
// tiles to fill the chip.
typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr int kFarSplit = 16;  // wavefronts that share a tile at most

template <typename HT, bool TAB, bool SPLIT>
__global__ __launch_bounds__(SPLIT ? 64 * kFarSplit : 256) void k_mt_far(
    const HT* __restrict__ hist, int64_t ldh, int N0, const double* __restrict__ w, int ldw,
    const int* __restrict__ gprob, const int* __restrict__ gvalid, double* __restrict__ G) {
    constexpr int NC = SPLIT ? 1 : 4;  // one node per lane, or four in 16-byte loads
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int m = lane & 15, kg = lane >> 4;
    const int64_t i0 = (SPLIT ? (int64_t)blockIdx.x : (int64_t)blockIdx.x * 4 + wv) * (16 * NC);
    if (i0 >= ldh) return;
    const int64_t grp = i0 / kGroup;
    const int p = __builtin_amdgcn_readfirstlane(gprob[grp]);
    const int left = __builtin_amdgcn_readfirstlane(gvalid[grp]) - (int)(i0 % kGroup);
    if (p < 0 || left <= 0) return;  // SPLIT: the same for the whole workgroup
    int a = 0, b = N0;
    if constexpr (SPLIT) {
        const int ks = blockDim.x >> 6, per = (N0 / 4 + ks - 1) / ks * 4;
        a = min(N0, wv * per);
        b = min(N0, a + per);
    }
    // the lane's nodes of column tile c: NC == 1: m; four FP32: 4 m + c; four
    // FP64: 32 (c / 2) + 2 m + c % 2
    typedef HT v2 __attribute__((ext_vector_type(2)));
    typedef HT v4 __attribute__((ext_vector_type(4)));
    auto nodes = [&](const HT* q, double (&x)[NC]) {
        if constexpr (NC == 1) {
            x[0] = (double)__builtin_nontemporal_load(q + min(m, left - 1));
        } else if constexpr (sizeof(HT) == 4) {
            const v4 v = __builtin_nontemporal_load(
                reinterpret_cast<const v4*>(q + min(4 * m, (left - 1) & ~3)));
#pragma unroll
            for (int c = 0; c < 4; ++c) x[c] = (double)v[c];
        } else {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const v2 v = __builtin_nontemporal_load(
                    reinterpret_cast<const v2*>(q + min(32 * h + 2 * m, (left - 1) & ~1)));
                x[2 * h] = (double)v.x;
                x[2 * h + 1] = (double)v.y;
            }
        }
    };
    f64x4 acc[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[c] = f64x4{0.0, 0.0, 0.0, 0.0};
    const HT* hp = hist + (int64_t)(a + kg) * ldh + i0;
    const double* wp = TAB ? w + ((int64_t)p * ldw + a) * kHistBlock + lane % 16 + 16 * kg
                           : w + (int64_t)p * ldw + (N0 - a - 1 + m - kg);
    constexpr int ws = TAB ? 4 * kHistBlock : -4;  // weight stride of four slots
    constexpr int U = NC == 1 ? 8 : 4;             // products whose loads go out together
    int s = a;
    for (; s + 4 * U <= b; s += 4 * U) {
        double x[U][NC], v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            nodes(hp + (int64_t)(4 * u) * ldh, x[u]);
            v[u] = wp[ws * u];
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int c = 0; c < NC; ++c)
                acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(v[u], x[u][c], acc[c], 0, 0, 0);
        hp += (int64_t)(4 * U) * ldh;
        wp += ws * U;
    }
    for (; s < b; s += 4) {
        double x[NC];
        nodes(hp, x);
        const double v = wp[0];
#pragma unroll
        for (int c = 0; c < NC; ++c)
            acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(v, x[c], acc[c], 0, 0, 0);
        hp += 4 * ldh;
        wp += ws;
    }
    auto node = [&](int c) {
        return NC == 1 ? m : sizeof(HT) == 4 ? 4 * m + c : 32 * (c >> 1) + 2 * m + (c & 1);
    };
    if constexpr (!SPLIT) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int c = 0; c < NC; ++c)
                if (node(c) < left) G[(int64_t)(4 * r + kg) * ldh + i0 + node(c)] = acc[c][r];
    } else {
        __shared__ double part[kFarSplit][4][64];
        const int ks = blockDim.x >> 6;
#pragma unroll
        for (int r = 0; r < 4; ++r) part[wv][r][lane] = acc[0][r];
        __syncthreads();
        for (int r = wv; r < 4; r += ks) {
            double v = 0.0;
            for (int k = 0; k < ks; ++k) v += part[k][r][lane];
            if (m < left) G[(int64_t)(4 * r + kg) * ldh + i0 + m] = v;
        }
    }
}

// A value that is the same on every lane, as the compiler can know it: it then
// lives in scalar registers and its uses as an address are scalar.
template <typename T>
__device__ __forceinline__ T same_on_lanes(const T& v) {
    static_assert(sizeof(T) % 4 == 0, "whole words");
    union U {
        T t;
        int w[sizeof(T) / 4];
        __device__ U() {}
    } u;
    u.t = v;
#pragma unroll
    for (size_t i = 0; i < sizeof(T) / 4; ++i) u.w[i] = __builtin_amdgcn_readfirstlane(u.w[i]);
    return u.t;
}

// Read-only data (written by earlier launches) at addresses that are the same
// on every lane: scalar loads.
typedef const __attribute__((address_space(4))) double* const_doubles;
__device__ __forceinline__ const_doubles scalar_ptr(const double* p) { return (const_doubles)p; }

// A problem's history sums of kMtSub steps at a time.  The far sums and the
// block's slots so far are read once per kMtSub steps, for all of them; each
// step then adds its own increment, which is in registers, to the sums of the
// steps left.  Read anew for every step, the slots cost up to six trips to
// the cache per step, a third of a step on one 200-node problem (44 -> 39 us per
// 16 steps; 1024 AB problems 178 -> 124, 4096 psi problems 1260 -> 1200).
constexpr int kMtSub = 4;

// acc[t][r], t < T: the sums of the step with history index n + t, in a block
// that starts at N0, over the far sums G (null: none) and the slots
// N0 .. n - 1, oldest first, for the elements e = r*nl + g < len (lanes past
// len repeat the last one).  w[(n-1-s) ws + t]: slot s's weight at step n + t.
template <typename HT, int CM>
__device__ __forceinline__ void mt_fill(const HT* hist, int64_t ldh, int64_t hoff, int len, int N0,
                                        int n, int T, const double* G, const double* w, int ws,
                                        int g, int nl, double (&acc)[kMtSub][CM]) {
    const const_doubles wc = scalar_ptr(w);
    int e[CM];
#pragma unroll
    for (int r = 0; r < CM; ++r) e[r] = min(r * nl + g, len - 1);
#pragma unroll
    for (int t = 0; t < kMtSub; ++t) {
#pragma unroll
        for (int r = 0; r < CM; ++r)
            acc[t][r] = G && t < T ? G[(int64_t)(n + t - N0) * ldh + hoff + e[r]] : 0.0;
    }
    constexpr int U = CM >= 16 ? 1 : 16 / CM;  // slots whose loads go out together
    const HT* h = hist + hoff;
    for (int s = N0; s < n; s += U) {
        HT x[U][CM];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int r = 0; r < CM; ++r) x[u][r] = h[(int64_t)min(s + u, n - 1) * ldh + e[r]];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (s + u >= n) break;
#pragma unroll
            for (int t = 0; t < kMtSub; ++t) {
                if (t >= T) break;
                const double v = wc[(n - 1 - s - u) * ws + t];
#pragma unroll
                for (int r = 0; r < CM; ++r) acc[t][r] = fma(v, (double)x[u][r], acc[t][r]);
            }
        }
    }
}

// After the step with history index n, left steps of its kMtSub to go: its
// increment d (as stored) joins their sums, and the next step's become acc[0].
template <int CM>
__device__ __forceinline__ void mt_push(int left, const double* w, int ws, const double (&d)[CM],
                                        double (&acc)[kMtSub][CM]) {
    const const_doubles wc = scalar_ptr(w);
#pragma unroll
    for (int t = 1; t < kMtSub; ++t) {
        if (t > left) break;
        const double v = wc[t - ws];
#pragma unroll
        for (int r = 0; r < CM; ++r) acc[t - 1][r] = fma(v, d[r], acc[t][r]);
    }
}

// ---------------------------------------------------------------- psi weights
// calc_int(alpha, a, a+1, A, tau, 1) of mt_psi_caputo.cpp:720-740 for
// g(t) = t^beta: Taylor series around g(tj) (_kb_row, 497-566) or, for
// intervals in the first half (t1 <= A/2), Newton binomial in g(tj) times the
// Taylor series of the inverse's derivative around g(t1) (_kb_row2,
// 567-719); both stop at term size global_eps = 1e-5 as the reference does.
// The reference caches the inner integrals of _kb_row2 per interval; they
// depend only on the interval, so recomputing them gives the same values.
constexpr double kPsiEps = 1e-5;
constexpr int kPsiMaxIt = 100000;

__device__ inline double psi_inv_der(double beta, double t, int n, double d) {
    if (n == 0) return pow(t, 1.0 / beta);
    if (n == 1) return ((1.0 / beta) * pow(t, (1.0 / beta) - 1)) * (d / pow(t, 1.0 / beta));
    return d * ((1.0 / beta) - n + 1) / t;
}

// Reciprocals of whole numbers and of i + 1 - alpha, which the series' terms
// divide by: a division costs about as much as the rest of a term, and a
// workgroup's weights are all of one problem.  4096 problems, 400 steps: 12.0
// -> 10.2 ms with them; against extended precision the series' error stays the same
// (median 1.8e-16 below half the past, 1.1e-14 above).
constexpr int kPsiRecip = 128;
struct PsiRecip {
    double n[kPsiRecip];   // 1 / i, i >= 1
    double na[kPsiRecip];  // 1 / (i + 1 - alpha)
    __device__ double by_n(int i) const { return i < kPsiRecip ? n[i] : 1.0 / i; }
    __device__ double by_na(int i, double alpha) const {
        return i < kPsiRecip ? na[i] : 1.0 / (i - alpha + 1.0);
    }
};

// v_first = f'(gtj) gtj^(1-alpha), the series' first factor (the same for
// every interval of a step)
__device__ double psi_kb_row(double beta, double gt0, double gt1, double gtj, double alpha,
                             double v_first, const PsiRecip& rc) {
    double sum = 0.0;
    int i = 0;
    double v = v_first;
    // term i: the reference forms f^(i+1)(gtj) = f^(i)(gtj) (1/beta - i)/gtj
    // and multiplies by -gtj/i; gtj cancels (the terms agree with the
    // reference's to rounding)
    const double q1 = fabs(1.0 - gt1 / gtj), q0 = fabs(1.0 - gt0 / gtj), ib = 1.0 / beta;
    double v3 = pow(q1, 1 - alpha);
    double v4 = pow(q0, 1 - alpha);
    double v2 = -(v3 - v4) / (1 - alpha);
    sum += v2 * v;
    while (fabs(v * v2) > kPsiEps) {
        ++i;
        v *= (i - ib) * rc.by_n(i);
        v3 *= q1;
        v4 *= q0;
        v2 = -(v3 - v4) * rc.by_na(i, alpha);
        sum += v2 * v;
        if (i > kPsiMaxIt) break;
        if (!isfinite(sum)) break;
    }
    return sum;
}

// gtj_na = gtj^-alpha (the same for every interval of a step); v4_first: the
// first derivative of the inverse at g(t1), which starts every term's inner
// series (the same in every step)
__device__ double psi_kb_row2(double beta, double t0, double t1, double gt0, double gt1, double gtj,
                              double alpha, double gtj_na, double v4_first, const PsiRecip& rc) {
    double sum = 0.0, v1 = 1.0, v2, v3, v4, v5, v6, v7;
    int niter = 0, i = 0, m;
    v2 = gtj_na * gt1;
    v6 = gt0 / gt1;
    const double ib = 1.0 / beta, igt1 = 1.0 / gt1, rg = (gt0 - gt1) / gt1;
    const double r2 = gt1 / gtj, r6 = gt0 / gt1;
    do {
        if (i != 0) {
            v1 *= -(-alpha - i + 1.0) * rc.by_n(i);
            v2 *= r2;
            v6 *= r6;
        }
        if (i == 0) {
            v3 = (t1 - t0) / gt1;
        } else {
            v3 = 0.0;
            m = 0;
            v4 = v4_first;
            v5 = rc.by_n(i + 1) * (1.0 - v6);
            v3 += v4 * v5;
            v7 = 1;
            // inner term m: the reference forms f^(m+1)(gt1) / m / ((i+m+1) /
            // (gt1 m)) and v7 (gt0-gt1) ((m-1)/m) ((i+m)/(gt1 (m-1))); gt1, m
            // and m-1 cancel
            while (fabs(v4 * v5) > (fabs(v3) * kPsiEps)) {
                ++m;
                v4 *= (ib - m) * rc.by_n(i + m + 1);
                if (m == 1)
                    v7 = igt1 * (v6 * (gt0 - gt1));
                else
                    v7 *= rg * (i + m) * rc.by_n(m);
                v5 = -(v5 + v7);
                v3 += v4 * v5;
                if (++niter > kPsiMaxIt) break;
                if (!isfinite(v3)) break;
            }
        }
        sum += v1 * v2 * v3;
        ++i;
        if (++niter > kPsiMaxIt) break;
        if (!isfinite(sum)) break;
    } while (fabs(v1 * v2 * v3) > kPsiEps);
    return sum;
}

// The factors of calc_int that depend only on the target g(A tau) of the
// step, formed once per problem and step: gtj, f'(gtj) gtj^(1-alpha) and
// gtj^-alpha (the same pow calls the per-interval series would make).
struct PsiStep {
    double gtj, v_first, gtj_na;
};

__device__ inline PsiStep psi_step(double alpha, double beta, int A, double tau) {
    PsiStep q;
    q.gtj = pow(A * tau, beta);
    double v = psi_inv_der(beta, q.gtj, 1, psi_inv_der(beta, q.gtj, 0, 1));
    v *= pow(q.gtj, 1 - alpha);
    q.v_first = v;
    q.gtj_na = pow(q.gtj, -alpha);
    return q;
}

// g(a tau) and the inverse's first derivative there, per problem, a = 0 ..
// gl - 1: the series' factors that depend on the interval only (five of the
// up to nine pow calls of a weight), made once per solver.
__global__ __launch_bounds__(256) void k_psi_tables(const MtProbDev* __restrict__ pr, int gl,
                                                    double tau, double* __restrict__ g,
                                                    double* __restrict__ dg) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= gl) return;
    const double beta = pr[blockIdx.y].beta;
    const double gt = pow(a * tau, beta);
    g[(int64_t)blockIdx.y * gl + a] = gt;
    dg[(int64_t)blockIdx.y * gl + a] = psi_inv_der(beta, gt, 1, psi_inv_der(beta, gt, 0, 0));
}

// g, dg: the problem's rows of k_psi_tables
__device__ double psi_calc_int(double alpha, double beta, int a, int A, double tau,
                               const double* __restrict__ g, const double* __restrict__ dg,
                               const PsiStep& q, const PsiRecip& rc) {
    if ((a + 1 <= 0.5 * A) && !(beta == 1))
        return psi_kb_row2(beta, a * tau, (a + 1) * tau, g[a], g[a + 1], q.gtj, alpha, q.gtj_na,
                           dg[a + 1], rc);
    return psi_kb_row(beta, g[a], g[a + 1], q.gtj, alpha, q.v_first, rc);
}

// The reference's fallback where a series is not finite: _kb(1, t0, t1,
// gtj, sing, alpha) (mt_psi_caputo.cpp:476-494), the integral of
// (gtj - g(t))^-alpha over [t0, t1] by midpoint rules on 1 and 2 panels,
// halving the interval while they differ by more than global_eps; below
// global_eps in width the two rules' mean, or on the interval that ends at
// the target (sing) the adaptive 3/8-rule march of ___kb (447-473).  The
// recursion runs on an explicit stack of frames, left half first, each
// interval's value the sum of its halves' as in the reference.  Returns NaN
// if the subdivision would pass kPsiQuadDepth levels or the march
// kPsiQuadMaxIt steps (the reference has no such bounds; widths below
// global_eps end the subdivision after log2(width / 1e-5) levels).
constexpr int kPsiQuadDepth = 48;
constexpr int kPsiQuadMaxIt = 1 << 20;

__device__ inline double psi_kb_mid(double beta, int n, double t0, double t1, double gtj,
                                    double alpha) {
#pragma clang fp contract(off)
    double ret = 0.0;
    const double step = (t1 - t0) / n;
    for (int i = 0; i < n; i++) ret += step * pow(gtj - pow(t0 + (i + 0.5) * step, beta), -alpha);
    return ret;
}

__device__ double psi_kb_sing(double beta, int n, double t0, double t1, double gtj, double alpha) {
#pragma clang fp contract(off)
    double f = pow(gtj - pow(t0, beta), -alpha), f1, f2, f3, f4;
    double sum = 0.0, v, t = t0, step = (t1 - t0) / n;
    int it = 0;
    do {
        f1 = pow(gtj - pow(t + 0.5 * step, beta), -alpha);
        f3 = pow(gtj - pow(t + step / 3.0, beta), -alpha);
        f4 = pow(gtj - pow(t + 2.0 * step / 3.0, beta), -alpha);
        f2 = pow(gtj - pow(t + step, beta), -alpha);
        v = (f + 3 * f3 + 3 * f4 + f2) * step / 8.0;
        if (!isfinite(v)) break;
        sum += v;
        t += step;
        if ((f1 / f) < (f2 / f1)) step /= (f2 / f1) / (f1 / f);
        // a finite step reaches 0 within 1100 halvings; an infinite one
        // (t1 - t0 overflowing) is cut off here
        for (int hv = 0; (t + step) > t1; ++hv) {
            if (hv > 1100) return NAN;
            step /= 2.0;
        }
        f = f2;
        if (++it > kPsiQuadMaxIt) return NAN;
    } while ((t1 - t) > kPsiEps * kPsiEps * kPsiEps);
    return sum;
}

__device__ double psi_kb_quad(double beta, double t0, double t1, double gtj, bool sing,
                              double alpha) {
#pragma clang fp contract(off)
    struct Frame {
        double t0, t1, left;
        int phase;  // 0: not yet evaluated, 1: left half pending, 2: right half pending
    };
    Frame fr[kPsiQuadDepth];
    int sp = 0;
    fr[0] = {t0, t1, 0.0, 0};
    double ret = 0.0;
    for (;;) {
        Frame& F = fr[sp];
        if (F.phase == 0) {
            const double v1 = psi_kb_mid(beta, 1, F.t0, F.t1, gtj, alpha);
            const double v2 = psi_kb_mid(beta, 2, F.t0, F.t1, gtj, alpha);
            if ((F.t1 - F.t0) < kPsiEps) {
                ret = sing ? psi_kb_sing(beta, 16, F.t0, F.t1, gtj, alpha) : 0.5 * (v1 + v2);
            } else if (fabs(v2 - v1) > kPsiEps) {
                if (sp + 1 >= kPsiQuadDepth) return NAN;
                F.phase = 1;
                fr[sp + 1] = {F.t0, 0.5 * (F.t0 + F.t1), 0.0, 0};
                ++sp;
                continue;
            } else {
                ret = v2;
            }
        } else if (F.phase == 1) {  // the left half's value arrived
            F.left = ret;
            F.phase = 2;
            fr[sp + 1] = {0.5 * (F.t0 + F.t1), F.t1, 0.0, 0};
            ++sp;
            continue;
        } else {  // the right half's value arrived
            ret = F.left + ret;
        }
        if (sp == 0) return ret;
        --sp;
    }
}

// The weights of a block of steps (kind psi).  Step j of the block that starts
// at history index N0 is k = N0 + j + 3; its weight of slot s < N0 + j is
// (1-alpha) kb_time of interval s + 1, stored at w[(p*ldw + s)*kHistBlock + j],
// and its current-step factor Da (1-alpha) kb_time[k] at d0[(j + 2)*nprob + p]
// (j = -2, -1: the two steps before the first increment is stored).
struct PsiArgs {
    const MtProbDev* pr;
    int nprob, N0, capacity;
    double tau;
    const double *g, *dg;  // k_psi_tables
    int gl;
    double* w;
    int ldw;
    double* d0;
    int* bad;
    int2* queue;           // (problem, slot * 32 + j, or -(j + 3) for a current-step factor)
    int qcap;
    int* qcount;           // [2] queue lengths, by the block's parity
};

__device__ inline void psi_store(const PsiArgs& a, const MtProbDev& P, int p, int s, int j,
                                 double v) {
    if (s >= 0)
        a.w[((int64_t)p * a.ldw + s) * kHistBlock + j] = v * (1 - P.alpha);
    else
        a.d0[(int64_t)(j + 2) * a.nprob + p] = P.Da * v * (1 - P.alpha);
}

// One workgroup: 16 slots x the block's 16 steps of one problem (grid row), a
// lane per weight with the steps fastest, so that its stores are contiguous;
// the last workgroup of a row: the current-step factors.
__global__ __launch_bounds__(256) void k_psi_weights(PsiArgs a) {
    constexpr int J = kHistBlock;
    const int p = blockIdx.y;
    const MtProbDev P = a.pr[p];
    const bool cur = blockIdx.x == gridDim.x - 1;
    __shared__ PsiStep q[J + 2];
    __shared__ PsiRecip rc;
    if (threadIdx.x < kPsiRecip)
        rc.n[threadIdx.x] = 1.0 / (int)threadIdx.x;  // entry 0 is never read
    else
        rc.na[threadIdx.x - kPsiRecip] = 1.0 / ((int)threadIdx.x - kPsiRecip - P.alpha + 1.0);
    const int j0 = cur && a.N0 == 0 ? -2 : 0;
    if (threadIdx.x < J - j0)
        q[threadIdx.x] = psi_step(P.alpha, P.beta, a.N0 + j0 + (int)threadIdx.x + 4, a.tau);
    __syncthreads();
    int s = -1, j, k;
    if (cur) {
        j = j0 + (int)threadIdx.x;
        k = a.N0 + j + 3;
        if (j >= J || k > a.capacity) return;
    } else {
        s = blockIdx.x * 16 + threadIdx.x / J;
        j = threadIdx.x % J;
        k = a.N0 + j + 3;
        if (s >= a.N0 + j || k > a.capacity) return;
    }
    const double* g = a.g + (int64_t)p * a.gl;
    const double* dg = a.dg + (int64_t)p * a.gl;
    const double v = psi_calc_int(P.alpha, P.beta, cur ? k : s + 1, k + 1, a.tau, g, dg, q[j - j0], rc);
    if (!isfinite(v)) {
        // calc_int falls back to _kb here: k_psi_quad computes and stores it
        const int slot = atomicAdd(&a.qcount[(a.N0 / J) & 1], 1);
        if (slot < a.qcap)
            a.queue[slot] = make_int2(p, cur ? -(j + 3) : s * 32 + j);
        else
            atomicOr(a.bad, 4);
        return;
    }
    psi_store(a, P, p, s, j, v);
}

// One thread per queued weight whose series was not finite: calc_int's _kb
// fallback, stored as k_psi_weights stores a weight.  A value that is still
// not finite sets bad bit 1.  Workgroup 0 clears the queue length that the
// next block appends to (the last reader of that one, the block before's
// k_psi_quad, has finished).
__global__ __launch_bounds__(64) void k_psi_quad(PsiArgs a) {
    const int par = (a.N0 / kHistBlock) & 1;
    const int nq = min(a.qcount[par], a.qcap);
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t == 0) a.qcount[par ^ 1] = 0;
    for (int q = t; q < nq; q += gridDim.x * blockDim.x) {
        const int2 e = a.queue[q];
        const MtProbDev P = a.pr[e.x];
        const int s = e.y < 0 ? -1 : e.y >> 5, j = e.y < 0 ? -e.y - 3 : e.y & 31;
        const int k = a.N0 + j + 3, i = s < 0 ? k : s + 1;
        const double gtj = pow((k + 1) * a.tau, P.beta);
        const double v = psi_kb_quad(P.beta, i * a.tau, (i + 1) * a.tau, gtj, i == k, P.alpha);
        if (!isfinite(v)) atomicOr(a.bad, 1);
        psi_store(a, P, e.x, s, j, v);
    }
}

__global__ void k_diag_psi_kb_quad(const double* __restrict__ c, int n, double* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double* r = c + 6 * (int64_t)i;
    out[i] = psi_kb_quad(r[1], r[2], r[3], r[4], r[5] != 0.0, r[0]);
}

// ---------------------------------------------------------------- steps
struct MtStepArgs {
    const MtProbDev* pr;
    const int* order;  // problems, largest first
    double* U;
    void* hist;
    int64_t ldh;
    const double* G;   // the block's far sums (null: no settled slots)
    const double* w;   // weights, as k_mt_far takes them
    int ldw;
    const double* d0;  // per problem, or (kind psi, TAB) the block's table
    int nprob;
    int N0;            // the block's start (history index)
    int k0, ks;        // steps k0 .. k0 + ks - 1, all of one block
    int picard;
};

// A problem's line lies in LDS with one pad double per chunk of CM elements
// (element e at e + e/CM): lanes reading their chunks, and lanes reading
// consecutive elements, both spread over the banks.
template <int CM>
__device__ __forceinline__ int pad_at(int e) {
    return e + e / CM;
}

// What the wavefronts of a problem tell each other.
struct MtShare {
    double Kf[kMtMaxW], Ke[kMtMaxW];  // first and last conductivity of a wavefront
    Mob m[kMtMaxW];                   // alpha maps
    double fP[kMtMaxW], fQ[kMtMaxW], bP[kMtMaxW], bQ[kMtMaxW];  // beta and back maps
    double un, x0;
    double es[kMtMaxW];               // kind AB: squared errors
};

// Runs steps a.k0 .. a.k0 + a.ks - 1 of problem p on W wavefronts of one
// workgroup (64 W CM >= its unknowns).  State, history sums and increments are
// handled in element order (consecutive lanes, consecutive nodes), the Thomas
// recurrences in chunk order (CM consecutive elements per lane); X holds the
// current iterate's interior nodes, Y the Picard-independent part of the
// right-hand side.  The conductivity is evaluated once per node and exchanged
// with the neighbouring lane; a constant matrix (FORM_CONST, L1) is factored
// once per launch.
template <int CM, typename HT, bool TAB>
__device__ __forceinline__ void mt_steps(const MtStepArgs& a, int p, int W, double* X, double* Y,
                                         MtShare& sh) {
    const int lane = threadIdx.x & 63, wl = same_on_lanes((int)(threadIdx.x >> 6));
    const MtProbDev P = same_on_lanes(a.pr[p]);
    const int N = P.N, n = N - 1;
    const int g = threadIdx.x, nl = 64 * W, e0 = g * CM, last = (n - 1) / CM;
    double* Ug = a.U + P.uoff;
    HT* hist = static_cast<HT*>(a.hist);
    double u[CM];
#pragma unroll
    for (int r = 0; r < CM; ++r) u[r] = Ug[min(r * nl + g, n - 1) + 1];
    double xN = Ug[N];
    if (g == 0) sh.x0 = Ug[0];
#pragma unroll
    for (int r = 0; r < CM; ++r)
        if (r * nl + g < n) X[pad_at<CM>(r * nl + g)] = u[r];
    const bool fixed = P.form == FRM_FORM_CONST && !TAB;
    bool factored = false;
    const double idL = 1.0 / P.dL;
    double A[CM], f[CM], al[CM];
    if constexpr (!TAB) {
#pragma unroll
        for (int k = 0; k < CM; ++k) A[k] = f[k] = al[k] = 0.0;
    }
    double acc[kMtSub][CM];  // history sums of this step and those left of its kMtSub
    for (int st = 0; st < a.ks; ++st) {
        const int step = a.k0 + st, h = step - 3;  // history index: slot h is this step's
        double d0;
        const double* w;  // slot h - 1's weight (slot 0's own in the first step)
        if constexpr (TAB) {
            const int j = h - a.N0;
            d0 = scalar_ptr(a.d0)[(int64_t)(j + 2) * a.nprob + p];
            w = a.w + ((int64_t)p * a.ldw + h - 1) * kHistBlock + j;
        } else {
            d0 = scalar_ptr(a.d0)[p];
            w = a.w + (int64_t)p * a.ldw;
        }
        constexpr int ws = TAB ? -kHistBlock : 1;
        // steps of this one's kMtSub after it, as far as the launch goes
        const int left = min(kMtSub - 1 - ((h - a.N0) & (kMtSub - 1)), a.ks - 1 - st);
        if (h >= 0 && (st == 0 || ((h - a.N0) & (kMtSub - 1)) == 0))
            mt_fill<HT, CM>(hist, a.ldh, P.hoff, n, a.N0, h, left + 1, a.G, w, ws, g, nl, acc);
#pragma unroll
        for (int r = 0; r < CM; ++r) {
            const int e = r * nl + g;
            double o = -d0 * u[r];
            if (h > 0) o += P.Da * acc[0][r];
            if (e < n) Y[pad_at<CM>(e)] = o;
        }
        for (int it = 0; it < a.picard; ++it) {
            __syncthreads();  // X, Y and x0 are in
            const double x0 = sh.x0;
            // top boundary: al1 / bt1 (mt_minimal.cpp:831-834, 944-947)
            int first_order;
            if (P.top == FRM_TOP_DIRICHLET) first_order = 0;
            else if (P.top == FRM_TOP_FLUX) first_order = 1;
            else first_order = (mt_inv(P, x0) != 1e20);
            const double al_first = first_order ? 1.0 : 0.0;
            double b0;
            if (P.top == FRM_TOP_DIRICHLET) {
                b0 = P.top_val;
            } else {
                const double Uc = 1.0 * P.dL * (P.Ev - 0.0) / mt_KK(P, x0);
                b0 = first_order ? -Uc : -Uc * mt_KK(P, X[0]) / P.dL;
            }
            double om[CM];
            if constexpr (TAB) {
#pragma unroll
                for (int k = 0; k < CM; ++k) A[k] = f[k] = al[k] = 0.0;
            }
#pragma unroll
            for (int k = 0; k < CM; ++k) om[k] = e0 + k < n ? Y[g * (CM + 1) + k] : 0.0;
            const double xp = X[pad_at<CM>(n - 1)];  // U_{N-1} of the last iterate
            if (!(fixed && factored)) {
                // A, B, R of al1 (B in f, R in al until the recurrence); the
                // conductivity slides along the chunk, its ends come from
                // the neighbouring lanes and wavefronts
                const int el = min(e0 + CM, n) - 1 - e0;  // the chunk's last element
                const double* xc = X + g * (CM + 1);
                const double Kf = mt_KK(P, xc[0]), Ke = mt_KK(P, xc[max(el, 0)]);
                double Km = __shfl_up(Ke, 1), Kr = __shfl_down(Kf, 1);
                if (W > 1) {
                    if (lane == 0) sh.Kf[wl] = Kf;
                    if (lane == 63) sh.Ke[wl] = Ke;
                    __syncthreads();
                    if (lane == 0 && wl > 0) Km = sh.Ke[wl - 1];
                    if (lane == 63 && wl < W - 1) Kr = sh.Kf[wl + 1];
                }
                // node 0 and node N, one evaluation for both ends
                const double Kx = mt_KK(P, g == 0 ? x0 : xN);
                if (g == 0) Km = Kx;
                if (g == last) Kr = last == 0 ? mt_KK(P, xN) : Kx;
                Mob m{1.0, 0.0, 0.0, 1.0};
                double Kc = Kf;
#pragma unroll
                for (int k = 0; k < CM; ++k) {
                    double Kp = Kr;
                    if (k < CM - 1 && k < el) Kp = k + 1 == el ? Ke : mt_KK(P, xc[k + 1]);
                    if (e0 + k < n) {
                        const double inv = mt_inv(P, xc[k]);
                        A[k] = P.Dg * Km * inv;
                        f[k] = P.Dg * Kp * inv;
                        al[k] = inv * (Kp + Km) * P.Dg + d0;
                        om[k] += (Kc - Km) * idL;
                        // alpha: Al[i+1] = B/(R - A Al[i]), a Moebius map of
                        // Al: [[0, B], [-A, R]] times the product so far
                        const double t0 = f[k] * m.m10, t1 = f[k] * m.m11;
                        m.m10 = al[k] * m.m10 - A[k] * m.m00;
                        m.m11 = al[k] * m.m11 - A[k] * m.m01;
                        m.m00 = t0;
                        m.m01 = t1;
                    }
                    Km = Kc;
                    Kc = Kp;
                    if (k % 4 == 3) m = mob_scale(m);
                }
                Mob tot;
                const Mob pre = scan_mob_up_total<false>(m, lane, tot);
                double ya = al_first, yb = 1.0;  // Al entering the wavefront, as a quotient
                if (W > 1) {
                    if (lane == 0) sh.m[wl] = tot;
                    __syncthreads();
                    for (int w = 0; w < wl; ++w) {
                        const Mob q = sh.m[w];
                        const double t = q.m00 * ya + q.m01 * yb;
                        yb = q.m10 * ya + q.m11 * yb;
                        ya = t;
                    }
                }
                double y = (pre.m00 * ya + pre.m01 * yb) / (pre.m10 * ya + pre.m11 * yb);
#pragma unroll
                for (int k = 0; k < CM; ++k) {
                    if (e0 + k < n) {
                        const double den = 1.0 / (al[k] - A[k] * y);
                        y = f[k] * den;
                        al[k] = y;   // Al[i+1]
                        f[k] = den;  // Al[i+1] / B
                    }
                }
                factored = true;
            }
            // beta: Bt[i+1] = (Al[i+1]/B)(A Bt[i] - Om)
            double Pp = 1.0, Qq = 0.0, Pt, Qt;
#pragma unroll
            for (int k = 0; k < CM; ++k) {
                if (e0 + k < n) {
                    const double pk = f[k] * A[k], qk = -f[k] * om[k];
                    Qq = pk * Qq + qk;
                    Pp = pk * Pp;
                }
            }
            scan_affine_up_total(Pp, Qq, lane, Pt, Qt);
            double bt = b0;  // value entering the wavefront
            if (W > 1) {
                if (lane == 0) {
                    sh.fP[wl] = Pt;
                    sh.fQ[wl] = Qt;
                }
                __syncthreads();
                for (int w = 0; w < wl; ++w) bt = sh.fP[w] * bt + sh.fQ[w];
            }
            bt = Pp * bt + Qq;
#pragma unroll
            for (int k = 0; k < CM; ++k) {
                if (e0 + k < n) {
                    bt = f[k] * (A[k] * bt - om[k]);
                    om[k] = bt;  // om now holds Bt[i+1]
                }
            }
            // bottom boundary (mt_minimal.cpp:987-1020), gamma = 1 so Qb = -0
#pragma unroll
            for (int k = 0; k < CM; ++k) {
                if (e0 + k == n - 1) {
                    const double BtN = om[k], AlN = al[k], Qb = -0.0;
                    double UN;
                    if (P.bottom_cond == 1)
                        UN = P.Hbottom;
                    else if (fabs(BtN + Qb) > 1e-15)
                        UN = (fabs(1.0 - AlN) > 1e-15) ? (BtN + Qb) / (1.0 - AlN) : xp + Qb;
                    else
                        UN = (fabs(1.0 - AlN) > 1e-15) ? 0.0 : xp + Qb;
                    sh.un = UN;
                }
            }
            // back substitution U_i = Al[i+1] U_{i+1} + Bt[i+1]
            Pp = 1.0;
            Qq = 0.0;
#pragma unroll
            for (int k = CM - 1; k >= 0; --k) {
                if (e0 + k < n) {
                    Qq = al[k] * Qq + om[k];
                    Pp = al[k] * Pp;
                }
            }
            scan_affine_down_total(Pp, Qq, lane, Pt, Qt);
            if (lane == 0) {
                sh.bP[wl] = Pt;
                sh.bQ[wl] = Qt;
            }
            __syncthreads();
            xN = sh.un;
            double y = xN;
            for (int w = W - 1; w > wl; --w) y = sh.bP[w] * y + sh.bQ[w];
            y = Pp * y + Qq;
#pragma unroll
            for (int k = CM - 1; k >= 0; --k) {
                if (e0 + k < n) {
                    y = al[k] * y + om[k];
                    X[g * (CM + 1) + k] = y;
                }
            }
            if (g == 0) sh.x0 = al_first * y + b0;
        }
        __syncthreads();
        double d[CM] = {};
#pragma unroll
        for (int r = 0; r < CM; ++r) {
            const int e = r * nl + g;
            if (e < n) {
                const double v = X[pad_at<CM>(e)];
                const HT inc = (HT)(v - u[r]);
                if (h >= 0) hist[(int64_t)h * a.ldh + P.hoff + e] = inc;
                d[r] = (double)inc;
                u[r] = v;
            }
        }
        if (h >= 0) mt_push<CM>(left, w, ws, d, acc);
    }
#pragma unroll
    for (int r = 0; r < CM; ++r)
        if (r * nl + g < n) Ug[r * nl + g + 1] = u[r];
    if (g == 0) {
        Ug[0] = sh.x0;
        Ug[N] = xN;
        Ug[N + 1] = xN;
    }
}

// One workgroup per problem, a wavefront per 64 kMtCM of the largest problem's
// unknowns; wavefronts that a smaller problem does not need leave at once, and
// a workgroup's place is free as soon as its own problem is done.
template <typename HT, bool TAB>
__global__ __launch_bounds__(64 * kMtMaxW) __attribute__((amdgpu_waves_per_eu(3, 8))) void k_mt_steps(MtStepArgs a) {
    constexpr int CM = kMtCM;
    __shared__ double X[64 * kMtMaxW * (CM + 1)], Y[64 * kMtMaxW * (CM + 1)];
    __shared__ MtShare sh;
    const int p = same_on_lanes(a.order[blockIdx.x]);
    const int W = (same_on_lanes(a.pr[p].N) - 1 + 64 * CM - 1) / (64 * CM);
    if ((int)(threadIdx.x >> 6) >= W) return;
    mt_steps<CM, HT, TAB>(a, p, W, X, Y, sh);
}

// ---------------------------------------------------------------- AB kind
// The manufactured solutions of MF_int_series.cpp:860-873 (F_func = src);
// E is the Mittag-Leffler factor of the source at time t.
constexpr double kAbPi = 3.14159265358979323846;

__host__ __device__ inline double ab_CC(int F, double x, double t) {
    if (F == 0) return t * t * t * t;
    if (F == 1) return x * (x - 1.0) * t * t;
    if (F == 2) return t * t * t * t * t * sin(kAbPi * x);
    return 0.0;
}

// sp, cp: sin and cos of pi x (F = 2 only; the same in every step)
__device__ inline double ab_f(int F, double x, double t, double a, double E, double sp, double cp) {
    if (F == 0) return (24.0 / (1.0 - a)) * t * t * t * t * E;
    if (F == 1) return (2.0 * x - 1.0) * t * t - 2 * t * t + (2.0 / (1.0 - a)) * x * (x - 1.0) * t * t * E;
    if (F == 2)
        return (120.0 / (1.0 - a)) * t * t * t * t * t * sp * E +
               kAbPi * t * t * t * t * t * (kAbPi * sp + cp);
    return 0.0;
}

__device__ inline double ab_CC_in(int F, double x, double t, double sp) {
    return F == 2 ? t * t * t * t * t * sp : ab_CC(F, x, t);
}

struct AbStepArgs {
    const MtProbDev* pr;
    const int* order;    // problems, largest first
    double* U;
    double* hist;        // slot k - 1 takes step k's (C^k - C^{k-1})/tau
    int64_t ldh;
    const double* G;     // the block's far sums (null: no settled slots)
    const double* w;     // lag-indexed I(lag+1) per problem
    int ldw;
    const double* d0;    // I(1)/(1-alpha) per problem
    const double* cf;    // per history node: -1/(B - A Al_{j-1})
    const double* cal;   // per history node: -Al_j
    const double* ml;    // [nprob][ldml] source factor at step k
    int ldml;
    const double* ser;   // series problems: MF_intF_choice's value per history node
    int N0;              // the block's start (history index)
    int k0, ks;          // steps k0 .. k0 + ks - 1, t = k tau; k_ab_steps takes series
                         // problems one step at a time
    double tau;
    double* err;         // per problem: running sum of (C_j - CC)^2
};

// Steps a.k0 .. of problem p on W wavefronts of one workgroup: right-hand side
// Rp_j = I(1)/(1-a) C_j + f - history/(1-a) (MF_int_series.cpp:922-931), the
// Thomas sweep with the exact Dirichlet ends (935-945) through the scan-seeded
// line solve (the constant alpha recurrence is precomputed), the increment
// push and the squared error against CC (947-951).  Everything but the
// recurrences runs in element order; the source's sines are taken once per
// launch.
template <int CM>
__device__ __forceinline__ void ab_steps(const AbStepArgs& a, int p, int W, double* X, double* SC,
                                         MtShare& sh) {
    const int lane = threadIdx.x & 63, wl = same_on_lanes((int)(threadIdx.x >> 6));
    const MtProbDev P = same_on_lanes(a.pr[p]);
    const int m = P.N, n = m - 1;
    const int g = threadIdx.x, nl = 64 * W, e0 = g * CM;
    const double h = P.dL, alpha = P.alpha, i1a = 1.0 / (1.0 - alpha), Ii1a = scalar_ptr(a.d0)[p];
    const double A = -(1.0 / (h * h)) - (1.0 / (2.0 * h));
    double* C = a.U + P.uoff;
    // the sines and cosines wait in LDS (each lane's own), for the registers' sake
    double c0[CM], *sp = SC + g, *cp = sp + 64 * kMtMaxW * CM;
    constexpr int cs = 64 * kMtMaxW;
#pragma unroll
    for (int r = 0; r < CM; ++r) {
        const int e = min(r * nl + g, n - 1);
        c0[r] = C[e + 1];
        sp[r * cs] = P.src == 2 ? sinpi((e + 1) * h) : 0.0;
        cp[r * cs] = P.src == 2 ? cospi((e + 1) * h) : 0.0;
    }
    double cf[CM], cal[CM];
#pragma unroll
    for (int k = 0; k < CM; ++k) {
        const int e = min(e0 + k, n - 1);
        cf[k] = a.cf[P.hoff + e];
        cal[k] = a.cal[P.hoff + e];
    }
    double es = a.err[p], b0 = 0.0, un = 0.0;
    double acc[kMtSub][CM];  // history sums of this step and those left of its kMtSub
    for (int st = 0; st < a.ks; ++st) {
        const int step = a.k0 + st, hi = step - 1;  // history index: slot hi is this step's
        const double t = step * a.tau;
        const double E = scalar_ptr(a.ml)[(int64_t)p * a.ldml + hi];
        const double* w = a.w + (int64_t)p * a.ldw;
        const int left = min(kMtSub - 1 - ((hi - a.N0) & (kMtSub - 1)), a.ks - 1 - st);
        if (!P.ser && (st == 0 || ((hi - a.N0) & (kMtSub - 1)) == 0))
            mt_fill<double, CM>(a.hist, a.ldh, P.hoff, n, a.N0, hi, left + 1, a.G, w, 1, g, nl, acc);
        double hs[CM];
        if (hi > 0) {
            if (P.ser) {  // MF_intF_choice's value, already over (1 - a)
#pragma unroll
                for (int r = 0; r < CM; ++r) hs[r] = a.ser[P.hoff + min(r * nl + g, n - 1)];
            } else {
#pragma unroll
                for (int r = 0; r < CM; ++r) hs[r] = acc[0][r] * i1a;
            }
        }
#pragma unroll
        for (int r = 0; r < CM; ++r) {
            const int e = r * nl + g;
            double rp = Ii1a * c0[r] + ab_f(P.src, (e + 1) * h, t, alpha, E, sp[r * cs], cp[r * cs]);
            if (hi > 0) rp -= hs[r];
            if (e < n) X[pad_at<CM>(e)] = rp;
        }
        __syncthreads();
        b0 = ab_CC(P.src, 0.0, t);
        un = ab_CC(P.src, m * h, t);
        double v[CM], Pp = 1.0, Qq = 0.0, Pt, Qt;
#pragma unroll
        for (int k = 0; k < CM; ++k) v[k] = e0 + k < n ? X[g * (CM + 1) + k] : 0.0;
#pragma unroll
        for (int k = 0; k < CM; ++k) {
            if (e0 + k < n) {
                const double pk = cf[k] * A, qk = -cf[k] * v[k];
                Qq = pk * Qq + qk;
                Pp = pk * Pp;
            }
        }
        scan_affine_up_total(Pp, Qq, lane, Pt, Qt);
        double y = b0;  // value entering the wavefront
        if (W > 1) {
            if (lane == 0) {
                sh.fP[wl] = Pt;
                sh.fQ[wl] = Qt;
            }
            __syncthreads();
            for (int w = 0; w < wl; ++w) y = sh.fP[w] * y + sh.fQ[w];
        }
        y = Pp * y + Qq;
#pragma unroll
        for (int k = 0; k < CM; ++k) {
            if (e0 + k < n) {
                y = cf[k] * (A * y - v[k]);
                v[k] = y;
            }
        }
        Pp = 1.0;
        Qq = 0.0;
#pragma unroll
        for (int k = CM - 1; k >= 0; --k) {
            if (e0 + k < n) {
                Qq = cal[k] * Qq + v[k];
                Pp = cal[k] * Pp;
            }
        }
        scan_affine_down_total(Pp, Qq, lane, Pt, Qt);
        y = un;
        if (W > 1) {
            if (lane == 0) {
                sh.bP[wl] = Pt;
                sh.bQ[wl] = Qt;
            }
            __syncthreads();
            for (int w = W - 1; w > wl; --w) y = sh.bP[w] * y + sh.bQ[w];
        }
        y = Pp * y + Qq;
#pragma unroll
        for (int k = CM - 1; k >= 0; --k) {
            if (e0 + k < n) {
                y = cal[k] * y + v[k];
                X[g * (CM + 1) + k] = y;
            }
        }
        __syncthreads();
        double d2 = 0.0, inc[CM] = {};
#pragma unroll
        for (int r = 0; r < CM; ++r) {
            const int e = r * nl + g;
            if (e < n) {
                const double c = X[pad_at<CM>(e)];
                inc[r] = (c - c0[r]) / a.tau;
                a.hist[(int64_t)hi * a.ldh + P.hoff + e] = inc[r];
                c0[r] = c;
                const double d = fabs(c - ab_CC_in(P.src, h * (e + 1), t, sp[r * cs]));
                d2 += d * d;
            }
        }
        if (!P.ser) mt_push<CM>(left, w, 1, inc, acc);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) d2 += __shfl_xor(d2, o);
        if (W > 1) {
            if (lane == 0) sh.es[wl] = d2;
            __syncthreads();
            d2 = sh.es[0];
            for (int w = 1; w < W; ++w) d2 += sh.es[w];
        }
        es += d2;  // the two ends equal CC exactly
    }
#pragma unroll
    for (int r = 0; r < CM; ++r)
        if (r * nl + g < n) C[r * nl + g + 1] = c0[r];
    if (g == 0) {
        C[0] = b0;  // bt[0] - al[0] C[1] with al[0] = 0
        C[m] = un;
        a.err[p] = es;
    }
}

__global__ __launch_bounds__(64 * kMtMaxW) __attribute__((amdgpu_waves_per_eu(3, 8))) void k_ab_steps(AbStepArgs a) {
    constexpr int CM = kMtCM;
    __shared__ double X[64 * kMtMaxW * (CM + 1)], SC[2 * 64 * kMtMaxW * CM];
    __shared__ MtShare sh;
    const int p = same_on_lanes(a.order[blockIdx.x]);
    const int W = (same_on_lanes(a.pr[p].N) - 1 + 64 * CM - 1) / (64 * CM);
    if ((int)(threadIdx.x >> 6) >= W) return;
    ab_steps<CM>(a, p, W, X, SC, sh);
}

// ---------------------------------------------------------------- AB series history
struct AbSeriesArgs {
    const MtProbDev* pr;
    const int* gprob;       // 128-node group -> problem
    int64_t ldh;
    const double* tab;      // per-step coefficient rows (ab_series_tables)
    const int* choice;      // per step: 1 series, 2 integral form
    const double* F;        // (C^{i-1} - C^{i-2}) / tau per history node
    double* lc1;            // [maxL][ldh] MF_intF's accumulators
    double* lc2;            // [maxL][ldh] MF_intF_Fv's accumulators
    signed char* lflag;     // [maxL][ldh] 0, or the sign of a log-form Lc2
    double* part;           // out: the series value per history node
    int i;                  // step, >= 2
    int* bad;               // bit 2: a non-finite term with ab_maxl above kRecountMaxL
};

// The longest series the sorted-pyramid recount holds in LDS.
constexpr int kRecountMaxL = 4096;

// The non-finite branch of MF_intF (MF_int_series.cpp:594-609 with
// F_nosorting = 1, where the `else` binds to the finiteness test) for the node
// of lc1, whose last non-finite term is `last`: each non-finite term replaces the
// running sum by sum_sort_pyramid (200-218) of all products Lc1[l] Kc[l]
// (0 where either is not finite), and the finite terms after the last such
// term are added to it in increasing l.  The whole workgroup works on the
// node: the products are sorted by decreasing magnitude in LDS (bitonic),
// then added pairwise level by level, an odd level's last element folded
// into the level's last sum.  Elements of equal magnitude and opposite sign
// may be ordered differently from std::sort; their sums are the same unless
// such a pair straddles a pair boundary.  Every thread of the workgroup
// calls it with the same node; thread 0 gets the sum.
//
// ab_pyramid: the workgroup's sort of v[0 .. n2) (a power of two, zeros from
// maxl on) and its pairwise sum; returns where the sum lies (v or w).
__device__ __forceinline__ const double* ab_pyramid(double* v, double* w, int n2, int maxl) {
#pragma clang fp contract(off)
    const int tid = threadIdx.x;
    for (int k = 2; k <= n2; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int l = tid; l < n2; l += blockDim.x) {
                const int m = l ^ j;
                if (m > l) {
                    const double x = v[l], y = v[m];
                    const bool desc = (l & k) == 0;
                    if (desc ? fabs(x) < fabs(y) : fabs(x) > fabs(y)) {
                        v[l] = y;
                        v[m] = x;
                    }
                }
            }
            __syncthreads();
        }
    // the levels: v -> w -> v ...; the zeros padding v beyond maxl are never
    // read
    double* src = v;
    double* dst = w;
    int m = maxl;
    if (m == 1 && tid == 0) v[0] += v[0];  // a single element is doubled
    while (m > 1) {
        const int m2 = m >> 1;
        for (int j = tid; j < m2; j += blockDim.x) dst[j] = src[2 * j] + src[2 * j + 1];
        __syncthreads();
        if ((m & 1) && tid == 0) dst[m2 - 1] += src[m - 1];
        __syncthreads();
        double* t = src;
        src = dst;
        dst = t;
        m = m2;
    }
    return src;
}

__device__ __forceinline__ double ab_block_recount(const double* lc1, int64_t ld, const double* T,
                                                   int maxl, int last, double* v, double* w) {
#pragma clang fp contract(off)
    int n2 = 1;
    while (n2 < maxl) n2 <<= 1;
    for (int l = threadIdx.x; l < n2; l += blockDim.x) {
        double x = 0.0;
        if (l < maxl) {
            const double c1 = lc1[(int64_t)l * ld], kc = T[(int64_t)l * kAbSeriesRows];
            if (isfinite(c1) && isfinite(kc)) x = c1 * kc;
        }
        v[l] = x;
    }
    __syncthreads();
    const double* src = ab_pyramid(v, w, n2, maxl);
    double ret = 0.0;
    if (threadIdx.x == 0) {
        ret = src[0];
        for (int l = last + 1; l < maxl; ++l) {
            const double c1 = lc1[(int64_t)l * ld], kc = T[(int64_t)l * kAbSeriesRows];
            if (isfinite(c1) && isfinite(kc)) ret += c1 * kc;
        }
    }
    __syncthreads();  // v and w are reused by the next node
    return ret;
}

// One term of a node's step: kc, lk its value coefficient (in log form where lk
// is not 0), k1 and k2, k2l the factors the increment F enters Lc1 and Lc2
// with (k2l for the log form, where lF = log|F|); updates Lc1 (series phase), Lc2 and its log
// flag, adds the term to ret.  False where the series phase met a non-finite
// Lc1 or kc.  Products and sums are rounded separately, as the reference's
// x86-64 build does.
__device__ __forceinline__ bool ab_term(bool series, double kc, double lk, double k1, double k2,
                                        double k2l, double F, double lF, double& c1, double& c2,
                                        int& fl, double& ret) {
#pragma clang fp contract(off)
    if (fl == 0) {
        const double nv = c2 + k2 * F;
        if (!isfinite(nv)) {
            fl = c2 > 0.0 ? 1 : -1;
            c2 = log(fabs(c2));
        } else {
            c2 = nv;
        }
    } else {
        c2 = k2l + lF;
        fl = F > 0.0 ? -1 : 1;
    }
    if (series) {
        c1 = c1 + k1 * F;
        if (!isfinite(c1) || !isfinite(kc)) return false;
        ret += c1 * kc;
        return true;
    }
    double v = 0.0;
    if (fl == 0 && lk == 0) v = c2 * kc;
    if (fl != 0 && lk == 0) v = fl * (kc > 0.0 ? 1.0 : -1.0) * exp(c2 + log(fabs(kc)));
    if (fl == 0 && lk != 0) v = lk * (c2 > 0.0 ? 1.0 : -1.0) * exp(kc + log(fabs(c2)));
    if (fl != 0 && lk != 0) v = lk * fl * exp(kc + c2);
    if (!isfinite(v)) v = 0.0;
    ret += v;
    return true;
}

// Terms l0 .. l1 - 1 of MF_intF_choice(i, ..., on = i - 2, mn = 1, append_all =
// 1, Fvalue = F) (MF_int_series.cpp:839-853) on one node's accumulators, one
// lane per node.  Both phases append to MF_intF_Fv's Lc2 (779-804: add sk F, or
// keep log|Lc2| with its sign once the sum overflows, after which the newest
// term alone is kept in log form); the series phase adds dp F to MF_intF's Lc1
// and returns sum Lc1 Kc (598-603), the integral phase returns sum of the
// products of Lc2 and Kc with either in log form (806-822), terms in increasing
// l.  Returns in *last the last term whose Lc1 or Kc was not finite.  T: the
// step's coefficients, the same on every lane.
__device__ __forceinline__ double ab_series_node(const_doubles T, bool series, double F, int64_t ld,
                                                 double* __restrict__ lc1, double* __restrict__ lc2,
                                                 signed char* __restrict__ lflag, int l0, int l1,
                                                 int* last) {
    // the accumulators are only this node's: no access aliases another, so
    // the loads of several terms can be in flight together
    constexpr int R = kAbSeriesRows;
    const double lF = log(fabs(F));
    double ret = 0.0;
    // one term: the accumulators of term l as loaded (c2, fl, c1)
    auto term = [&](int l, double c2, int fl, double c1) {
        const int64_t q = (int64_t)l * ld;
        const const_doubles t = T + (int64_t)l * R;
        const int f0 = fl;
        if (!ab_term(series, t[0], t[1], t[2], t[3], t[4], F, lF, c1, c2, fl, ret)) *last = l;
        lc2[q] = c2;
        if (fl != f0) lflag[q] = (signed char)fl;
        if (series) lc1[q] = c1;
    };
    // the accumulators of 8 terms are loaded before any is updated (the
    // terms are still added in increasing l)
    constexpr int B = 8;
    int l = l0;
    for (; l + B <= l1; l += B) {
        double c2[B], c1[B];
        int fl[B];
#pragma unroll
        for (int u = 0; u < B; ++u) {
            const int64_t q = (int64_t)(l + u) * ld;
            c2[u] = lc2[q];
            fl[u] = lflag[q];
            c1[u] = series ? lc1[q] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < B; ++u) term(l + u, c2[u], fl[u], c1[u]);
    }
    for (; l < l1; ++l) {
        const int64_t q = (int64_t)l * ld;
        term(l, lc2[q], lflag[q], series ? lc1[q] : 0.0);
    }
    return ret;
}

// One thread per node (ab_series_node); then the workgroup recounts, one
// node after another, the sums of its nodes that met a non-finite term
// (ab_block_recount), overwriting their part.  Three workgroups per CU: the
// recount's code would otherwise raise the kernel to 175 VGPRs (two waves
// per SIMD instead of three); held to 168 it spills 36 bytes per lane
// outside the term loop.
__global__ __launch_bounds__(256, 3) void k_ab_series(AbSeriesArgs a) {
    __shared__ double v[kRecountMaxL];
    __shared__ double w[kRecountMaxL / 2];
    __shared__ int2 todo[256];
    __shared__ int ntodo;
    if (threadIdx.x == 0) ntodo = 0;
    __syncthreads();
    const int64_t h = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int last_bad = -1, maxl = 0;
    const int p = h < a.ldh ? a.gprob[h / kGroup] : -1;  // a wavefront's nodes are one problem's
    if (__builtin_amdgcn_readfirstlane(p) >= 0) {
        const MtProbDev& P = a.pr[__builtin_amdgcn_readfirstlane(p)];
        if (P.ser && h - P.hoff < P.N - 1) {
            maxl = P.ser_maxl;
            const const_doubles T =
                scalar_ptr(a.tab + same_on_lanes(P.ser_off)) +
                (int64_t)(a.i - 2) * kAbSeriesRows * same_on_lanes(P.ser_maxl);
            a.part[h] = ab_series_node(T, a.choice[P.ser_coff + a.i - 2] == 1, a.F[h], a.ldh,
                                       a.lc1 + h, a.lc2 + h, a.lflag + h, 0, maxl, &last_bad) /
                        (1.0 - P.alpha);
        }
    }
    if (last_bad >= 0) {
        if (maxl <= kRecountMaxL)
            todo[atomicAdd(&ntodo, 1)] = make_int2((int)h, last_bad);
        else
            atomicOr(a.bad, 2);
    }
    __syncthreads();
    const int n = ntodo;
    for (int q = 0; q < n; ++q) {
        const int2 e = todo[q];
        const MtProbDev& P = a.pr[a.gprob[e.x / kGroup]];
        const double ret = ab_block_recount(
            a.lc1 + e.x, a.ldh,
            a.tab + P.ser_off + (int64_t)(a.i - 2) * kAbSeriesRows * P.ser_maxl, P.ser_maxl, e.y, v, w);
        if (threadIdx.x == 0) a.part[e.x] = ret / (1.0 - P.alpha);
    }
}

// ---------------------------------------------------------------- AB series, fused steps
// Steps of the problems with the series history, any number per launch: the
// problems are independent, so one workgroup stays with a problem from step to
// step and keeps its accumulators in LDS, where a series kernel and a sweep per
// step moved 34 bytes per node and term through the last-level cache each time
// (50 us of 60 us per step on 1024 problems of 100 intervals and 50 terms).
// NG = ceil(n / 64) wavefronts hold the nodes, (WAVES - 1) / NG of them a
// node's terms in equal runs; their partial sums meet in LDS, where one more
// wavefront takes them for the sweep.  Three sizes of LDS, so that small
// problems share a CU.  That batch over 600 steps: 35.5 -> 12.6 ms; the sums
// alone take about 3.4 us of the 4.9 us a problem's step has, the sweep 2.4
// (with the accumulators left in global memory two problems per CU did not fit
// L2 and it ran 34 ms; in registers the unrolled terms spilled, 53 ms).
constexpr int kSerSteps = 256;  // steps per launch of a batch with nothing else
constexpr int kSerNodes = 320;  // the sweep's 5 nodes per lane

struct SerSplit {
    int ng, groups, terms;  // wavefronts by nodes, by terms, terms of each
    bool fits;              // in `waves` wavefronts and `bytes` of LDS
};

// LDS: [maxl][n] (Lc1, Lc2); [groups][64 ng] partial sums; increment, state,
// sin and cos of pi x [n]; three lines in chunk order; recount [1.5 n2];
// last non-finite term per node [n], their count.
__host__ __device__ inline SerSplit ser_split(int n, int maxl, int waves, int bytes) {
    SerSplit s{(n + 63) / 64, 0, 0, false};
    if (n > kSerNodes || s.ng > waves - 1) return s;
    s.groups = (waves - 1) / s.ng;
    s.terms = (maxl + s.groups - 1) / s.groups;
    s.groups = (maxl + s.terms - 1) / s.terms;
    int n2 = 1;
    while (n2 < maxl) n2 <<= 1;
    const int64_t need = (int64_t)maxl * n * 16 + (int64_t)s.groups * s.ng * 512 + 4 * n * 8 +
                         3 * 64 * 6 * 8 + (int64_t)n2 * 12 + n * 4 + 16;
    s.fits = s.terms <= 64 && need <= bytes;
    return s;
}

struct SerShare {
    double2* c12;                        // [maxl][n]
    double *part, *F, *c, *sp, *cp, *X, *cf, *cal, *v, *w;
    int *bad, *nbad;
    __device__ SerShare(char* lds, int n, int maxl, const SerSplit& q) {
        int n2 = 1;
        while (n2 < maxl) n2 <<= 1;
        c12 = reinterpret_cast<double2*>(lds);
        part = reinterpret_cast<double*>(c12 + maxl * n);
        F = part + q.groups * q.ng * 64;
        c = F + n;
        sp = c + n;
        cp = sp + n;
        X = cp + n;
        cf = X + 64 * 6;
        cal = cf + 64 * 6;
        v = cal + 64 * 6;
        w = v + n2;
        bad = reinterpret_cast<int*>(w + (n2 + 1) / 2);
        nbad = bad + n;
    }
};

// The sweep of one step on one wavefront, as ab_steps: the state and the
// increment in element order, the recurrences in chunk order.  First the part
// of the right-hand side that does not need the series' value, then the rest;
// returns this lane's part of the sum of (C_j - CC)^2.  One wavefront's LDS
// accesses are in order.
template <int CM>
__device__ __forceinline__ void ser_rhs(const AbStepArgs& a, const MtProbDev& P, int step, double E,
                                        double Ii1a, const SerShare& sh) {
    const int lane = threadIdx.x & 63, n = P.N - 1;
    const double h = P.dL, t = step * a.tau;
#pragma unroll
    for (int r = 0; r < CM; ++r) {
        const int e = r * 64 + lane;
        if (e < n)
            sh.X[pad_at<CM>(e)] =
                Ii1a * sh.c[e] + ab_f(P.src, (e + 1) * h, t, P.alpha, E, sh.sp[e], sh.cp[e]);
    }
}

template <int CM>
__device__ __forceinline__ double ser_sweep(const AbStepArgs& a, const MtProbDev& P, int step,
                                            double i1a, double itau, int groups,
                                            const SerShare& sh) {
    const int lane = threadIdx.x & 63;
    const int m = P.N, n = m - 1, e0 = lane * CM, nn = (n + 63) / 64 * 64;
    const double h = P.dL, A = -(1.0 / (h * h)) - (1.0 / (2.0 * h)), t = step * a.tau;
    if (step >= 2) {
#pragma unroll
        for (int r = 0; r < CM; ++r) {
            const int e = r * 64 + lane;
            if (e < n) {
                double ret = sh.part[e];
                for (int q = 1; q < groups; ++q) ret += sh.part[q * nn + e];
                sh.X[pad_at<CM>(e)] -= ret * i1a;
            }
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    const double b0 = ab_CC(P.src, 0.0, t), un = ab_CC(P.src, m * h, t);
    double v[CM], Pp = 1.0, Qq = 0.0, Pt, Qt;
#pragma unroll
    for (int k = 0; k < CM; ++k) {
        v[k] = 0.0;
        if (e0 + k < n) {
            const double cf = sh.cf[lane * (CM + 1) + k];
            v[k] = sh.X[lane * (CM + 1) + k];
            const double pk = cf * A, qk = -cf * v[k];
            Qq = pk * Qq + qk;
            Pp = pk * Pp;
        }
    }
    scan_affine_up_total(Pp, Qq, lane, Pt, Qt);
    double y = Pp * b0 + Qq;
#pragma unroll
    for (int k = 0; k < CM; ++k) {
        if (e0 + k < n) {
            y = sh.cf[lane * (CM + 1) + k] * (A * y - v[k]);
            v[k] = y;
        }
    }
    Pp = 1.0;
    Qq = 0.0;
#pragma unroll
    for (int k = CM - 1; k >= 0; --k) {
        if (e0 + k < n) {
            const double cal = sh.cal[lane * (CM + 1) + k];
            Qq = cal * Qq + v[k];
            Pp = cal * Pp;
        }
    }
    scan_affine_down_total(Pp, Qq, lane, Pt, Qt);
    y = Pp * un + Qq;
#pragma unroll
    for (int k = CM - 1; k >= 0; --k) {
        if (e0 + k < n) {
            y = sh.cal[lane * (CM + 1) + k] * y + v[k];
            sh.X[lane * (CM + 1) + k] = y;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    double d2 = 0.0;
#pragma unroll
    for (int r = 0; r < CM; ++r) {
        const int e = r * 64 + lane;
        if (e < n) {
            const double c = sh.X[pad_at<CM>(e)], f = (c - sh.c[e]) * itau;
            a.hist[(int64_t)(step - 1) * a.ldh + P.hoff + e] = f;
            sh.F[e] = f;
            sh.c[e] = c;
            const double d = fabs(c - ab_CC_in(P.src, h * (e + 1), t, sh.sp[e]));
            d2 += d * d;
        }
    }
    return d2;
}

// A lane's run of terms of one step on the accumulators in LDS (c12: its node's
// first one, the next term's n further on), as ab_term, in increasing order;
// neg, pos: the terms whose Lc2 is in log form, by its sign.  Four terms at a
// time, together where no lane has anything rare among them (an Lc2 that
// overflows just now, a value that is not finite, a log form in the integral
// phase): two multiply-adds, a product and the finiteness tests each.
__device__ __forceinline__ double ser_terms(const_doubles T, bool series, double F, double2* c12,
                                            int n, int terms, int l0, uint64_t& neg, uint64_t& pos,
                                            int* last) {
#pragma clang fp contract(off)
    constexpr int B = 4, R = kAbSeriesRows;
    const double lF = __any((neg | pos) != 0) ? log(fabs(F)) : 0.0;  // log forms read it
    double ret = 0.0;
    for (int i0 = 0; i0 < terms; i0 += B) {
        double2 c[B];
        double v[B];
        const uint32_t logs = (uint32_t)((neg | pos) >> i0) & 15u;
        int plain = 1;  // & rather than &&: no branches
#pragma unroll
        for (int j = 0; j < B; ++j) c[j] = c12[min(i0 + j, terms - 1) * n];
#pragma unroll
        for (int j = 0; j < B; ++j) {
            const const_doubles t = T + min(i0 + j, terms - 1) * R;
            const double kc = t[0];
            const bool lg = logs >> j & 1;
            const double n2 = c[j].y + t[3] * F;
            plain &= (int)lg | (int)isfinite(n2);
            c[j].y = lg ? t[4] + lF : n2;
            if (series) {
                c[j].x = c[j].x + t[2] * F;
                v[j] = c[j].x * kc;
                plain &= (int)isfinite(c[j].x) & (int)isfinite(kc);
            } else {
                v[j] = c[j].y * kc;
                plain &= (int)!lg & (int)(t[1] == 0) & (int)isfinite(v[j]);
            }
        }
        if (__all(plain)) {
#pragma unroll
            for (int j = 0; j < B; ++j) {
                if (i0 + j < terms) {
                    c12[(i0 + j) * n] = c[j];
                    ret += v[j];
                }
            }
            const uint64_t m = uint64_t(15) << i0, l = (uint64_t)logs << i0;
            neg = (neg & ~m) | (F > 0.0 ? l : 0);
            pos = (pos & ~m) | (F > 0.0 ? 0 : l);
        } else {
#pragma unroll 1
            for (int i = i0; i < min(i0 + B, terms); ++i) {
                const const_doubles t = T + i * R;
                double2 x = c12[i * n];
                int fl = (int)(pos >> i & 1) - (int)(neg >> i & 1);
                if (!ab_term(series, t[0], t[1], t[2], t[3], t[4], F, lF, x.x, x.y, fl, ret))
                    *last = l0 + i;
                c12[i * n] = x;
                neg = (neg & ~(uint64_t(1) << i)) | (uint64_t)(fl < 0) << i;
                pos = (pos & ~(uint64_t(1) << i)) | (uint64_t)(fl > 0) << i;
            }
        }
    }
    return ret;
}

// After a step's series sums: the nodes that met a non-finite term, one after
// another, by the whole workgroup (sh.bad, sh.nbad).
__device__ __forceinline__ void ser_recounts(const double* T, int n, int maxl, int groups, int nn,
                                             const SerShare& sh) {
    for (int q = 0; q < n; ++q) {
        const int lb = sh.bad[q];  // the same on every lane
        if (lb < 0) continue;
        const double ret = ab_block_recount(&sh.c12[q].x, 2 * n, T, maxl, lb, sh.v, sh.w);
        if (threadIdx.x == 0) {
            sh.part[q] = ret;
            for (int g = 1; g < groups; ++g) sh.part[g * nn + q] = 0.0;
        }
    }
    __syncthreads();
}

template <int WAVES, int BYTES>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_ab_series_steps(
    AbStepArgs a, AbSeriesArgs b) {
    __shared__ __attribute__((aligned(16))) char lds[BYTES];
    const int lane = threadIdx.x & 63, wv = same_on_lanes((int)(threadIdx.x >> 6));
    const int p = same_on_lanes(a.order[blockIdx.x]);
    const MtProbDev P = same_on_lanes(a.pr[p]);
    const int m = P.N, n = m - 1, maxl = P.ser_maxl;
    const SerSplit sp = ser_split(n, maxl, WAVES, BYTES);
    const SerShare sh(lds, n, maxl, sp);
    const int nn = 64 * sp.ng, sweeper = sp.ng * sp.groups;
    if (wv > sweeper) return;  // before any barrier
    const int64_t ld = a.ldh, tstep = (int64_t)maxl * kAbSeriesRows;
    const double* tab = b.tab + P.ser_off;
    if (wv == sweeper) {
        const int cm = n <= 128 ? 2 : 5;
        double* C = a.U + P.uoff;
        for (int e = lane; e < n; e += 64) {
            const double x = (e + 1) * P.dL;
            sh.c[e] = C[e + 1];
            sh.F[e] = a.k0 >= 2 ? a.hist[(int64_t)(a.k0 - 2) * ld + P.hoff + e] : 0.0;
            sh.sp[e] = P.src == 2 ? sinpi(x) : 0.0;
            sh.cp[e] = P.src == 2 ? cospi(x) : 0.0;
            sh.cf[e + e / cm] = a.cf[P.hoff + e];
            sh.cal[e + e / cm] = a.cal[P.hoff + e];
            sh.bad[e] = -1;
        }
        if (lane == 0) *sh.nbad = 0;
        const double Ii1a = scalar_ptr(a.d0)[p], i1a = 1.0 / (1.0 - P.alpha), itau = 1.0 / a.tau;
        double es = 0.0;
        __syncthreads();
        for (int st = 0; st < a.ks; ++st) {
            const int step = a.k0 + st;
            const double E = scalar_ptr(a.ml)[(int64_t)p * a.ldml + step - 1];
            if (cm == 2) ser_rhs<2>(a, P, step, E, Ii1a, sh);
            else ser_rhs<5>(a, P, step, E, Ii1a, sh);
            __syncthreads();  // the series' sums are in
            if (*sh.nbad) {
                ser_recounts(tab + (step - 2) * tstep, n, maxl, sp.groups, nn, sh);
                for (int e = lane; e < n; e += 64) sh.bad[e] = -1;
                if (lane == 0) *sh.nbad = 0;
            }
            double d2 = cm == 2 ? ser_sweep<2>(a, P, step, i1a, itau, sp.groups, sh)
                                : ser_sweep<5>(a, P, step, i1a, itau, sp.groups, sh);
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) d2 += __shfl_xor(d2, o);
            es += d2;  // the two ends equal CC exactly
            __syncthreads();  // the increment is in
        }
        for (int e = lane; e < n; e += 64) C[e + 1] = sh.c[e];
        if (lane == 0) {
            const double t = (a.k0 + a.ks - 1) * a.tau;
            C[0] = ab_CC(P.src, 0.0, t);
            C[m] = ab_CC(P.src, m * P.dL, t);
            a.err[p] += es;
        }
        return;
    }
    const int tg = wv / sp.ng, l0 = tg * sp.terms, e = (wv - tg * sp.ng) * 64 + lane;
    const int terms = min(sp.terms, maxl - l0);
    const bool live = e < n;
    double2* c12 = sh.c12 + (int64_t)l0 * n + min(e, n - 1);
    uint64_t neg = 0, pos = 0;
    if (live)
        for (int i = 0; i < terms; ++i) {
            const int64_t q = (int64_t)(l0 + i) * ld + P.hoff + e;
            c12[i * n] = make_double2(b.lc1[q], b.lc2[q]);
            const int f = b.lflag[q];
            neg |= (uint64_t)(f < 0) << i;
            pos |= (uint64_t)(f > 0) << i;
        }
    __syncthreads();
    for (int st = 0; st < a.ks; ++st) {
        const int step = a.k0 + st;
        if (step >= 2) {
            double ret = 0.0;
            int last = -1;
            if (live)
                ret = ser_terms(scalar_ptr(tab + (step - 2) * tstep + (int64_t)l0 * kAbSeriesRows),
                                same_on_lanes(b.choice[P.ser_coff + step - 2]) == 1, sh.F[e], c12, n,
                                terms, l0, neg, pos, &last);
            sh.part[tg * nn + e] = ret;
            if (last >= 0) {
                atomicMax(&sh.bad[e], last);
                *sh.nbad = 1;
            }
        }
        __syncthreads();
        if (step >= 2 && *sh.nbad) ser_recounts(tab + (step - 2) * tstep, n, maxl, sp.groups, nn, sh);
        __syncthreads();
    }
    if (live)
        for (int i = 0; i < terms; ++i) {
            const int64_t q = (int64_t)(l0 + i) * ld + P.hoff + e;
            const double2 x = c12[i * n];
            b.lc1[q] = x.x;
            b.lc2[q] = x.y;
            b.lflag[q] = (signed char)((int)(pos >> i & 1) - (int)(neg >> i & 1));
        }
}

// The variants, smallest first: wavefronts and LDS of a workgroup.
#define FRM_SER_CASES(X) X(4, 36 * 1024) X(8, 76 * 1024) X(16, 156 * 1024)

// ---------------------------------------------------------------- fitting error
// solve_and_test (mt_minimal.cpp:1277-1330) for every problem of the batch:
// one thread per problem walks the observations of the current step in
// order (so the sum is the reference's, term by term).
struct FitArgs {
    const MtProbDev* pr;
    int nprob;
    const double* U;
    const double* T;   // observation times, depths, values
    const double* Z;
    const double* F;
    const int* idx;    // the observations of this step, in order
    int cnt;
    double tt, tau;
    double* vs;        // [nprob][nobs] values before the step
    int nobs;
    double* err;       // [nprob]
    int* dead;         // [nprob]: U[0] was not finite after a step
};

// U at depth z between nodes j, j+1 with dL j < z <= dL (j+1), j < jmax;
// false when no such j
__device__ inline bool fit_interp(const double* U, double dL, int jmax, double z, double& v) {
    const double r = z / dL;
    if (!(r > 0.0) || r > jmax + 2.0) return false;  // no interval (also NaN)
    int j = (int)floor(r) - 1;
    if (j < 0) j = 0;
    for (int q = 0; q < 3 && j < jmax; ++q, ++j)
        if (((dL * j) < z) && ((dL * (j + 1)) >= z)) {
            const double k2 = (z - (dL * j)) / dL;
            v = (1 - k2) * U[j] + k2 * U[j + 1];
            return true;
        }
    return false;
}

__global__ __launch_bounds__(256) void k_fit_before(FitArgs a) {
#pragma clang fp contract(off)
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= a.nprob) return;
    const MtProbDev& P = a.pr[p];
    const double* U = a.U + P.uoff;
    for (int q = 0; q < a.cnt; ++q) {
        const int o = a.idx[q];
        double v;
        if (fit_interp(U, P.dL, P.N - 1, a.Z[o], v)) a.vs[(int64_t)p * a.nobs + o] = v;
    }
}

__global__ __launch_bounds__(256) void k_fit_after(FitArgs a) {
#pragma clang fp contract(off)
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= a.nprob || a.dead[p]) return;
    const MtProbDev& P = a.pr[p];
    const double* U = a.U + P.uoff;
    double e = a.err[p];
    for (int q = 0; q < a.cnt; ++q) {
        const int o = a.idx[q];
        const double k1 = (a.T[o] - a.tt) / a.tau;
        double v;
        if (fit_interp(U, P.dL, P.N, a.Z[o], v)) {
            v = (1 - k1) * a.vs[(int64_t)p * a.nobs + o] + k1 * v;
            if (v > 0.0) v = 0.0;
            e += (a.F[o] - v) * (a.F[o] - v);
        }
    }
    if (!isfinite(U[0])) {
        e = 1e300;
        a.dead[p] = 1;
    }
    a.err[p] = e;
}

}  // namespace frm

using namespace frm;

namespace frm {
// A kernel launch of one step: function, shape and a copy of its argument
// values (hipKernelNodeParams takes pointers to them).
struct KRec {
    const void* func = nullptr;
    dim3 grid, block;
    bool branch = false;  // weights formed ahead (kind psi): a branch of the graph
    bool join = false;    // the first launch that reads weights formed on the branch
    alignas(16) unsigned char buf[448];
    size_t used = 0;
    size_t off[16];
    int n = 0;
    template <class T>
    void arg(const T& v) {
        static_assert(sizeof(T) <= 448, "kernel argument too large");
        used = (used + alignof(T) - 1) / alignof(T) * alignof(T);
        std::memcpy(buf + used, &v, sizeof(T));
        off[n++] = used;
        used += sizeof(T);
    }
    void ptrs(void** p) {
        for (int i = 0; i < n; ++i) p[i] = buf + off[i];
    }
};
// The launches of up to kGraphSteps consecutive steps as an instantiated
// graph (kernel nodes in a chain; for kind psi the next block's weights on a
// branch beside it), reused for every run of steps that issues the same
// kernels in the same order: only the nodes' arguments and grids change
// between launches.
constexpr int kGraphSteps = 32;
struct StepGraph {
    std::vector<const void*> funcs;
    std::vector<int> tags;  // join * 2 + branch of every node
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    std::vector<hipGraphNode_t> nodes;
};
}  // namespace frm

struct frm_mt1d {
    frm_ctx* ctx = nullptr;
    int nprob = 0, kind = 0, capacity = 0, precision = 0, picard = 1;
    double tau = 0;
    int tstep = 1;
    int depth = 0;
    int slots = 0;
    int64_t nU = 0, ldh = 0, ngroups = 0;
    int maxN = 0;
    std::vector<MtProbDev> hprobs;
    MtProbDev* probs = nullptr;
    int* gprob = nullptr;
    int* gvalid = nullptr;    // real nodes per group (0 for padding groups)
    int* order = nullptr;     // problems by size, largest first
    int min_chunk = 32;       // fewest slots a wavefront of a split far pass takes
    int graph = 0;                  // steps as HIP graphs, built once per launch sequence
    std::vector<frm::StepGraph> graphs;  // one instantiated graph per launch sequence
    std::vector<frm::KRec>* rec = nullptr;  // while set, launches are recorded, not issued
    bool rec_join = false;                   // the next launch waits for the branch
    hipStream_t lstream = nullptr;          // while set, launches go to this stream
    // kind psi: the weights of block b + 1 are formed on the context's second
    // stream while block b's steps run on its stream (the weights do not
    // depend on the state); w and d0 then hold two buffers, block b using
    // buffer b & 1.  wready[q]: buffer q's weights are formed; wfree[q]: the
    // last launch that read buffer q is done.
    hipStream_t wstream = nullptr;
    hipEvent_t wready[2] = {nullptr, nullptr}, wfree[2] = {nullptr, nullptr};
    int wblock = -1;                        // the block whose weights the stream's work has
    int wahead = -1;                        // the block whose weights were launched ahead
    size_t wsz = 0;                         // elements of one w buffer (0: one buffer)
    int64_t hnodes = 0, hnodes_mt = 0;  // real history nodes (all; full-history problems)
    double* U = nullptr;
    void* hist = nullptr;     // slots * ldh (FP64 or FP32)
    double* part = nullptr;   // series problems: the series value per node
    double* far = nullptr;    // [kHistBlock][ldh] far sums of the current block
    double* w = nullptr;      // nprob * ldw weights, lag-indexed; kind psi: a block's table
    double* d0 = nullptr;     // per-problem current-step coefficient (kind psi: per step too)
    double* psi_g = nullptr;  // kind psi: g(a tau) and the inverse's derivative there,
                              // [2][nprob][capacity + 2]
    int* bad = nullptr;       // set when a psi weight is not finite
    int ldw = 0;
    // kind AB
    double* ab_cf = nullptr;  // [ldh] -1/(B - A Al_{j-1})
    double* ab_cal = nullptr; // [ldh] -Al_j
    double* ab_ml = nullptr;  // [nprob][capacity] source factors
    double* ab_err = nullptr; // [nprob]
    // kind AB, series history (ab_series)
    int ser_maxL = 0, ser_count = 0;
    int ser_waves = 0;  // k_ab_series_steps: the variant's wavefronts (0: not all series
                        // problems fit one)
    int* gprob_mt = nullptr;  // group -> problem for the full-history sums (-1: series)
    double* ser_tab = nullptr;
    int* ser_choice = nullptr;
    double* ser_lc = nullptr;        // [2][maxL][ldh]: Lc1, Lc2
    signed char* ser_flag = nullptr; // [maxL][ldh]
    // kind psi: (problem, interval) pairs whose weight series was not finite
    int2* psi_queue = nullptr;
    int* psi_qcount = nullptr;       // [2] queue lengths (by step parity)
    int psi_qcap = 0;
    std::vector<double> ser_bytes;   // per step i >= 2: algorithmic bytes of k_ab_series
    double ser_state_bytes = 0.0;    // the accumulators read and written once
    // fitting error (solve_and_test)
    int nobs = 0;
    std::vector<double> obs_T;       // host copy: which observations fall in which step
    double tt = 0.0;                 // start of the next step, accumulated as the reference does
    double* fit_obs = nullptr;       // [3][nobs] T, Z, F
    int* fit_idx = nullptr;          // [nobs] scratch: the observations of one step
    double* fit_vs = nullptr;        // [nprob][nobs]
    double* fit_err = nullptr;       // [nprob]
    int* fit_dead = nullptr;         // [nprob]
    std::vector<int> fit_off;        // [capacity+1]: observations of step k at fit_idx[off[k-1] ..]
};

// Issues a kernel launch on the context's stream, or records it for the
// step graph while s->rec is set; arguments are converted to the kernel's
// parameter types.
template <typename... KArgs, typename... Args>
static hipError_t mt_launch(frm_mt1d* s, void (*kern)(KArgs...), dim3 grid, dim3 block,
                            Args&&... args) {
    static_assert(sizeof...(KArgs) == sizeof...(Args), "argument count");
    frm::KRec r;
    r.func = (const void*)kern;
    r.grid = grid;
    r.block = block;
    (r.arg(static_cast<std::decay_t<KArgs>>(args)), ...);
    if (s->rec) {
        r.branch = s->lstream != nullptr;
        if (!r.branch) {
            r.join = s->rec_join;
            s->rec_join = false;
        }
        s->rec->push_back(r);
        return hipSuccess;
    }
    void* p[16];
    r.ptrs(p);
    return hipLaunchKernel(r.func, grid, block, p, 0, s->lstream ? s->lstream : s->ctx->stream);
}

// The weight buffers of block b (kind psi: two, by parity).
static double* mt_w(const frm_mt1d* s, int b) {
    return s->w + (s->wsz ? (size_t)(b & 1) * s->wsz : 0);
}
static double* mt_d0(const frm_mt1d* s, int b) {
    return s->d0 + (s->wsz ? (size_t)(b & 1) * s->nprob * (kHistBlock + 2) : 0);
}

// Kind psi: the weights of block b, then the quadrature fallback of those
// whose series was not finite.
static hipError_t mt_launch_psi_weights(frm_mt1d* s, int b) {
    PsiArgs a;
    a.pr = s->probs;
    a.nprob = s->nprob;
    a.N0 = b * kHistBlock;
    a.capacity = s->capacity;
    a.tau = s->tau;
    a.gl = s->capacity + 2;
    a.g = s->psi_g;
    a.dg = s->psi_g + (size_t)s->nprob * a.gl;
    a.w = mt_w(s, b);
    a.ldw = s->ldw;
    a.d0 = mt_d0(s, b);
    a.bad = s->bad;
    a.queue = s->psi_queue;
    a.qcap = s->psi_qcap;
    a.qcount = s->psi_qcount;
    // 16 slots per workgroup up to the block's last step's newest, and one
    // workgroup for the current-step factors
    const dim3 grid((unsigned)(b + 2), (unsigned)s->nprob);
    hipError_t e = mt_launch(s, k_psi_weights, grid, dim3(256), a);
    // a fixed grid: threads beyond the queue's length exit at once
    if (e == hipSuccess) e = mt_launch(s, k_psi_quad, dim3(64), dim3(64), a);
    return e;
}

// The same on the weight stream, once the last reader of block b's buffers
// is done; wready of the buffer marks the end.  While a graph is recorded
// the launches become a branch of it, ordered by the graph's edges instead.
static hipError_t mt_launch_psi_weights_ahead(frm_mt1d* s, int b) {
    hipError_t e = s->rec ? hipSuccess : hipStreamWaitEvent(s->wstream, s->wfree[b & 1], 0);
    s->lstream = s->wstream;
    if (e == hipSuccess) e = mt_launch_psi_weights(s, b);
    s->lstream = nullptr;
    if (e == hipSuccess && !s->rec) e = hipEventRecord(s->wready[b & 1], s->wstream);
    return e;
}

// Wavefronts that share a tile of the far pass over N0 slots: one where the
// batch has the tiles for kMemtermWaves wavefronts of four nodes per lane;
// else as many as bring its one-node tiles there, none of them with fewer
// than min_chunk slots (the history block length).
static int mt_far_split(const frm_mt1d* s, int N0) {
    if (s->ldh / (4 * 16) >= kMemtermWaves) return 1;
    const int64_t tiles = s->ldh / 16;
    int ks = 2;
    while (ks < kFarSplit && ks * tiles < kMemtermWaves && N0 / (2 * ks) >= s->min_chunk) ks *= 2;
    return ks;
}

template <typename HT, bool TAB>
static hipError_t mt_launch_far_t(frm_mt1d* s, int N0) {
    const int ks = mt_far_split(s, N0);
    const int* gprob = s->gprob_mt ? s->gprob_mt : s->gprob;
    const double* w = mt_w(s, N0 / kHistBlock);
    if (ks == 1)
        return mt_launch(s, k_mt_far<HT, TAB, false>, dim3((unsigned)(s->ldh / 256)), dim3(256),
                         (const HT*)s->hist, s->ldh, N0, w, s->ldw, gprob, s->gvalid, s->far);
    return mt_launch(s, k_mt_far<HT, TAB, true>, dim3((unsigned)(s->ldh / 16)),
                     dim3((unsigned)(64 * ks)), (const HT*)s->hist, s->ldh, N0, w, s->ldw, gprob,
                     s->gvalid, s->far);
}

// The series problems' step k (>= 2 for k_ab_series, which reads F).
static AbSeriesArgs mt_series_args(const frm_mt1d* s, int k) {
    AbSeriesArgs c;
    c.pr = s->probs;
    c.gprob = s->gprob;
    c.ldh = s->ldh;
    c.tab = s->ser_tab;
    c.choice = s->ser_choice;
    c.F = k >= 2 ? (const double*)s->hist + (size_t)(k - 2) * s->ldh : nullptr;  // step k - 1's
    c.lc1 = s->ser_lc;
    c.lc2 = s->ser_lc + (size_t)s->ser_maxL * s->ldh;
    c.lflag = s->ser_flag;
    c.part = s->part;
    c.i = k;
    c.bad = s->bad;
    return c;
}

// The far sums of the block that starts at history index N0.
static hipError_t mt_launch_far(frm_mt1d* s, int N0) {
    const bool tab = s->kind == FRM_MT_PSI;
    if (s->precision == FRM_PREC_F32C)
        return tab ? mt_launch_far_t<float, true>(s, N0) : mt_launch_far_t<float, false>(s, N0);
    return tab ? mt_launch_far_t<double, true>(s, N0) : mt_launch_far_t<double, false>(s, N0);
}

// Steps k .. k + ks - 1 of every problem, all in block b (a batch of nothing
// but fused series problems has no blocks).
static hipError_t mt_launch_steps(frm_mt1d* s, int b, int k, int ks) {
    const int fused = s->ser_waves ? s->ser_count : 0;
    const dim3 g((unsigned)(s->nprob - fused)), t((unsigned)(64 * ((s->maxN - 2 + 64 * kMtCM) / (64 * kMtCM))));
    if (s->kind == FRM_MT_AB) {
        AbStepArgs a;
        a.pr = s->probs;
        a.order = s->order;
        a.U = s->U;
        a.hist = (double*)s->hist;
        a.ldh = s->ldh;
        a.G = b > 0 ? s->far : nullptr;
        a.w = s->w;
        a.ldw = s->ldw;
        a.d0 = s->d0;
        a.cf = s->ab_cf;
        a.cal = s->ab_cal;
        a.ml = s->ab_ml;
        a.ldml = s->capacity;
        a.ser = s->part;
        a.N0 = b * kHistBlock;
        a.k0 = k;
        a.ks = ks;
        a.tau = s->tau;
        a.err = s->ab_err;
        if (fused < s->nprob) {
            const hipError_t e = mt_launch(s, k_ab_steps, g, t, a);
            if (e != hipSuccess || fused == 0) return e;
        }
        a.order = s->order + (s->nprob - fused);
        const AbSeriesArgs c = mt_series_args(s, k);
        const dim3 gs((unsigned)fused), ts((unsigned)(64 * s->ser_waves));
#define X(WAVES, BYTES) \
    if (s->ser_waves == WAVES) return mt_launch(s, k_ab_series_steps<WAVES, BYTES>, gs, ts, a, c);
        FRM_SER_CASES(X)
#undef X
        return hipErrorInvalidValue;
    }
    MtStepArgs a;
    a.pr = s->probs;
    a.order = s->order;
    a.U = s->U;
    a.hist = s->hist;
    a.ldh = s->ldh;
    a.G = b > 0 ? s->far : nullptr;
    a.w = mt_w(s, b);
    a.ldw = s->ldw;
    a.d0 = mt_d0(s, b);
    a.nprob = s->nprob;
    a.N0 = b * kHistBlock;
    a.k0 = k;
    a.ks = ks;
    a.picard = s->picard;
    const bool psi = s->kind == FRM_MT_PSI;
    if (s->precision == FRM_PREC_F32C)
        return psi ? mt_launch(s, k_mt_steps<float, true>, g, t, a)
                   : mt_launch(s, k_mt_steps<float, false>, g, t, a);
    return psi ? mt_launch(s, k_mt_steps<double, true>, g, t, a)
               : mt_launch(s, k_mt_steps<double, false>, g, t, a);
}

static void mt_free(frm_mt1d* s) {
    if (!s) return;
    (void)hipFree(s->probs);
    (void)hipFree(s->gprob);
    (void)hipFree(s->gvalid);
    (void)hipFree(s->order);
    for (auto& g : s->graphs) {
        if (g.exec) (void)hipGraphExecDestroy(g.exec);
        if (g.graph) (void)hipGraphDestroy(g.graph);
    }
    (void)hipFree(s->U);
    (void)hipFree(s->hist);
    (void)hipFree(s->part);
    (void)hipFree(s->far);
    if (s->wstream) (void)hipStreamSynchronize(s->wstream);  // the context's, shared
    for (int b = 0; b < 2; ++b) {
        if (s->wready[b]) (void)hipEventDestroy(s->wready[b]);
        if (s->wfree[b]) (void)hipEventDestroy(s->wfree[b]);
    }
    (void)hipFree(s->w);
    (void)hipFree(s->d0);
    (void)hipFree(s->psi_g);
    (void)hipFree(s->bad);
    (void)hipFree(s->ab_cf);
    (void)hipFree(s->ab_cal);
    (void)hipFree(s->ab_ml);
    (void)hipFree(s->ab_err);
    (void)hipFree(s->gprob_mt);
    (void)hipFree(s->fit_obs);
    (void)hipFree(s->fit_idx);
    (void)hipFree(s->fit_vs);
    (void)hipFree(s->fit_err);
    (void)hipFree(s->fit_dead);
    (void)hipFree(s->ser_tab);
    (void)hipFree(s->ser_choice);
    (void)hipFree(s->ser_lc);
    (void)hipFree(s->ser_flag);
    (void)hipFree(s->psi_queue);
    (void)hipFree(s->psi_qcount);
    delete s;
}

// Kind AB: kernel integrals I(d) (history weights I(lag + 1), current
// I(1)/(1-a)), the constant Thomas alpha recurrence of solve_and_check
// (MF_int_series.cpp:906-940) and the Mittag-Leffler factors of the source
// for every step, all in FP64 on the host.
static int ab_setup(frm_ctx* ctx, frm_mt1d* s, const frm_mt1d_desc* d) {
    const int cap = s->capacity;
    std::vector<double> w((size_t)s->nprob * s->ldw, 0.0), d0(s->nprob);
    std::vector<double> cf(s->ldh, 0.0), cal(s->ldh, 0.0), ml((size_t)s->nprob * cap);
    // problems with the same order and weight method share I(1..cap+1), and
    // with the same order and source the Mittag-Leffler factors
    std::map<std::tuple<double, int, int, double, int>, std::vector<double>> icache;
    std::map<std::pair<double, int>, std::vector<double>> mcache;
    for (int p = 0; p < s->nprob; ++p) {
        const frm_mt1d_problem& q = d->probs[p];
        const MtProbDev& P = s->hprobs[p];
        const double a = q.alpha, tau = d->tau;
        const int maxl = q.ab_maxl > 0 ? q.ab_maxl : 1000;
        const int maxk = q.ab_maxkiter > 0 ? q.ab_maxkiter : 1000;
        const double eps = q.ab_eps > 0 ? q.ab_eps : 1e-10;
        const auto key = std::make_tuple(a, maxl, maxk, eps, q.ab_exact ? 1 : q.ab_series ? 2 : 0);
        auto it = icache.find(key);
        if (it == icache.end()) {
            std::vector<double> I(cap + 1, 0.0);  // I[d-1] = I(d)
            if (q.ab_exact) {
                ab_exact_weights(a, tau, cap + 1, I.data());
            } else {
                // the current weight takes the problem's eps, the history
                // 1e-10 (MF_int_series.cpp:917 and the cached I of
                // MF_intF_simple); the series history needs I(1) only
                AbIntegrator cur(a, maxl, maxk, eps);
                I[0] = cur.integral(tau, tau, 0.0);
                if (!q.ab_series) {
                    AbIntegrator hist(a, maxl, maxk, 1e-10);
                    for (int dd = 2; dd <= cap + 1; ++dd) I[dd - 1] = hist.integral(dd * tau, tau, 0.0);
                }
            }
            it = icache.emplace(key, std::move(I)).first;
        }
        const std::vector<double>& I = it->second;
        const double Ii = I[0];
        for (int l = 1; l <= s->slots; ++l) w[(size_t)p * s->ldw + l - 1] = I[l];
        d0[p] = Ii / (1.0 - a);
        const int m = P.N;
        const double h = 1.0 / m;
        const double A = -(1.0 / (h * h)) - (1.0 / (2.0 * h));
        const double B = (Ii / (1.0 - a)) + (2.0 / (h * h));
        const double Cc = -(1.0 / (h * h)) + (1.0 / (2.0 * h));
        double al = 0.0;
        for (int j = 1; j < m; ++j) {
            const double den = B - A * al;
            al = Cc / den;
            cf[P.hoff + j - 1] = -1.0 / den;
            cal[P.hoff + j - 1] = -al;
        }
        const double beta = q.src == 0 ? 5.0 : (q.src == 1 ? 3.0 : 6.0);
        auto mt = mcache.find({a, q.src});
        if (mt == mcache.end()) {
            std::vector<double> v(cap);
            for (int k = 1; k <= cap; ++k)
                v[k - 1] = ml_eval(a, beta, (-a / (1.0 - a)) * std::pow(k * tau, a), 1e-20);
            mt = mcache.emplace(std::make_pair(a, q.src), std::move(v)).first;
        }
        std::copy(mt->second.begin(), mt->second.end(), ml.begin() + (size_t)p * cap);
    }
    // series history: the node-independent coefficients of every step, per
    // distinct (alpha, maxl, maxkiter, eps)
    std::vector<double> stab;
    std::vector<int> sch;
    if (s->ser_count > 0 && cap >= 2) {
        std::map<std::tuple<double, int, int, double>, std::pair<int64_t, int64_t>> scache;
        for (int p = 0; p < s->nprob; ++p) {
            MtProbDev& P = s->hprobs[p];
            if (!P.ser) continue;
            const frm_mt1d_problem& q = d->probs[p];
            const int maxk = q.ab_maxkiter > 0 ? q.ab_maxkiter : 1000;
            const double eps = q.ab_eps > 0 ? q.ab_eps : 1e-10;
            const auto key = std::make_tuple(q.alpha, P.ser_maxl, maxk, eps);
            auto it = scache.find(key);
            if (it == scache.end()) {
                const int64_t off = (int64_t)stab.size(), coff = (int64_t)sch.size();
                const int64_t rows = (int64_t)(cap - 1) * kAbSeriesRows * P.ser_maxl;
                if (off + rows > (int64_t(1) << 28))
                    return set_error(ctx, FRM_E_INVALID,
                                     "frm_mt1d_create: series coefficient tables of %.1f GB "
                                     "(capacity x ab_maxl x %d doubles per distinct order)",
                                     8.0 * (off + rows) / 1e9, kAbSeriesRows);
                stab.resize(off + rows);
                sch.resize(coff + cap - 1);
                ab_series_tables(q.alpha, d->tau, P.ser_maxl, maxk, eps, cap, stab.data() + off,
                                 sch.data() + coff);
                it = scache.emplace(key, std::make_pair(off, coff)).first;
            }
            P.ser_off = it->second.first;
            P.ser_coff = it->second.second;
        }
        // per node and series term: Lc2 and its flag read and written, and in
        // the power-series phase Lc1 too; per node the increment and the value
        s->ser_bytes.assign(cap - 1, 0.0);
        for (int p = 0; p < s->nprob; ++p) {
            const MtProbDev& P = s->hprobs[p];
            if (!P.ser) continue;
            s->ser_state_bytes += 34.0 * P.ser_maxl * (P.N - 1);
            for (int i = 2; i <= cap; ++i) {
                const bool series = sch[P.ser_coff + i - 2] == 1;
                s->ser_bytes[i - 2] += (double)(P.N - 1) * (P.ser_maxl * (series ? 34.0 : 18.0) + 16.0);
            }
        }
    }
    hipError_t e = hipSuccess;
    if (s->ser_count > 0) {
        // the full-history sums skip the series problems' groups
        std::vector<int> gm(s->ngroups);
        e = hipMemcpy(gm.data(), s->gprob, sizeof(int) * gm.size(), hipMemcpyDeviceToHost);
        for (int& g : gm)
            if (g >= 0 && s->hprobs[g].ser) g = -1;
        const size_t nl = (size_t)s->ser_maxL * s->ldh;
        if (e == hipSuccess) e = hipMalloc(&s->gprob_mt, sizeof(int) * gm.size());
        if (e == hipSuccess) e = hipMemcpy(s->gprob_mt, gm.data(), sizeof(int) * gm.size(), hipMemcpyHostToDevice);
        if (e == hipSuccess && !stab.empty()) e = hipMalloc(&s->ser_tab, sizeof(double) * stab.size());
        if (e == hipSuccess && !sch.empty()) e = hipMalloc(&s->ser_choice, sizeof(int) * sch.size());
        if (e == hipSuccess && !stab.empty())
            e = hipMemcpy(s->ser_tab, stab.data(), sizeof(double) * stab.size(), hipMemcpyHostToDevice);
        if (e == hipSuccess && !sch.empty())
            e = hipMemcpy(s->ser_choice, sch.data(), sizeof(int) * sch.size(), hipMemcpyHostToDevice);
        if (e == hipSuccess) e = hipMalloc(&s->ser_lc, sizeof(double) * 2 * nl);
        if (e == hipSuccess) e = hipMalloc(&s->ser_flag, nl);
        if (e == hipSuccess) e = hipMemset(s->ser_lc, 0, sizeof(double) * 2 * nl);
        if (e == hipSuccess) e = hipMemset(s->ser_flag, 0, nl);
        if (e == hipSuccess)
            e = hipMemcpy(s->probs, s->hprobs.data(), sizeof(MtProbDev) * s->nprob, hipMemcpyHostToDevice);
    }
    if (e == hipSuccess) e = hipMalloc(&s->ab_cf, sizeof(double) * s->ldh);
    if (e == hipSuccess) e = hipMalloc(&s->ab_cal, sizeof(double) * s->ldh);
    if (e == hipSuccess) e = hipMalloc(&s->ab_ml, sizeof(double) * ml.size());
    if (e == hipSuccess) e = hipMalloc(&s->ab_err, sizeof(double) * s->nprob);
    if (e == hipSuccess) e = hipMemcpy(s->w, w.data(), sizeof(double) * w.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(s->d0, d0.data(), sizeof(double) * d0.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(s->ab_cf, cf.data(), sizeof(double) * cf.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(s->ab_cal, cal.data(), sizeof(double) * cal.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(s->ab_ml, ml.data(), sizeof(double) * ml.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemset(s->ab_err, 0, sizeof(double) * s->nprob);
    return e == hipSuccess ? FRM_OK : check_hip(ctx, e, "mt1d AB setup");
}

extern "C" {

int frm_mt1d_create(frm_ctx* ctx, const frm_mt1d_desc* d, frm_mt1d** out) {
    FRM_REQUIRE(ctx, ctx && d && out && d->probs, "frm_mt1d_create: null argument");
    *out = nullptr;
    FRM_REQUIRE(ctx, d->nprob >= 1 && d->capacity >= 1 && d->picard >= 1 && d->tau > 0,
                "frm_mt1d_create: bad batch descriptor");
    FRM_REQUIRE(ctx, d->kind == FRM_MT_L1 || d->kind == FRM_MT_PSI || d->kind == FRM_MT_AB,
                "frm_mt1d_create: kind %d", d->kind);
    FRM_REQUIRE(ctx, d->kind != FRM_MT_AB || (d->picard == 1 && d->precision == FRM_PREC_F64),
                "frm_mt1d_create: kind AB takes picard 1 and FRM_PREC_F64");
    FRM_REQUIRE(ctx, d->precision == FRM_PREC_F64 || d->precision == FRM_PREC_F32C,
                "frm_mt1d_create: precision %d", d->precision);
    FRM_REQUIRE(ctx, d->hist_block >= 0, "frm_mt1d_create: hist_block %d", d->hist_block);
    FRM_HIP(ctx, hipSetDevice(ctx->device));
    frm_mt1d* s = new frm_mt1d();
    s->ctx = ctx;
    s->nprob = d->nprob;
    s->kind = d->kind;
    s->capacity = d->capacity;
    s->precision = d->precision;
    s->picard = d->picard;
    s->tau = d->tau;
    s->graph = d->graph != 0;
    // L1/psi: increments enter from step 3 on; AB: every increment
    const bool is_ab = d->kind == FRM_MT_AB;
    s->slots = is_ab ? d->capacity : std::max(1, d->capacity - 2);
    // weights up to the lag of a block's last step, 0 past the slots
    s->ldw = s->slots + kHistBlock;
    s->min_chunk = d->hist_block > 0 ? d->hist_block : s->min_chunk;
    std::vector<int> gp, gv;
    int64_t uoff = 0, hoff = 0;
    for (int p = 0; p < d->nprob; ++p) {
        const frm_mt1d_problem& q = d->probs[p];
        const bool ser = is_ab && q.ab_series != 0;
        const int ser_maxl = q.ab_maxl > 0 ? q.ab_maxl : 1000;
        if (q.N < 2 || q.N > kMtMaxN || !(q.alpha > 0 && q.alpha < 1) || !(q.L > 0) ||
            q.form < 0 || q.form > 2 || q.top < 0 || q.top > 2 ||
            (is_ab && (q.src < 0 || q.src > 2)) || (ser && (q.ab_exact || ser_maxl < 3))) {
            mt_free(s);
            return set_error(ctx, FRM_E_INVALID, "frm_mt1d_create: problem %d invalid (N=%d)", p,
                             q.N);
        }
        MtProbDev P{};
        P.N = q.N;
        P.form = q.form;
        P.top = q.top;
        P.bottom_cond = q.bottom_cond;
        P.src = q.src;
        P.uoff = uoff;
        P.hoff = hoff;
        P.dL = is_ab ? 1.0 / q.N : q.L / q.N;
        P.Dg = std::pow(P.dL, -2) / 1.0;  // Gamma(2 - gamma) = Gamma(1) = 1
        P.alpha = q.alpha;
        P.beta = q.beta;
        P.Da = (d->kind == FRM_MT_PSI ? std::pow(d->tau, -1) : std::pow(d->tau, -q.alpha)) /
               std::tgamma(2.0 - q.alpha);
        P.D = q.D;
        P.k = q.k;
        P.k0 = q.k0;
        P.b = q.b;
        P.top_val = q.top_val;
        P.Ev = q.Ev;
        P.Hbottom = q.Hbottom;
        P.ser = ser ? 1 : 0;
        P.ser_maxl = ser ? ser_maxl : 0;
        if (ser) {
            s->ser_count += 1;
            s->ser_maxL = std::max(s->ser_maxL, ser_maxl);
        }
        s->hprobs.push_back(P);
        const int ng = (q.N - 1 + kGroup - 1) / kGroup;
        for (int g = 0; g < ng; ++g) {
            gp.push_back(p);
            gv.push_back(std::min(kGroup, q.N - 1 - g * kGroup));
        }
        s->hnodes += q.N - 1;
        if (!ser) s->hnodes_mt += q.N - 1;
        hoff += (int64_t)ng * kGroup;
        uoff += q.N + 2;
        s->maxN = std::max(s->maxN, q.N);
    }
    s->nU = uoff;
    // whole memory-term workgroups: 64-node groups of kMemtermThreads/64 waves
    const int64_t wg_nodes = 2 * kMemtermThreads;
    s->ldh = (hoff + wg_nodes - 1) / wg_nodes * wg_nodes;
    s->ngroups = s->ldh / kGroup;
    while ((int64_t)gp.size() < s->ngroups) {
        gp.push_back(-1);
        gv.push_back(0);
    }
    const size_t esz = d->precision == FRM_PREC_F32C ? sizeof(float) : sizeof(double);
    hipError_t e = hipMalloc(&s->probs, sizeof(MtProbDev) * d->nprob);
    if (e == hipSuccess) e = hipMalloc(&s->gprob, sizeof(int) * gp.size());
    if (e == hipSuccess) e = hipMalloc(&s->gvalid, sizeof(int) * gv.size());
    if (e == hipSuccess) e = hipMalloc(&s->U, sizeof(double) * s->nU);
    if (e == hipSuccess) e = hipMalloc(&s->hist, esz * (size_t)s->slots * s->ldh);
    if (e == hipSuccess && s->ser_count > 0) e = hipMalloc(&s->part, sizeof(double) * s->ldh);
    if (e == hipSuccess && s->slots > kHistBlock)
        e = hipMalloc(&s->far, sizeof(double) * (size_t)kHistBlock * s->ldh);
    std::vector<int> order(d->nprob);
    for (int p = 0; p < d->nprob; ++p) order[p] = p;
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) {
        const MtProbDev &X = s->hprobs[x], &Y = s->hprobs[y];  // series problems last
        return X.ser != Y.ser ? X.ser < Y.ser : X.N > Y.N;
    });
    // the smallest variant of the fused series kernel that every series problem fits
#define X(WAVES, BYTES)                                                       \
    if (s->ser_count > 0 && !s->ser_waves) {                                  \
        s->ser_waves = WAVES;                                                 \
        for (const MtProbDev& P : s->hprobs)                                  \
            if (P.ser && !ser_split(P.N - 1, P.ser_maxl, WAVES, BYTES).fits)  \
                s->ser_waves = 0;                                             \
    }
    FRM_SER_CASES(X)
#undef X
    if (e == hipSuccess) e = hipMalloc(&s->order, sizeof(int) * d->nprob);
    if (e == hipSuccess)
        e = hipMemcpy(s->order, order.data(), sizeof(int) * d->nprob, hipMemcpyHostToDevice);
    // kind psi: two buffers of a block's weights, the next block's formed ahead
    const bool psi = d->kind == FRM_MT_PSI;
    const size_t wn = (size_t)d->nprob * s->ldw * (psi ? kHistBlock : 1);
    const size_t dn = (size_t)d->nprob * (psi ? kHistBlock + 2 : 1);
    if (psi) s->wsz = wn;
    if (e == hipSuccess) e = hipMalloc(&s->w, sizeof(double) * (psi ? 2 : 1) * wn);
    if (e == hipSuccess) e = hipMalloc(&s->d0, sizeof(double) * (psi ? 2 : 1) * dn);
    if (e == hipSuccess && psi)
        e = hipMalloc(&s->psi_g, sizeof(double) * 2 * (size_t)d->nprob * (s->capacity + 2));
    if (e == hipSuccess && d->kind == FRM_MT_PSI) {
        if (!ctx->aux_stream) e = hipStreamCreateWithFlags(&ctx->aux_stream, hipStreamNonBlocking);
        s->wstream = ctx->aux_stream;
        for (int b = 0; b < 2 && e == hipSuccess; ++b) {
            e = hipEventCreateWithFlags(&s->wready[b], hipEventDisableTiming);
            if (e == hipSuccess) e = hipEventCreateWithFlags(&s->wfree[b], hipEventDisableTiming);
        }
    }
    if (e == hipSuccess) e = hipMalloc(&s->bad, sizeof(int));
    if (e == hipSuccess && d->kind == FRM_MT_PSI) {
        // one entry per weight of a block, up to 2^20 per step (more set bad bit 4)
        s->psi_qcap = (int)std::min<int64_t>(
            (int64_t)d->nprob * (s->capacity + 1) * (kHistBlock + 2), (1 << 20) * kHistBlock);
        e = hipMalloc(&s->psi_queue, sizeof(int2) * s->psi_qcap);
        if (e == hipSuccess) e = hipMalloc(&s->psi_qcount, 2 * sizeof(int));
        if (e == hipSuccess) e = hipMemset(s->psi_qcount, 0, 2 * sizeof(int));
    }
    if (e != hipSuccess) {
        mt_free(s);
        return check_hip(ctx, e, "hipMalloc(mt1d)");
    }
    // L1 weights: kappa(l+2) = (l+2)^(1-a) - (l+1)^(1-a) as the reference forms
    // them (mt_minimal.cpp:926-931); psi weights are rebuilt every step.
    std::vector<double> w(psi ? 0 : wn, 0.0), d0(psi ? 0 : dn);
    for (int p = 0; p < d->nprob && !psi; ++p) {
        const double a = d->probs[p].alpha;
        d0[p] = s->hprobs[p].Da;
        if (d->kind == FRM_MT_L1)
            for (int l = 0; l < s->slots; ++l)
                w[(size_t)p * s->ldw + l] =
                    std::pow((double)(l + 2), 1.0 - a) - std::pow((double)(l + 1), 1.0 - a);
    }
    e = hipMemcpy(s->probs, s->hprobs.data(), sizeof(MtProbDev) * d->nprob, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(s->gprob, gp.data(), sizeof(int) * gp.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(s->gvalid, gv.data(), sizeof(int) * gv.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess && !psi) {
        e = hipMemcpy(s->w, w.data(), sizeof(double) * w.size(), hipMemcpyHostToDevice);
        if (e == hipSuccess)
            e = hipMemcpy(s->d0, d0.data(), sizeof(double) * d0.size(), hipMemcpyHostToDevice);
    } else if (e == hipSuccess) {
        // steps past the capacity have no weights: zeros, not stale memory
        e = hipMemset(s->w, 0, sizeof(double) * 2 * wn);
        const int gl = s->capacity + 2;
        if (e == hipSuccess) {
            hipLaunchKernelGGL(k_psi_tables, dim3((unsigned)((gl + 255) / 256), (unsigned)d->nprob),
                               dim3(256), 0, ctx->stream, s->probs, gl, s->tau, s->psi_g,
                               s->psi_g + (size_t)d->nprob * gl);
            e = hipGetLastError();
        }
        if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    }
    if (e == hipSuccess) e = hipMemset(s->bad, 0, sizeof(int));
    if (e == hipSuccess) e = hipMemset(s->hist, 0, esz * (size_t)s->slots * s->ldh);
    if (e != hipSuccess) {
        mt_free(s);
        return check_hip(ctx, e, "mt1d setup copies");
    }
    if (is_ab) {
        const int rc = ab_setup(ctx, s, d);
        if (rc) {
            mt_free(s);
            return rc;
        }
    }
    *out = s;
    return FRM_OK;
}

int frm_mt1d_destroy(frm_mt1d* s) {
    if (!s) return FRM_OK;
    (void)hipStreamSynchronize(s->ctx->stream);
    mt_free(s);
    return FRM_OK;
}

int frm_mt1d_set_state(frm_mt1d* s, const double* h_U) {
    if (!s || !h_U) return set_error(s ? s->ctx : nullptr, FRM_E_INVALID, "frm_mt1d_set_state: null");
    frm_ctx* ctx = s->ctx;
    FRM_HIP(ctx, hipMemcpyAsync(s->U, h_U, sizeof(double) * s->nU, hipMemcpyHostToDevice, ctx->stream));
    FRM_HIP(ctx, hipStreamSynchronize(ctx->stream));
    s->tstep = 1;
    s->depth = 0;
    // weights formed so far were for the old run (done: the stream waited on them)
    s->wblock = s->wahead = -1;
    if (s->psi_qcount) {
        FRM_HIP(ctx, hipMemsetAsync(s->psi_qcount, 0, 2 * sizeof(int), ctx->stream));
        FRM_HIP(ctx, hipStreamSynchronize(ctx->stream));
    }
    if (s->ab_err) {
        FRM_HIP(ctx, hipMemsetAsync(s->ab_err, 0, sizeof(double) * s->nprob, ctx->stream));
        FRM_HIP(ctx, hipStreamSynchronize(ctx->stream));
    }
    s->tt = 0.0;
    if (s->fit_err) {
        FRM_HIP(ctx, hipMemsetAsync(s->fit_err, 0, sizeof(double) * s->nprob, ctx->stream));
        FRM_HIP(ctx, hipMemsetAsync(s->fit_dead, 0, sizeof(int) * s->nprob, ctx->stream));
        FRM_HIP(ctx, hipStreamSynchronize(ctx->stream));
    }
    if (s->ser_lc) {
        const size_t nl = (size_t)s->ser_maxL * s->ldh;
        FRM_HIP(ctx, hipMemsetAsync(s->ser_lc, 0, sizeof(double) * 2 * nl, ctx->stream));
        FRM_HIP(ctx, hipMemsetAsync(s->ser_flag, 0, nl, ctx->stream));
        FRM_HIP(ctx, hipStreamSynchronize(ctx->stream));
    }
    return FRM_OK;
}

int frm_mt1d_step(frm_mt1d* s, int32_t nsteps) {
    if (!s) return set_error(nullptr, FRM_E_INVALID, "frm_mt1d_step: null solver");
    frm_ctx* ctx = s->ctx;
    FRM_REQUIRE(ctx, nsteps >= 0, "frm_mt1d_step: nsteps %d", nsteps);
    if (s->tstep - 1 + nsteps > s->capacity)
        return set_error(ctx, FRM_E_RANGE, "frm_mt1d_step: %d steps exceed capacity %d",
                         s->tstep - 1 + nsteps, s->capacity);
    const size_t esz = s->precision == FRM_PREC_F32C ? sizeof(float) : sizeof(double);
    // the next steps, at most `most` and all of one block, queued on the
    // context's stream; steps with observations go one by one between the
    // kernels that score them, steps with series problems one by one after
    // the series kernel
    auto run_some = [&](int most) -> int {
        constexpr int J = kHistBlock;
        const int off = s->kind == FRM_MT_AB ? 1 : 3;  // first step that stores an increment
        const int k = s->tstep, h = k - off, b = std::max(0, h) / J;
        auto obs = [&](int st) { return s->nobs ? s->fit_off[st] - s->fit_off[st - 1] : 0; };
        const int fcnt = obs(k);
        const bool all_fused = s->ser_waves && s->ser_count == s->nprob;  // no history sums
        int ks = std::min(most, all_fused ? kSerSteps : (b + 1) * J - h);
        if (fcnt > 0 || (s->ser_count > 0 && !s->ser_waves)) ks = 1;
        for (int i = 1; i < ks; ++i)
            if (obs(k + i) > 0) ks = i;
        FitArgs fa{};
        if (fcnt > 0) {
            fa.pr = s->probs;
            fa.nprob = s->nprob;
            fa.U = s->U;
            fa.T = s->fit_obs;
            fa.Z = s->fit_obs + s->nobs;
            fa.F = s->fit_obs + 2 * (size_t)s->nobs;
            fa.idx = s->fit_idx + s->fit_off[k - 1];
            fa.cnt = fcnt;
            fa.tt = s->tt;
            fa.tau = s->tau;
            fa.vs = s->fit_vs;
            fa.nobs = s->nobs;
            fa.err = s->fit_err;
            fa.dead = s->fit_dead;
            LaunchTimer t(ctx, FRM_K_OTHER, 0.0);
            FRM_HIP(ctx, mt_launch(s, k_fit_before, dim3((unsigned)((s->nprob + 255) / 256)),
                                   dim3(256), fa));
        }
        const bool psi_start = s->kind == FRM_MT_PSI && s->wblock != b;
        if (psi_start) {
            // the block's weights: formed during the block before, or here
            if (s->wahead == b) {
                if (s->rec) s->rec_join = true;
                else FRM_HIP(ctx, hipStreamWaitEvent(ctx->stream, s->wready[b & 1], 0));
            } else {
                LaunchTimer t(ctx, FRM_K_OTHER, 0.0);
                FRM_HIP(ctx, mt_launch_psi_weights(s, b));
            }
            s->wahead = -1;
            s->wblock = b;
        }
        if (b > 0 && h == b * J && s->ser_count < s->nprob) {
            // algorithmic bytes: the problems' own nodes
            LaunchTimer t(ctx, FRM_K_MEMTERM,
                          (double)(s->gprob_mt ? s->hnodes_mt : s->hnodes) *
                              ((double)h * esz + J * sizeof(double)));
            FRM_HIP(ctx, mt_launch_far(s, h));
        }
        // the next block's weights overlap this block's steps unless launches
        // are timed one by one
        if (psi_start && s->wstream && !ctx->timing_mask && (b + 1) * J + off <= s->capacity) {
            FRM_HIP(ctx, mt_launch_psi_weights_ahead(s, b + 1));
            s->wahead = b + 1;
        }
        if (s->kind == FRM_MT_AB && s->ser_count > 0 && !s->ser_waves && k >= 2) {
            const AbSeriesArgs c = mt_series_args(s, k);
            LaunchTimer t(ctx, FRM_K_MEMTERM, s->ser_bytes.empty() ? 0.0 : s->ser_bytes[k - 2]);
            FRM_HIP(ctx, mt_launch(s, k_ab_series, dim3((unsigned)((s->ldh + 255) / 256)), dim3(256),
                                   c));
        }
        {
            // fused series problems: their accumulators in and out, once
            const bool fused = s->ser_waves != 0;
            LaunchTimer t(ctx, fused ? FRM_K_MEMTERM : FRM_K_SWEEP1D, fused ? s->ser_state_bytes : 0.0);
            FRM_HIP(ctx, mt_launch_steps(s, b, k, ks));
        }
        // once the block's last steps are through, its buffers are free
        if (s->wstream && !s->rec) FRM_HIP(ctx, hipEventRecord(s->wfree[b & 1], ctx->stream));
        s->tstep = k + ks;
        s->depth = std::max(0, s->tstep - off);
        if (fcnt > 0) {
            LaunchTimer t(ctx, FRM_K_OTHER, 0.0);
            FRM_HIP(ctx, mt_launch(s, k_fit_after, dim3((unsigned)((s->nprob + 255) / 256)),
                                   dim3(256), fa));
        }
        for (int i = 0; i < ks; ++i) s->tt += s->tau;
        return FRM_OK;
    };
    const int goal = s->tstep + nsteps;
    // Graph mode: the launches of up to kGraphSteps steps are recorded,
    // matched with the graph built for the same kernel sequence (instantiated
    // once), the nodes get these steps' arguments and grids
    // (hipGraphExecKernelNodeSetParams) and the graph is launched once.  Runs
    // of steps differ only in arguments and grids (depth, slots), so a run
    // uses a handful of graphs.  Not while per-launch timing is on.
    if (!s->graph || ctx->timing_mask != 0) {
        while (s->tstep < goal)
            if (int rc = run_some(goal - s->tstep)) return rc;
        // a synchronisation of the context's stream also covers the weights
        // formed ahead
        if (s->wahead >= 0) FRM_HIP(ctx, hipStreamWaitEvent(ctx->stream, s->wready[s->wahead & 1], 0));
        return FRM_OK;
    }
    std::vector<KRec> recs;
    std::vector<void*> ptrs;
    struct At {
        int tstep, depth, wblock, wahead;
        double tt;
    };
    auto at = [&] { return At{s->tstep, s->depth, s->wblock, s->wahead, s->tt}; };
    auto back = [&](const At& t) {
        s->tstep = t.tstep;
        s->depth = t.depth;
        s->wblock = t.wblock;
        s->wahead = t.wahead;
        s->tt = t.tt;
    };
    while (s->tstep < goal) {
        recs.clear();
        const At start = at();
        const int stop = std::min(goal, s->tstep + kGraphSteps);
        // record steps until the run is full; a launch that fails is taken
        // back with its steps (the solver stays where it was before them)
        // and ends the run
        int rc = FRM_OK;
        s->rec = &recs;
        s->rec_join = false;
        while (s->tstep < stop) {
            const size_t mark = recs.size();
            const At t = at();
            rc = run_some(stop - s->tstep);
            if (rc) {
                recs.resize(mark);
                back(t);
                break;
            }
        }
        s->rec = nullptr;
        // none of the run's steps is launched: the solver goes back to its start
        auto unrun = [&](int code) {
            back(start);
            return code;
        };
        if (!recs.empty()) {
            StepGraph* g = nullptr;
            for (auto& c : s->graphs) {
                if (c.funcs.size() != recs.size()) continue;
                bool same = true;
                for (size_t i = 0; i < recs.size() && same; ++i)
                    same = c.funcs[i] == recs[i].func && c.tags[i] == recs[i].join * 2 + recs[i].branch;
                if (same) {
                    g = &c;
                    break;
                }
            }
            ptrs.resize(16 * recs.size());
            auto params = [&](size_t i) {
                void** pp = ptrs.data() + 16 * i;
                recs[i].ptrs(pp);
                hipKernelNodeParams q{};
                q.blockDim = recs[i].block;
                q.extra = nullptr;
                q.func = const_cast<void*>(recs[i].func);
                q.gridDim = recs[i].grid;
                q.kernelParams = pp;
                q.sharedMemBytes = 0;
                return q;
            };
            if (!g) {
                // Edges: the launches in order.  Weights formed ahead start
                // after what was launched before them (the last reader of
                // their buffers among it) and after the weights before them
                // (they share the fallback queue); the block that reads them
                // starts when they are done.
                StepGraph ng;
                FRM_HIP(ctx, hipGraphCreate(&ng.graph, 0));
                hipError_t e = hipSuccess;
                hipGraphNode_t main_last = nullptr, br_last = nullptr;
                for (size_t i = 0; i < recs.size() && e == hipSuccess; ++i) {
                    const KRec& r = recs[i];
                    hipGraphNode_t dep[2];
                    size_t nd = 0;
                    if (main_last) dep[nd++] = main_last;
                    if ((r.branch || r.join) && br_last) dep[nd++] = br_last;
                    hipKernelNodeParams q = params(i);
                    hipGraphNode_t node = nullptr;
                    e = hipGraphAddKernelNode(&node, ng.graph, nd ? dep : nullptr, nd, &q);
                    (r.branch ? br_last : main_last) = node;
                    ng.nodes.push_back(node);
                    ng.funcs.push_back(r.func);
                    ng.tags.push_back(r.join * 2 + r.branch);
                }
                if (e == hipSuccess) e = hipGraphInstantiate(&ng.exec, ng.graph, nullptr, nullptr, 0);
                if (e != hipSuccess) {
                    if (ng.exec) (void)hipGraphExecDestroy(ng.exec);
                    (void)hipGraphDestroy(ng.graph);
                    return unrun(check_hip(ctx, e, "frm_mt1d_step: step graph"));
                }
                s->graphs.push_back(ng);
                g = &s->graphs.back();
            } else {
                for (size_t i = 0; i < recs.size(); ++i) {
                    hipKernelNodeParams q = params(i);
                    const hipError_t e = hipGraphExecKernelNodeSetParams(g->exec, g->nodes[i], &q);
                    if (e != hipSuccess) return unrun(check_hip(ctx, e, "frm_mt1d_step: node update"));
                }
            }
            const hipError_t e = hipGraphLaunch(g->exec, ctx->stream);
            if (e != hipSuccess) return unrun(check_hip(ctx, e, "frm_mt1d_step: graph launch"));
        }
        if (rc) return rc;
    }
    // the weight buffers' events, for steps launched eagerly later: every
    // graph so far is ahead of them on the context's stream
    if (s->wstream)
        for (int b = 0; b < 2; ++b) {
            FRM_HIP(ctx, hipEventRecord(s->wfree[b], ctx->stream));
            FRM_HIP(ctx, hipEventRecord(s->wready[b], ctx->stream));
        }
    return FRM_OK;
}

int frm_mt1d_get_state(frm_mt1d* s, double* h_U) {
    if (!s || !h_U) return set_error(s ? s->ctx : nullptr, FRM_E_INVALID, "frm_mt1d_get_state: null");
    frm_ctx* ctx = s->ctx;
    int bad = 0;
    FRM_HIP(ctx, hipMemcpyAsync(h_U, s->U, sizeof(double) * s->nU, hipMemcpyDeviceToHost, ctx->stream));
    FRM_HIP(ctx, hipMemcpyAsync(&bad, s->bad, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
    FRM_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (bad & 1)
        return set_error(ctx, FRM_E_STATE,
                         "frm_mt1d: a psi weight was not finite after the adaptive quadrature "
                         "fallback of calc_int (mt_psi_caputo.cpp:736-737)");
    if (bad & 4)
        return set_error(ctx, FRM_E_STATE,
                         "frm_mt1d: more psi weight series than the fallback queue holds (2^20) "
                         "were not finite in one step");
    if (bad & 2)
        return set_error(ctx, FRM_E_STATE,
                         "frm_mt1d: a term of the AB power series was not finite with ab_maxl "
                         "above 4096, the longest series whose sorted-pyramid recount "
                         "(MF_int_series.cpp:600-609) this path holds in LDS");
    return FRM_OK;
}

int frm_mt1d_ab_error(frm_mt1d* s, double* out) {
    if (!s || !out) return set_error(s ? s->ctx : nullptr, FRM_E_INVALID, "frm_mt1d_ab_error: null");
    frm_ctx* ctx = s->ctx;
    FRM_REQUIRE(ctx, s->kind == FRM_MT_AB, "frm_mt1d_ab_error: batch kind %d is not AB", s->kind);
    std::vector<double> e(s->nprob);
    FRM_HIP(ctx, hipMemcpyAsync(e.data(), s->ab_err, sizeof(double) * s->nprob, hipMemcpyDeviceToHost,
                                ctx->stream));
    FRM_HIP(ctx, hipStreamSynchronize(ctx->stream));
    const int steps = s->tstep - 1;
    for (int p = 0; p < s->nprob; ++p)
        out[p] = steps > 0 ? e[p] / ((s->hprobs[p].N + 1.0) * steps) : 0.0;
    return FRM_OK;
}

int frm_mt1d_set_observations(frm_mt1d* s, int32_t nobs, const double* T, const double* Z,
                              const double* F) {
    if (!s) return set_error(nullptr, FRM_E_INVALID, "frm_mt1d_set_observations: null solver");
    frm_ctx* ctx = s->ctx;
    FRM_REQUIRE(ctx, nobs >= 0 && (nobs == 0 || (T && Z && F)),
                "frm_mt1d_set_observations: bad arguments");
    (void)hipFree(s->fit_obs);
    (void)hipFree(s->fit_idx);
    (void)hipFree(s->fit_vs);
    s->fit_obs = s->fit_vs = nullptr;
    s->fit_idx = nullptr;
    s->nobs = 0;
    s->fit_off.clear();
    // which step each observation falls in: the reference's loop variable
    // tt starts at 0 and grows by tau per step; step k covers [tt, tt + tau)
    std::vector<std::vector<int>> per(s->capacity + 1);
    double tt = 0.0;
    for (int k = 1; k <= s->capacity; ++k) {
        for (int o = 0; o < nobs; ++o)
            if ((T[o] >= tt) && (T[o] < (tt + s->tau))) per[k].push_back(o);
        tt += s->tau;
    }
    std::vector<int> idx;
    s->fit_off.assign(s->capacity + 1, 0);
    for (int k = 1; k <= s->capacity; ++k) {
        idx.insert(idx.end(), per[k].begin(), per[k].end());
        s->fit_off[k] = (int)idx.size();
    }
    hipError_t e = hipSuccess;
    if (!s->fit_err) {
        e = hipMalloc(&s->fit_err, sizeof(double) * s->nprob);
        if (e == hipSuccess) e = hipMalloc(&s->fit_dead, sizeof(int) * s->nprob);
    }
    if (e == hipSuccess) e = hipMemset(s->fit_err, 0, sizeof(double) * s->nprob);
    if (e == hipSuccess) e = hipMemset(s->fit_dead, 0, sizeof(int) * s->nprob);
    if (nobs > 0) {
        std::vector<double> obs((size_t)3 * nobs);
        std::copy(T, T + nobs, obs.begin());
        std::copy(Z, Z + nobs, obs.begin() + nobs);
        std::copy(F, F + nobs, obs.begin() + 2 * (size_t)nobs);
        if (e == hipSuccess) e = hipMalloc(&s->fit_obs, sizeof(double) * obs.size());
        if (e == hipSuccess) e = hipMalloc(&s->fit_idx, sizeof(int) * std::max<size_t>(1, idx.size()));
        if (e == hipSuccess) e = hipMalloc(&s->fit_vs, sizeof(double) * (size_t)nobs * s->nprob);
        if (e == hipSuccess)
            e = hipMemcpy(s->fit_obs, obs.data(), sizeof(double) * obs.size(), hipMemcpyHostToDevice);
        if (e == hipSuccess && !idx.empty())
            e = hipMemcpy(s->fit_idx, idx.data(), sizeof(int) * idx.size(), hipMemcpyHostToDevice);
        if (e == hipSuccess) e = hipMemset(s->fit_vs, 0, sizeof(double) * (size_t)nobs * s->nprob);
        s->nobs = nobs;
    }
    return e == hipSuccess ? FRM_OK : check_hip(ctx, e, "frm_mt1d_set_observations");
}

int frm_mt1d_fit_error(frm_mt1d* s, double* out) {
    if (!s || !out) return set_error(s ? s->ctx : nullptr, FRM_E_INVALID, "frm_mt1d_fit_error: null");
    frm_ctx* ctx = s->ctx;
    FRM_REQUIRE(ctx, s->fit_err != nullptr, "frm_mt1d_fit_error: no observations were set");
    std::vector<double> e(s->nprob);
    FRM_HIP(ctx, hipMemcpyAsync(e.data(), s->fit_err, sizeof(double) * s->nprob, hipMemcpyDeviceToHost,
                                ctx->stream));
    FRM_HIP(ctx, hipStreamSynchronize(ctx->stream));
    for (int p = 0; p < s->nprob; ++p) out[p] = std::isfinite(e[p]) ? e[p] : 1e300;
    return FRM_OK;
}

int frm_mt1d_hist_block(const frm_mt1d* s, int32_t* len) {
    if (!s || !len) return set_error(nullptr, FRM_E_INVALID, "frm_mt1d_hist_block: null");
    *len = s->min_chunk;
    return FRM_OK;
}

int frm_mt1d_tstep(const frm_mt1d* s, int32_t* tstep) {
    if (!s || !tstep) return set_error(nullptr, FRM_E_INVALID, "frm_mt1d_tstep: null");
    *tstep = s->tstep;
    return FRM_OK;
}

}  // extern "C"

extern "C" int frm_diag_psi_kb_quad(frm_ctx* ctx, int32_t n, const double* h_cases,
                                    double* h_out) {
    FRM_REQUIRE(ctx, ctx && h_cases && h_out && n > 0 && n <= (1 << 20),
                "frm_diag_psi_kb_quad: bad arguments (1 <= n <= 2^20)");
    for (int32_t i = 0; i < n; ++i) {
        const double* r = h_cases + 6 * (int64_t)i;
        FRM_REQUIRE(ctx, std::isfinite(r[2]) && std::isfinite(r[3]) && std::isfinite(r[4]) &&
                             r[1] > 0.0 && r[0] >= 0.0 && r[0] < 1.0 && r[2] <= r[3],
                    "frm_diag_psi_kb_quad: case %d: need 0 <= alpha < 1, beta > 0, finite "
                    "t0 <= t1 and gtj", i);
    }
    double *dc = nullptr, *dout = nullptr;
    hipError_t e = hipMalloc(&dc, sizeof(double) * 6 * (size_t)n);
    if (e == hipSuccess) e = hipMalloc(&dout, sizeof(double) * (size_t)n);
    if (e == hipSuccess)
        e = hipMemcpyAsync(dc, h_cases, sizeof(double) * 6 * (size_t)n, hipMemcpyHostToDevice,
                           ctx->stream);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(frm::k_diag_psi_kb_quad, dim3((unsigned)((n + 63) / 64)), dim3(64), 0,
                           ctx->stream, dc, n, dout);
        e = hipGetLastError();
    }
    if (e == hipSuccess)
        e = hipMemcpyAsync(h_out, dout, sizeof(double) * (size_t)n, hipMemcpyDeviceToHost,
                           ctx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    (void)hipFree(dc);
    (void)hipFree(dout);
    return e == hipSuccess ? FRM_OK : check_hip(ctx, e, "frm_diag_psi_kb_quad");
}
