// 2D locally-one-dimensional fractional solver (the hot path of
// TG_solver::calc_step, fr_d_t_g_2d.cpp:2552-2718, dt_alg = 0, g(t) = t).
//
// Per step n the reference, for every row j, forms Om (3306-3492) with the
// full history sum over s = n-1..0, builds Al/Bt (3267-3304, 3494-3553) and
// back-substitutes (2548-2550); then the same for every column with the
// extra half-step term kb(n,1,0,1/2)*(C_n - C_{n+1/2}) (3430-3436).  Its
// OpenCL version launches Om, Al, Bt and U separately, with Al/Bt/U on one
// work-item per system and a Finish() after each launch.
//
// Here one step is two or three launches on one stream:
//   1. memterm, both half-step history sums (rows use kb(s,1/2,0,1), columns
//      kb(s,1,0,1)).  Where they depend on the lag n-s only (g(t) = t) the
//      full-history forms sum the settled past once per block of steps
//      (frm_blockhist.hip) and the row kernel adds the newest slots; the
//      sum-of-exponentials recurrences, the blocked Toeplitz parts
//      (frm_mfma.hip) and the other series run every step;
//   2. rows: one to four wavefronts per row -- RHS assembly, Thomas forward
//      and back substitution (chunked over lanes, scan seeds), boundary
//      nodes; the half-step field goes to a buffer of its own, so that C_n
//      stays for step 3;
//   3. cols: the same per column, plus the push of Delta_n = C_{n+1} - C_n
//      into the history store.
// With g(t) = t and a time-independent operator the tridiagonal matrices do
// not change between steps, so their Thomas alpha coefficients are computed
// once on the host in FP64, with the reference's formula and order.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "frm_blockhist.hpp"
#include "frm_gpow.hpp"
#include "frm_history.hpp"
#include "frm_iaibk.hpp"
#include "frm_stream.hpp"
#include "frm_mfma.hpp"
#include "frm_wavescan.hpp"
#include "frm_soe.hpp"
#include "frm_weights.hpp"

namespace frm {
// Launch shape of a sweep: chunk length CM, wavefronts per line W, and for the
// columns the lines per workgroup LW.
struct SweepShape {
    int cm = 0, w = 1, lw = 0;
};
}  // namespace frm

struct frm_lod2d {
    frm_ctx* ctx = nullptr;
    int sN = 0, M = 0, ld = 0;
    int NX = 0, NY = 0;  // interior nodes per row / per column
    int capacity = 0;
    int tstep = 0;
    double alpha = 0, tau = 0, sigma = 0, C1 = 0, S = 0;
    double sg = 0;                  // sigma / tau
    double kr0 = 0, kc0 = 0, kch = 0;  // current-step weights
    frm_hist* hist = nullptr;
    double* C = nullptr;       // state, reference layout
    double* crhs = nullptr;    // the columns' right-hand sides, interior nodes, compact order
    double* w = nullptr;       // [2][ldw] lag-indexed history weights, 0 past the capacity
    int ldw = 0;               // capacity + kHistBlock
    double* far = nullptr;     // far sums of the current block: [2][kHistBlock][hist->ld]
                               // (full history) or [2][kSoeBlock][hist->ld] (SOE, FP64 states)
    bool small = false;        // the grid takes k_lod_small, not the sweeps
    int ring = 0;              // slots of an increment ring (0: the whole history is stored)
    double* rcoef = nullptr;   // rows:    a, f, al interleaved per line (load_coefs)
    double* ccoef = nullptr;   // columns: the same
    bool rsame = false, csame = false;  // one line's coefficients serve all
    frm::SweepShape rsh, csh;  // launch shapes of the row / column sweeps
    int precision = FRM_PREC_F64;
    std::vector<double> hw;    // host copy: kr0, kc0, kch, then [2][capacity] weights
    // sum-of-exponentials form
    int soe_L = 0, soe_f32 = 0;
    double soe_err = 0.0;
    void* soe_H = nullptr;     // [L][ld] mode states (FP32 or FP64)
    double* soe_q = nullptr;   // [L] (FP32 states)
    double* soe_c = nullptr;   // [2][L]
    double* soe_tab = nullptr; // FP64 states: per mode the block's factors (k_soe_block)
    double soe_w1r = 0.0, soe_w1c = 0.0;  // exact lag-1 weights
    // FRM_PREC_BINOMIAL: moments [2][terms][ld] and per-step coefficient tables
    int bin_terms = 0;
    double bin_Da = 0.0;
    double* bin_H = nullptr;
    double* bin_upd = nullptr;  // [capacity-1][terms]
    double* bin_er = nullptr;
    double* bin_ec = nullptr;
    int* bin_cnt = nullptr;     // [capacity-1][4]
    // restricted summation: lags beyond trunc_L are not read (weights past a
    // direction's own cut-off are zero)
    int trunc_L = 0;
    // blocked MFMA form: FP32 increments in hist, BF16-exact weight parts,
    // far part of the current 64-step block
    void* atab = nullptr;      // weight-operand fragments (atab_build)
    int atab_chunks = 0;
    int mfma_nprod = 6;        // 3 (two parts) or 6 (three parts)
    int far_slices = 8;        // node slices of a block's far product (1 to 64)
    float* F = nullptr;        // [2][128][ld]: far parts of this block and the next
    float* G = nullptr;        // [2][kMidBlock][ld] mid part of the current sub-block
    // g(t) = t^p (g_func 3): the weights and the sweeps' Thomas coefficients
    // are rebuilt every step
    int g_func = 0;
    double g_pow = 1.0, int_err = 1e-6, Da = 0.0;
    double* lineAB = nullptr;  // off-diagonals per line: rows A, B [M-1][NX], cols A, B [sN-1][NY]
    int* flag = nullptr;       // set when a weight series reached its safety bound
    // FRM_PREC_IAIBK: per-node coefficient slots [2][slots][MAXAK][ld] and
    // both directions' operation plans
    double* ia_H = nullptr;
    frm::IaOp* ia_ops[2] = {nullptr, nullptr};
    double* ia_vals[2] = {nullptr, nullptr};
    std::vector<int> ia_off[2];
    int ia_slots = 0;
    double ia_ak[frm::kIaMaxAk] = {};
    double ia_scale = 0.0;     // Da tau^(1-alpha) / (1-alpha)
};

namespace frm {

// ------------------------------------------------------------- kernels
// A line of n unknowns is split into NL = 64 W chunks of CM elements, one
// per lane of the W wavefronts that share the line (W = 1, 2 or 4: the
// number of lanes that run the parallel scan levels before each lane's
// sequential Thomas replay of CM elements).
//
// Coefficient layout: for line L and array c (0: a, 1: f, 2: al), element
// e = g*CM + k of the line (chunk g = 64 wl + lane, position k) is stored at
//   ((L*3 + c)*CM + k)*NL + g,
// so that the k-th load of a coefficient is NL consecutive doubles.  Where all
// lines of a direction have the same coefficients (no velocity across it), one
// line's are stored and L is 0 for all: 24 bytes per node less in each sweep
// (1531 x 1531 AB model, MFMA form, both sweeps: 94.5 -> 78.9 us per step).
// Right-hand sides are staged through LDS: formed in element order
// (consecutive lanes, consecutive nodes), written to LDS at e + e/CM
// (chunk-major with one pad double per chunk, so that the chunk reads
// g*(CM+1) + k spread over the banks), read back per chunk.
template <int CM, int W>
__device__ inline void load_coefs(const double* coef, int line, int g, double (&a)[CM],
                                  double (&f)[CM], double (&al)[CM]) {
    constexpr int NL = kWave * W;
#pragma unroll
    for (int k = 0; k < CM; ++k) {
        a[k] = coef[((int64_t)(line * 3 + 0) * CM + k) * NL + g];
        f[k] = coef[((int64_t)(line * 3 + 1) * CM + k) * NL + g];
        al[k] = coef[((int64_t)(line * 3 + 2) * CM + k) * NL + g];
    }
}

// Where the row kernel takes its memory term from.
enum RowSrc {
    kRowPart,    // FP64 partial sums of both targets, formed by an earlier launch
    kRowNear64,  // FP64 far sums of the block + its newest FP64 slots
    kRowNear32,  // FP64 far sums of the block + its newest FP32 slots
    kRowNearMx,  // FP32 far and mid sums + the newest FP32 slots
};

// The newest slots s0 .. s0 + cnt - 1 of a block (cnt = n - s0) and the far
// sums of step n for both targets.
struct NearArgs {
    const void* hist;
    int64_t ld;
    int s0, cnt, mask;     // slot s is stored at s & mask (-1: the whole history)
    const double* w;       // lag-indexed weights [2][ldw]
    int ldw;
    const void *f0, *f1;   // far sums of the row / column target, or null
    const float *m0, *m1;  // kRowNearMx: mid sums, or null
};

struct RowArgs {
    double* C;
    double* crhs;        // out: the columns' right-hand sides
    const double* coef;  // interleaved, see load_coefs
    int same;            // one line's coefficients serve all
    const double* part;  // kRowPart: partial sums [nch][2][ldh]
    int64_t ldh;
    int nch;
    int ld, lines, n, NX;
    double negsk, S_half, sg, b0, al1;
    double col_negsk, kch;  // the columns' -sg kc0 and half-step weight
    NearArgs near;
};

// Both targets' sums of nodes q0 + r NL + g (r < CM, clamped to the line's
// last): far sums, then the newest slots oldest first, all in FP64.  Reading
// them here instead of in a kernel of their own saves that launch and, per
// node, the row target's sum written and read back.
template <typename HT, typename FT, int CM, int NL>
__device__ __forceinline__ void near_sums(const NearArgs& a, int64_t q0, int g, int n,
                                          double (&ts)[CM], double (&tc)[CM]) {
    int e[CM];
#pragma unroll
    for (int r = 0; r < CM; ++r) {
        e[r] = min(r * NL + g, n - 1);
        ts[r] = tc[r] = 0.0;
    }
    if (a.f0) {
        const FT* __restrict__ f0 = static_cast<const FT*>(a.f0) + q0;
        const FT* __restrict__ f1 = static_cast<const FT*>(a.f1) + q0;
#pragma unroll
        for (int r = 0; r < CM; ++r) {
            ts[r] = f0[e[r]];
            tc[r] = f1[e[r]];
        }
    }
    if constexpr (sizeof(FT) == 4) {
        if (a.m0) {
#pragma unroll
            for (int r = 0; r < CM; ++r) {
                ts[r] += (double)a.m0[q0 + e[r]];
                tc[r] += (double)a.m1[q0 + e[r]];
            }
        }
    }
    constexpr int U = CM >= 16 ? 1 : 16 / CM;  // slots whose loads go out together
    const HT* __restrict__ h = static_cast<const HT*>(a.hist) + q0;
    const double* __restrict__ w0 = a.w + a.cnt - 1;  // the oldest near slot's lag
    const double* __restrict__ w1 = w0 + a.ldw;
    auto batch = [&](int u, int m) {  // slots u .. u + m - 1, m <= U
        HT x[U][CM];
#pragma unroll
        for (int v = 0; v < U; ++v) {
            if (v >= m) break;
            const int64_t at = (int64_t)((a.s0 + u + v) & a.mask) * a.ld;
#pragma unroll
            for (int r = 0; r < CM; ++r) x[v][r] = h[at + e[r]];
        }
#pragma unroll
        for (int v = 0; v < U; ++v) {
            if (v >= m) break;
            const double p = w0[-(u + v)], q = w1[-(u + v)];
#pragma unroll
            for (int r = 0; r < CM; ++r) {
                ts[r] += p * (double)x[v][r];
                tc[r] += q * (double)x[v][r];
            }
        }
    };
    // The last batch makes one trip to memory, not one per slot.  Whole batches
    // without its tests are faster where the registers allow them: 4 elements
    // per lane (512 x 512 FP64 rows: 9.5 us, 9.8 with tests); from 6 on they cost
    // a wavefront per SIMD (1531 x 1531, 6 elements, up to 15 slots: 37.9 us, 31.1
    // with tests).
    int u = 0;
    if (CM < 6)
        for (; u + U <= a.cnt; u += U) batch(u, U);
    for (; u < a.cnt; u += U) batch(u, a.cnt - u);
}

// Rows: 4 wavefronts per workgroup, 4/W lines.  A lane holds its nodes' state and
// column sums over the solve, so that it can form the columns' right-hand
// sides itself: the columns read one array where they read the field after the
// rows and the column sums (8 bytes per node written and 8 read less; 1024 x
// 1024, MFMA form, both sweeps: 40.9 -> 38.7 us per step).
template <int CM, int W, int SRC>
__global__ __launch_bounds__(256) void k_lod_rows(RowArgs p) {
    constexpr int S = CM + 1;
    constexpr int LPB = 4 / W;
    constexpr int NL = kWave * W;
    __shared__ double lds[LPB][NL * S];
    __shared__ LineShare<W> share[LPB];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int li = wv / W, wl = wv % W;
    const int line = blockIdx.x * LPB + li;
    const bool live = line < p.lines;  // uniform per line; dead lines still reach the barriers
    const int n = p.n;
    const int g = wl * kWave + lane;
    const int e0 = g * CM;
    double* buf = lds[li];
    const int64_t qbase = (int64_t)line * p.NX;
    double* Crow = p.C + (int64_t)(line + 1) * p.ld;
    // The coefficients do not depend on the staging: their loads go out
    // first and overlap the state loads (up to 8 elements per lane; above that
    // the registers would spill).
    constexpr bool kEarly = CM <= 8;
    double a[CM], f[CM], al[CM], v[CM], u[CM], tc[CM];
#pragma unroll
    for (int k = 0; k < CM; ++k) a[k] = f[k] = al[k] = v[k] = u[k] = tc[k] = 0.0;
    if (kEarly && live) load_coefs<CM, W>(p.coef, p.same ? 0 : line, g, a, f, al);
    if (live) {
        // om in element order: C_n and the history sum.  Every load is
        // issued before the first store (clamped, unguarded indices; the
        // pointers do not alias), so the row costs one memory latency
        // instead of one per element group.
        const double* __restrict__ cr = Crow + 1;
        double ts[CM];
#pragma unroll
        for (int r = 0; r < CM; ++r) u[r] = cr[min(r * NL + g, n - 1)];
        if constexpr (SRC == kRowPart) {
            // the first partial-sum chunk is loaded with the state (0 + p0 =
            // p0 exactly, so the sum order is unchanged); further chunks follow
            const double* __restrict__ pt = p.part + qbase;
            const bool any = p.nch > 0;
#pragma unroll
            for (int r = 0; r < CM; ++r) {
                const int e = min(r * NL + g, n - 1);
                ts[r] = any ? pt[e] : 0.0;
                tc[r] = any ? pt[p.ldh + e] : 0.0;
            }
            for (int c = 1; c < p.nch; ++c) {
                const double* __restrict__ pc = pt + (int64_t)c * 2 * p.ldh;
                double x[CM], y[CM];
#pragma unroll
                for (int r = 0; r < CM; ++r) {
                    const int e = min(r * NL + g, n - 1);
                    x[r] = pc[e];
                    y[r] = pc[p.ldh + e];
                }
#pragma unroll
                for (int r = 0; r < CM; ++r) {
                    ts[r] += x[r];
                    tc[r] += y[r];
                }
            }
        } else if constexpr (SRC == kRowNear64) {
            near_sums<double, double, CM, NL>(p.near, qbase, g, n, ts, tc);
        } else if constexpr (SRC == kRowNear32) {
            near_sums<float, double, CM, NL>(p.near, qbase, g, n, ts, tc);
        } else {
            near_sums<float, float, CM, NL>(p.near, qbase, g, n, ts, tc);
        }
#pragma unroll
        for (int r = 0; r < CM; ++r) {
            const int e = r * NL + g;
            if (e < n) {
                double om = p.negsk * u[r];
                om += p.S_half;
                om += p.sg * ts[r];
                buf[e + e / CM] = om;
            }
        }
    }
    __syncthreads();
    if (live) {
        if (!kEarly) load_coefs<CM, W>(p.coef, p.same ? 0 : line, g, a, f, al);
#pragma unroll
        for (int k = 0; k < CM; ++k) v[k] = e0 + k < n ? buf[g * S + k] : 0.0;
    }
    const double un = line_solve_mw<CM, W>(a, f, al, v, e0, n, p.b0, lane, wl, &share[li], live);
    if (live) {
#pragma unroll
        for (int k = 0; k < CM; ++k)
            if (e0 + k < n) buf[g * S + k] = v[k];
    }
    __syncthreads();
    if (live) {
        double* __restrict__ cq = p.crhs + qbase;
#pragma unroll
        for (int r = 0; r < CM; ++r) {
            const int e = r * NL + g;
            if (e < n) {
                const double x = buf[e + e / CM];  // the field after the rows
                const double t = tc[r] + p.kch * (u[r] - x);
                double om = p.col_negsk * x;
                om += p.S_half;
                om += p.sg * t;
                cq[e] = om;
            }
        }
        // the boundary nodes, which neither sweep reads, go to the state
        if (g == 0) {
            Crow[0] = p.al1 * v[0] + p.b0;
            Crow[n + 1] = un;
            Crow[n + 2] = un;
        }
    }
}

struct ColArgs {
    double* C;           // in: C_n; out: C_{n+1}
    const double* rhs;   // right-hand sides, compact node order
    double* slot;        // history slot for Delta_n (compact node order)
    float* slotf;        // FP32 history slot instead of slot when non-null
    const double* coef;  // interleaved, see load_coefs
    int same;            // one line's coefficients serve all
    int ld, lines, n, NX;
    int groups;          // column groups of LW lines
    double b0, al1;
};

// Column lines per workgroup LW: a row segment of LW columns is one contiguous
// piece of the state and right-hand sides, so wider is better for the memory,
// but the workgroups of one chip's worth of lines get fewer; timed at creation.
// A workgroup has 256 threads or more and at most what its registers allow.
constexpr int kColWidths[] = {1, 2, 4, 8};
__host__ __device__ constexpr bool col_fits(int CM, int W, int LW) {
    return LW * W >= 4 && LW * W <= (CM >= 24 ? 4 : CM >= 12 ? 8 : 16) && (LW > 1 || CM >= 24);
}

template <int CM, int W, int LW>
__global__ __launch_bounds__((LW * kWave * W), CM == 12 ? 4 : 1) void k_lod_cols(ColArgs p) {
    constexpr int kColW = LW;
    constexpr int S = CM + 1;
    constexpr int NL = kWave * W;
    __shared__ double lds[kColW][NL * S];
    __shared__ LineShare<W> share[kColW];
    // Workgroups are dealt to the 8 XCDs round-robin (b -> XCD b % 8); the
    // group order below gives each XCD a contiguous run of column groups so
    // that neighbouring groups, which share cache lines, share an L2.
    const int per = gridDim.x / 8;
    const int grp = (blockIdx.x % 8) * per + blockIdx.x / 8;
    if (grp >= p.groups) return;  // whole workgroup, before any barrier
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int li = wv / W, wl = wv % W;
    const int line = grp * kColW + li;
    const bool live = line < p.lines;
    const int n = p.n;
    const int g = wl * kWave + lane;
    const int e0 = g * CM;
    const int64_t ld = p.ld;
    // staging map: column tc of the group, rows tr + NL r
    const int tc = threadIdx.x % kColW, tr = threadIdx.x / kColW;
    const int tline = grp * kColW + tc;
    const bool tlive = tline < p.lines;
    // coefficient loads first (they overlap the staging loads); the staging
    // thread keeps its C_n values for the increment push and is the only one
    // that overwrites them
    constexpr bool kEarly = CM <= 8;
    // From 12 elements on, C_n is read between the passes, so that 12 elements
    // fit in 128 registers and two workgroups in a CU (1531 x 1531: 33.7 -> 29.5 us).
    constexpr bool kLate = CM >= 12;
    double a[CM], f[CM], al[CM], v[CM], cp[CM];
#pragma unroll
    for (int k = 0; k < CM; ++k) a[k] = f[k] = al[k] = v[k] = cp[k] = 0.0;
    if (kEarly && live) load_coefs<CM, W>(p.coef, p.same ? 0 : line, g, a, f, al);
    if (tlive) {
        // all loads first (clamped indices), then the LDS writes
        const double* __restrict__ cc = p.C + (tline + 1);
        const double* __restrict__ q0 = p.rhs + tline;
        double om[CM];
#pragma unroll
        for (int r = 0; r < CM; ++r)
            om[r] = q0[(int64_t)min(r * NL + tr, n - 1) * p.NX];  // node (i, j = e+1)
#pragma unroll
        for (int r = 0; r < CM && !kLate; ++r)
            cp[r] = cc[(int64_t)(min(r * NL + tr, n - 1) + 1) * ld];
#pragma unroll
        for (int r = 0; r < CM; ++r) {
            const int e = r * NL + tr;
            if (e < n) lds[tc][e + e / CM] = om[r];
        }
    }
    __syncthreads();
    if (live) {
        if (!kEarly) load_coefs<CM, W>(p.coef, p.same ? 0 : line, g, a, f, al);
#pragma unroll
        for (int k = 0; k < CM; ++k) v[k] = e0 + k < n ? lds[li][g * S + k] : 0.0;
    }
    const double un = line_solve_mw(
        a, f, al, v, e0, n, p.b0, lane, wl, &share[li], live, nullptr, [&] {
            if (kLate && tlive) {
                const double* __restrict__ cc = p.C + (tline + 1);
#pragma unroll
                for (int r = 0; r < CM; ++r)
                    cp[r] = cc[(int64_t)(min(r * NL + tr, n - 1) + 1) * ld];
            }
        });
    if (live) {
#pragma unroll
        for (int k = 0; k < CM; ++k)
            if (e0 + k < n) lds[li][g * S + k] = v[k];
        double* Ccol = p.C + (line + 1);
        if (g == 0) {
            Ccol[0] = p.al1 * v[0] + p.b0;
            Ccol[(int64_t)(n + 1) * ld] = un;
            Ccol[(int64_t)(n + 2) * ld] = un;
        }
    }
    __syncthreads();
    if (tlive) {
        const int i = tline + 1;
        double* __restrict__ cc = p.C + i;
#pragma unroll
        for (int r = 0; r < CM; ++r) {
            const int e = r * NL + tr;
            if (e < n) {
                const int64_t q = (int64_t)e * p.NX + (i - 1);
                const double u = lds[tc][e + e / CM];
                cc[(int64_t)(e + 1) * ld] = u;
                const double d = u - cp[r];
                if (p.slotf)
                    p.slotf[q] = (float)d;
                else
                    p.slot[q] = d;
            }
        }
    }
}

// ------------------------------------------------------------- small grids
// Steps n0 .. n0 + ks - 1 (one block's) of a small grid in one workgroup: the
// sweeps' lines and the block's increments stay in LDS, the state and each
// line's coefficients in registers, and a barrier stands where the other path
// ends a kernel.  A line is one 16-lane row of a wavefront, CM elements per lane,
// so that four lines share each scan's instructions and 64 rows of lanes hold
// every line of a direction.  Memory-term sums, right-hand sides and increments
// go node by node in storage order.  What it takes: lines of at most
// kSmallLine in both directions, and 128 bytes of LDS per node for the field
// and the 15 increments that a block's steps read (1270 nodes).  40 x 33: 16.1
// us per step with its three launches, 4.0 here, bound by the instructions of 16
// wavefronts on one CU.  (Increments read back from memory: 8.4 us; kept in
// registers, two nodes per thread: spills, 17 us; a wavefront per line: 10 us.)
constexpr int kSmallLine = 64;
constexpr int kSmallThreads = 1024;
constexpr int kSmallLds = 159 * 1024;

struct SmallArgs {
    double* C;             // state, reference layout
    const double *rcoef, *ccoef;  // [3][lines][n]
    void* hist;
    int64_t ldh;
    const double *far;     // far sums of the block [2][kHistBlock][ldh], or null
    const double* w;       // lag-indexed [2][ldw]
    int ldw;
    int ld, NX, NY, N0, n0, ks;
    double r_negsk, c_negsk, S_half, sg, kch, C1;
};

// stride of a row in LDS: odd, so that a column's elements spread over the banks
__host__ __device__ constexpr int small_stride(int NX) { return NX | 1; }

// Bytes of LDS: the field and kHistBlock - 1 increments.
static int64_t small_bytes(int NX, int NY, size_t esz) {
    return (int64_t)NY * small_stride(NX) * 8 + (int64_t)(kHistBlock - 1) * NX * NY * esz;
}

// A barrier for LDS alone: __syncthreads also waits for global loads and
// stores, which here only their own thread looks at.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// One line per 16-lane row: its element e is x[e se] on entry (the right-hand
// side) and on exit (the solution), for lanes with `store`; first: the value
// before element 0 (line_solve's b0).  v0: the first element's solution on the
// row's first lane.  Returns u_n.
template <int CM>
__device__ __forceinline__ double small_line(const double (&a)[CM], const double (&f)[CM],
                                             const double (&al)[CM], double* x, int se, int n,
                                             double first, bool store, double& v0) {
    const int lane = threadIdx.x & 63, e0 = (lane & 15) * CM;
    double v[CM], P = 1.0, Q = 0.0;
#pragma unroll
    for (int k = 0; k < CM; ++k) v[k] = x[min(e0 + k, n - 1) * se];
#pragma unroll
    for (int k = 0; k < CM; ++k) {
        if (e0 + k < n) {
            const double p = f[k] * a[k], q = -f[k] * v[k];
            Q = p * Q + q;
            P = p * P;
        }
    }
    affine_level<kDppRowShr + 1>(P, Q);
    affine_level<kDppRowShr + 2>(P, Q);
    affine_level<kDppRowShr + 4>(P, Q);
    affine_level<kDppRowShr + 8>(P, Q);
    double y = dpp_move<kDppRowShr + 1>(1.0, P) * first + dpp_move<kDppRowShr + 1>(0.0, Q);
    double un = 0.0;
#pragma unroll
    for (int k = 0; k < CM; ++k) {
        if (e0 + k < n) {
            y = f[k] * (a[k] * y - v[k]);
            v[k] = y;
        }
        if (e0 + k == n - 1) un = y / (1.0 - al[k]);
    }
    un = __shfl(un, (lane & 48) + (n - 1) / CM);
    P = 1.0;
    Q = 0.0;
#pragma unroll
    for (int k = CM - 1; k >= 0; --k) {
        if (e0 + k < n) {
            Q = al[k] * Q + v[k];
            P = al[k] * P;
        }
    }
    affine_level<kDppRowShl + 1>(P, Q);
    affine_level<kDppRowShl + 2>(P, Q);
    affine_level<kDppRowShl + 4>(P, Q);
    affine_level<kDppRowShl + 8>(P, Q);
    y = dpp_move<kDppRowShl + 1>(1.0, P) * un + dpp_move<kDppRowShl + 1>(0.0, Q);
#pragma unroll
    for (int k = CM - 1; k >= 0; --k) {
        if (e0 + k < n) {
            y = al[k] * y + v[k];
            if (store) x[(e0 + k) * se] = y;
        }
    }
    v0 = y;
    return un;
}

// R nodes per thread; CX, CY elements per lane of the rows and columns.
template <typename HT, int R, int CX, int CY>
__global__ __launch_bounds__(kSmallThreads) void k_lod_small(SmallArgs p) {
    constexpr int J = kHistBlock;
    __shared__ __attribute__((aligned(8))) char lds[kSmallLds];
    const int NX = p.NX, NY = p.NY, SX = small_stride(NX), nodes = NX * NY;
    double* M = reinterpret_cast<double*>(lds);       // right-hand side of a sweep, then its solution
    HT* inc = reinterpret_cast<HT*>(M + NY * SX);     // [J - 1][nodes] the block's increments
    const int tid = threadIdx.x, j0 = p.n0 - p.N0, L = tid >> 4, e0 = tid & 15;
    HT* hist = static_cast<HT*>(p.hist) + (int64_t)p.N0 * p.ldh;
    // this thread's nodes (one past the end repeats the last and stores nothing)
    int q[R], at[R];
    double c[R], fr[R], fc[R];
    bool mine[R];
    // wavefronts without a line skip the sweep: the instructions of 16
    // wavefronts are what bounds a step
    const int wv0 = __builtin_amdgcn_readfirstlane(tid) & ~63;
    const bool rows = wv0 / 16 < NY, cols = wv0 / 16 < NX;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        mine[r] = tid + r * kSmallThreads < nodes;
        q[r] = min(tid + r * kSmallThreads, nodes - 1);
        const int y = q[r] / NX, x = q[r] - y * NX;
        at[r] = y * SX + x;
        c[r] = p.C[(int64_t)(y + 1) * p.ld + x + 1];
        fr[r] = p.far ? p.far[(int64_t)j0 * p.ldh + q[r]] : 0.0;
        fc[r] = p.far ? p.far[(int64_t)(J + j0) * p.ldh + q[r]] : 0.0;
        for (int u = 0; u < j0; ++u) {
            const HT x = hist[(int64_t)u * p.ldh + q[r]];
            if (mine[r]) inc[u * nodes + q[r]] = x;
        }
    }
    // this row of lanes' line in each direction (spare rows repeat the last)
    double ra[CX], rf[CX], rl[CX], ca[CY], cf[CY], cl[CY];
    const int Lr = min(L, NY - 1), Lc = min(L, NX - 1);
#pragma unroll
    for (int k = 0; k < CX; ++k) {
        const int e = Lr * NX + min(e0 * CX + k, NX - 1);
        ra[k] = p.rcoef[e];
        rf[k] = p.rcoef[nodes + e];
        rl[k] = p.rcoef[2 * nodes + e];
    }
#pragma unroll
    for (int k = 0; k < CY; ++k) {
        const int e = Lc * NY + min(e0 * CY + k, NY - 1);
        ca[k] = p.ccoef[e];
        cf[k] = p.ccoef[nodes + e];
        cl[k] = p.ccoef[2 * nodes + e];
    }
    // read-only data at addresses the same on every lane: scalar loads
    typedef const __attribute__((address_space(4))) double* const_doubles;
    const const_doubles wr = (const_doubles)p.w, wc = (const_doubles)(p.w + p.ldw);
    for (int st = 0; st < p.ks; ++st) {
        const int j = j0 + st;
        const bool out = st == p.ks - 1;
        // both targets' sums (own nodes: no barrier) and the rows' right-hand side
        double ts[R], tc[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            ts[r] = fr[r];
            tc[r] = fc[r];
        }
        constexpr int G = 5;  // lags whose reads go out together
        static_assert((J - 1) % G == 0, "whole groups");
#pragma unroll
        for (int l0 = 1; l0 < J; l0 += G) {
            if (l0 <= j) {  // lags past the block's first slot read that slot and weigh 0
                double x[G][R];
#pragma unroll
                for (int g = 0; g < G; ++g)
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        x[g][r] = (double)inc[max(j - l0 - g, 0) * nodes + q[r]];
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const double a = l0 + g <= j ? wr[l0 + g - 1] : 0.0;
                    const double b = l0 + g <= j ? wc[l0 + g - 1] : 0.0;
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        ts[r] += a * x[g][r];
                        tc[r] += b * x[g][r];
                    }
                }
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            double om = p.r_negsk * c[r];
            om += p.S_half;
            om += p.sg * ts[r];
            if (mine[r]) M[at[r]] = om;
            if (p.far && !out) {  // the next step's far sums, on their way during the sweeps
                fr[r] = p.far[(int64_t)(j + 1) * p.ldh + q[r]];
                fc[r] = p.far[(int64_t)(J + j + 1) * p.ldh + q[r]];
            }
        }
        lds_barrier();
        // the boundary nodes, which no sweep reads, are written with the last step
        double v0 = 0.0, un = 0.0;
        if (rows) un = small_line<CX>(ra, rf, rl, M + Lr * SX, 1, NX, p.C1, L < NY, v0);
        if (out && e0 == 0 && L < NY) {
            double* Crow = p.C + (int64_t)(L + 1) * p.ld;
            Crow[0] = p.C1;
            Crow[NX + 1] = un;
            Crow[NX + 2] = un;
        }
        lds_barrier();
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const double u = M[at[r]], t = tc[r] + p.kch * (c[r] - u);
            double om = p.c_negsk * u;
            om += p.S_half;
            om += p.sg * t;
            if (mine[r]) M[at[r]] = om;
        }
        lds_barrier();
        if (cols) un = small_line<CY>(ca, cf, cl, M + Lc, SX, NY, 0.0, L < NX, v0);
        if (out && e0 == 0 && L < NX) {
            double* Ccol = p.C + (L + 1);
            Ccol[0] = v0;
            Ccol[(int64_t)(NY + 1) * p.ld] = un;
            Ccol[(int64_t)(NY + 2) * p.ld] = un;
        }
        lds_barrier();
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const double u = M[at[r]];
            const HT x = (HT)(u - c[r]);
            c[r] = u;
            if (mine[r]) {
                hist[(int64_t)j * p.ldh + q[r]] = x;
                if (j < J - 1) inc[j * nodes + q[r]] = x;
            }
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int y = q[r] / NX, x = q[r] - y * NX;
        if (mine[r]) p.C[(int64_t)(y + 1) * p.ld + x + 1] = c[r];
    }
}

// ------------------------------------------------------------- g(t) = t^p
// History weights of step n, lag-indexed (w[t*cap + k] multiplies the
// increment of full step s = n-1-k): rows kb(s, 1/2, 0, 1), columns
// kb(s, 1, 0, 1), each by the _kb_row series (frm_gpow.hpp), one thread per
// weight; the reference rebuilds them for every s <= n each step
// (fr_d_t_g_2d.cpp:3059-3239).
__global__ __launch_bounds__(256) void k_gpow_weights(int n, double alpha, double tau, double p,
                                                      double int_err, double Da, int cap,
                                                      double* __restrict__ w,
                                                      int* __restrict__ flag) {
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= 2 * n) return;
    const int t = idx / n, k = idx % n;
    bool capped = false;
    const double v = kb_pow(alpha, tau, p, int_err, n, n - 1 - k, t ? 1.0 : 0.5, 0.0, 1.0, &capped);
    w[(int64_t)t * cap + k] = Da * v;
    if (capped) atomicOr(flag, 1);
}

// Thomas alpha coefficients (a, f, al) of every line for the diagonal
// sgk + A + B, in the reference's order (al1, fr_d_t_g_2d.cpp:3267-3304) --
// line_coefs on the GPU, one thread per line, written in the interleaved
// layout of load_coefs for chunk length cm and nl lanes per line.
__global__ __launch_bounds__(64) void k_line_coefs(const double* __restrict__ A,
                                                   const double* __restrict__ B, int lines, int n,
                                                   double sgk, double al_first, int cm, int nl,
                                                   double* __restrict__ out) {
    const int L = blockIdx.x * blockDim.x + threadIdx.x;
    if (L >= lines) return;
    const double* a = A + (int64_t)L * n;
    const double* b = B + (int64_t)L * n;
    double Al = al_first;
    for (int e = 0; e < n; ++e) {
        const double ae = a[e], be = b[e];
        const double R = sgk + ae + be;
        const double den = R - ae * Al;
        const double Aln = be / den;
        const double f = (Aln == 0.0 && be == 0.0) ? 1.0 / den : Aln / be;
        const int g = e / cm, k = e % cm;
        out[(((int64_t)L * 3 + 0) * cm + k) * nl + g] = ae;
        out[(((int64_t)L * 3 + 1) * cm + k) * nl + g] = f;
        out[(((int64_t)L * 3 + 2) * cm + k) * nl + g] = Aln;
        Al = Aln;
    }
}

// [3][lines][n] (a, f, al) -> the interleaved layout of load_coefs, for the
// first `stored` lines; zeros past a line's end.
__global__ __launch_bounds__(256) void k_layout_coefs(const double* __restrict__ plain, int lines,
                                                      int stored, int n, int cm, int nl,
                                                      double* __restrict__ out) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (int64_t)stored * 3 * cm * nl) return;
    const int e = (int)(q % nl) * cm + (int)(q / nl % cm);
    const int64_t lc = q / ((int64_t)cm * nl);  // line * 3 + array
    out[q] = e < n ? plain[(lc % 3 * lines + lc / 3) * n + e] : 0.0;
}

// ------------------------------------------------------------- ia/ibk memory term
// The reference's dt_alg 4 (calc_va, fr_d_t_g_2d.cpp:490-741) for every node:
// each direction's plan step (frm_iaibk.cpp) evaluates the node's valid
// approximations at x = n, adds the newest block exactly, then folds the
// newest increment Delta_{n-1} into the coefficient slots.  One lane per
// node; the operations are wavefront-uniform.
struct IaArgs {
    double* H;                 // [2][slots][MAXAK][ld]
    const double* ring;        // two-slot increment ring
    int64_t ld;
    int n, slots;
    const IaOp* ops[2];
    int o0[2], o1[2];          // this step's operation range per direction
    const double* vals[2];
    double ak[kIaMaxAk];
    double scale;
    double* part;              // [2][ld]
};

__global__ __launch_bounds__(256) void k_iaibk_memterm(IaArgs p) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= p.ld) return;
    const int64_t ld = p.ld;
    const double f = p.ring[(int64_t)((p.n - 1) % 2) * ld + i];  // the two-slot ring
#pragma unroll 1
    for (int t = 0; t < 2; ++t) {
        double* H = p.H + (int64_t)t * p.slots * kIaMaxAk * ld + i;
        const IaOp* ops = p.ops[t];
        const double* vals = p.vals[t];
        double V = 0.0;
        for (int o = p.o0[t]; o < p.o1[t]; ++o) {
            const IaOp op = ops[o];
            double* c = H + (int64_t)op.slot * kIaMaxAk * ld;
            const double* w = vals + op.off;
            if (op.kind == kIaEvalIa || op.kind == kIaEvalIbk) {
                double r = 0.0;
                for (int k = 0; k < op.nt; ++k) r += c[(int64_t)k * ld] * w[k];
                V += r;
            } else if (op.kind == kIaExact) {
                V += w[0] * f;
            } else if (op.kind == kIaCreate) {
                for (int k = 0; k < kIaMaxAk; ++k) c[(int64_t)k * ld] = k < op.nt ? p.ak[k] * (f * w[k]) : 0.0;
            } else if (op.kind == kIaAdd) {
                for (int k = 0; k < op.nt; ++k) c[(int64_t)k * ld] += p.ak[k] * (f * w[k]);
            } else if (op.kind == kIaCopy) {
                const double* src = H + (int64_t)op.src * kIaMaxAk * ld;
                for (int k = 0; k < kIaMaxAk; ++k) c[(int64_t)k * ld] = src[(int64_t)k * ld];
            }
        }
        p.part[(int64_t)t * ld + i] = V * p.scale;
    }
}

// ------------------------------------------------------------- SOE memory term
// History weights for lags k >= 2 replaced by sum_l c_{t,l} q_l^(k-2): per
// node, the mode states H_l = sum_{s <= n-2} q_l^(n-2-s) Delta_s follow
// H_l <- q_l H_l + Delta_{n-2} (the increment that just reached lag 2), and
// lag 1 is summed exactly from a two-slot ring of increments.  The decay
// multiply is done in FP64 so that slow modes keep their exact factor when
// the states are stored in FP32.
constexpr int kSoeLag0 = 2;
// largest relative error of a fitted exponential sum over the weights it
// replaces that frm_lod2d_create accepts
constexpr double kSoeFitTol = 1e-6;

// FP32 states take this step every step: their rounding after each is part of
// the form.  FP64 states advance once per block (k_soe_block).
template <bool NT>
__global__ __launch_bounds__(256) void k_soe_memterm(float* __restrict__ H, const double* __restrict__ ring,
                                                     int64_t ld, int n, int L,
                                                     const double* __restrict__ q,
                                                     const double* __restrict__ c, double w1r,
                                                     double w1c, double* __restrict__ part) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ld) return;
    const bool fold = n >= kSoeLag0;
    const double x = fold ? ring[(int64_t)((n - kSoeLag0) % kSoeLag0) * ld + i] : 0.0;
    double s0 = 0.0, s1 = 0.0;
    for (int l = 0; l < L; ++l) {
        // the mode planes are streamed once per step (non-temporal when
        // they exceed the cache)
        double h = (double)stream_load<NT>(H + (int64_t)l * ld + i);
        if (fold) {
            h = q[l] * h + x;
            stream_store<NT>((float)h, H + (int64_t)l * ld + i);
            h = (double)(float)h;
        }
        s0 += c[l] * h;
        s1 += c[L + l] * h;
    }
    if (n >= 1) {
        const double y = ring[(int64_t)((n - 1) % kSoeLag0) * ld + i];
        s0 += w1r * y;
        s1 += w1c * y;
    }
    part[i] = s0;
    part[ld + i] = s1;
}

// FP64 states, kSoeBlock = J steps at a time.  At a block start N0 the states
// are H_l = sum_{s <= N0-2} q_l^(N0-2-s) Delta_s; a step n = N0 + j of the
// block sums sum_l (c_{t,l} q_l^j) H_l over the slots before N0 - 1, formed
// here for all j at once, and takes the at most J newer slots N0-1 .. n-1 with
// their lags' weights (the exact one at lag 1, the fitted sum's values after)
// in the row kernel.  One pass over the mode planes, which are read and
// written once per J steps instead of every step, folds the J increments
// N0-1-J .. N0-2 that have left the last block's reach (q_l^J H_l +
// sum_i q_l^(J-1-i) Delta) and forms the 2 J sums.  The planes bound it (512 B
// per node and block at 32 modes, against 24 multiply-adds per mode); with
// J = 8 the sums add 128 B and the factors of a mode are 24 scalars.
// Measured at 1024 x 1024, 32 modes: 104 us every step before.
constexpr int kSoeBlock = 8;
constexpr int kSoeRing = 16;  // increment slots: this block's and the last one's
constexpr int kSoeTab = 3 * kSoeBlock;  // q^7 .. q^1, q^8, c_0 q^j, c_1 q^j

template <bool NT>
__global__ __launch_bounds__(256) void k_soe_block(double* __restrict__ H,
                                                   const double* __restrict__ ring, int64_t ld,
                                                   int N0, int L, const double* __restrict__ tab,
                                                   double* __restrict__ G) {
    constexpr int J = kSoeBlock;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ld) return;
    double x[J], g[2][J];
#pragma unroll
    for (int k = 0; k < J; ++k) {
        const int s = N0 - 1 - J + k;  // before the first increment: nothing
        x[k] = s >= 0 ? ring[(int64_t)(s & (kSoeRing - 1)) * ld + i] : 0.0;
        g[0][k] = g[1][k] = 0.0;
    }
    constexpr int U = 4;  // modes whose loads go out together
    for (int l0 = 0; l0 < L; l0 += U) {
        double h[U];
#pragma unroll
        for (int u = 0; u < U; ++u) h[u] = stream_load<NT>(H + (int64_t)min(l0 + u, L - 1) * ld + i);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (l0 + u < L) {
                const double* __restrict__ f = tab + (l0 + u) * kSoeTab;
                double v = f[J - 1] * h[u] + x[J - 1];
#pragma unroll
                for (int k = 0; k < J - 1; ++k) v += f[k] * x[k];
                stream_store<NT>(v, H + (int64_t)(l0 + u) * ld + i);
#pragma unroll
                for (int j = 0; j < J; ++j) {
                    g[0][j] += f[J + j] * v;
                    g[1][j] += f[2 * J + j] * v;
                }
            }
        }
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int j = 0; j < J; ++j) G[(int64_t)(t * J + j) * ld + i] = g[t][j];
}

// ------------------------------------------------------------- binomial-series memory term
// TG_solver's dt_alg = 3 (fr_d_t_g_2d.cpp:3385-3428): per node and sweep
// direction, moments H_k = sum over full steps s of g(t_{s+1})^(k+1) v3_k(s)
// Delta_s (Htmp1 for rows, Htmp2 for columns), each step taking the newest
// increment Delta_{n-1} = C_n - C_{n-1} from the two-slot ring into the
// first cnt moments, and the memory term Da sum_k f_k H_k with the binomial
// factors f_k of the direction's target (_kb_row2_fixed_coefs).  Products
// and sums are rounded separately, as the reference's x86-64 build does.
__global__ __launch_bounds__(256) void k_binomial_memterm(
    double* __restrict__ H, const double* __restrict__ ring, int64_t ld, int n, int terms,
    const double* __restrict__ upd, const double* __restrict__ er, const double* __restrict__ ec,
    const int* __restrict__ cnt, double Da, double* __restrict__ part) {
#pragma clang fp contract(off)
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ld) return;
    if (n == 0) {  // no full step yet: the row term is 0, the column one only its half step
        part[i] = 0.0;
        part[ld + i] = 0.0;
        return;
    }
    const int64_t r = (int64_t)(n - 1) * terms;
    const int* c = cnt + 4 * (int64_t)(n - 1);
    const double x = ring[(int64_t)((n - 1) % kSoeLag0) * ld + i];
    constexpr int B = 8;  // moments loaded together
#pragma unroll
    for (int dir = 0; dir < 2; ++dir) {
        double* __restrict__ Hd = H + (int64_t)dir * terms * ld + i;
        const double* __restrict__ f = (dir == 0 ? er : ec) + r;
        const int cu = c[dir], ce = c[2 + dir];
        double acc = 0.0;
        for (int k0 = 0; k0 < terms; k0 += B) {
            double h[B];
#pragma unroll
            for (int u = 0; u < B; ++u)
                if (k0 + u < terms) h[u] = Hd[(int64_t)(k0 + u) * ld];
#pragma unroll
            for (int u = 0; u < B; ++u) {
                const int k = k0 + u;
                if (k >= terms) break;
                if (k < cu) {
                    h[u] = h[u] + upd[r + k] * x;
                    Hd[(int64_t)k * ld] = h[u];
                }
                if (k < ce) acc += f[k] * h[u];
            }
        }
        part[(int64_t)dir * ld + i] = Da * acc;
    }
}

// ------------------------------------------------------------- host helpers
// Thomas alpha coefficients of one line in the reference's order
// (al1: fr_d_t_g_2d.cpp:3267-3304, R: 3257-3265); f = Al[i+1]/B(i), or the
// zero-pivot form 1/(R - A Al[i]) (3519-3522).
static void line_coefs(int n, const double* A, const double* B, int64_t stride, double sgk,
                       double al_first, double* oa, double* of, double* oal) {
    double Al = al_first;
    for (int e = 0; e < n; ++e) {
        const double a = A[e * stride], b = B[e * stride];
        const double R = sgk + a + b;
        const double Aln = b / (R - a * Al);
        oa[e] = a;
        if (Aln == 0.0 && b == 0.0)
            of[e] = 1.0 / (R - a * Al);
        else
            of[e] = Aln / b;
        oal[e] = Aln;
        Al = Aln;
    }
}

// nearest BF16 value (round to nearest even) of x, as a float
static float bf16_round(double x) {
    float f = (float)x;
    uint32_t u;
    std::memcpy(&u, &f, 4);
    u = (u + 0x7FFFu + ((u >> 16) & 1u)) & 0xFFFF0000u;
    std::memcpy(&f, &u, 4);
    return f;
}

// Whether all lines' coefficients ([arrays][lines][n]) are equal.
static bool same_lines(const double* p, int arrays, int lines, int n) {
    for (int c = 0; c < arrays; ++c, p += (size_t)lines * n) {
        for (int L = 1; L < lines; ++L)
            if (std::memcmp(p, p + (size_t)L * n, sizeof(double) * n)) return false;
    }
    return true;
}

// smallest chunk length that fits n unknowns on 64 W lanes (0: none)
static int pick_cm(int n, int W) {
    for (int cm : {4, 6, 8, 12, 16, 24, 32})
        if (n <= kWave * W * cm) return cm;
    return 0;
}


#define FRM_SWEEP_CM(X, W) X(4, W) X(6, W) X(8, W) X(12, W) X(16, W) X(24, W) X(32, W)
#define FRM_SWEEP_CASES(X) FRM_SWEEP_CM(X, 1) FRM_SWEEP_CM(X, 2) FRM_SWEEP_CM(X, 4)

template <int SRC>
static hipError_t launch_rows(SweepShape sh, hipStream_t st, const RowArgs& a) {
    const int lpb = 4 / sh.w;
    const dim3 grid((unsigned)((a.lines + lpb - 1) / lpb));
#define X(CM, W)                                                                     \
    if (sh.cm == CM && sh.w == W) {                                                  \
        hipLaunchKernelGGL((k_lod_rows<CM, W, SRC>), grid, dim3(256), 0, st, a);     \
        return hipGetLastError();                                                    \
    }
    FRM_SWEEP_CASES(X)
#undef X
    return hipErrorInvalidValue;
}

// The row kernel's memory-term source for a solver's form.
static RowSrc row_src(const frm_lod2d* s) {
    if (s->g_func == 0 && s->precision == FRM_PREC_F64) return kRowNear64;
    if (s->precision == FRM_PREC_SOE && !s->soe_f32) return kRowNear64;
    if (s->precision == FRM_PREC_F32C) return kRowNear32;
    if (s->precision == FRM_PREC_MFMA_BF16) return kRowNearMx;
    return kRowPart;
}

static hipError_t launch_rows(const frm_lod2d* s, hipStream_t st, const RowArgs& a) {
    switch (row_src(s)) {
        case kRowNear64: return launch_rows<kRowNear64>(s->rsh, st, a);
        case kRowNear32: return launch_rows<kRowNear32>(s->rsh, st, a);
        case kRowNearMx: return launch_rows<kRowNearMx>(s->rsh, st, a);
        default: return launch_rows<kRowPart>(s->rsh, st, a);
    }
}

template <int CM, int W, int LW>
static bool launch_cols_as(SweepShape sh, hipStream_t st, const ColArgs& a) {
    if constexpr (col_fits(CM, W, LW)) {
        if (sh.lw != LW) return false;
        const dim3 grid((unsigned)((a.groups + 7) / 8 * 8));
        hipLaunchKernelGGL((k_lod_cols<CM, W, LW>), grid, dim3(LW * kWave * W), 0, st, a);
        return true;
    } else {
        return false;
    }
}

static hipError_t launch_cols(SweepShape sh, hipStream_t st, const ColArgs& a) {
#define X(CM, W)                                                                        \
    if (sh.cm == CM && sh.w == W &&                                                     \
        (launch_cols_as<CM, W, 1>(sh, st, a) || launch_cols_as<CM, W, 2>(sh, st, a) ||  \
         launch_cols_as<CM, W, 4>(sh, st, a) || launch_cols_as<CM, W, 8>(sh, st, a)))   \
        return hipGetLastError();
    FRM_SWEEP_CASES(X)
#undef X
    return hipErrorInvalidValue;
}

// Kernel arguments of one step's sweeps (n = step index).  far, mid: the
// block's far and mid sums are formed (the near forms; otherwise there are
// none yet).
static RowArgs row_args(frm_lod2d* s, int nch, int n, bool far, bool mid) {
    RowArgs a;
    a.C = s->C;
    a.crhs = s->crhs;
    const int64_t hld = s->hist->ld;
    const bool soe = s->precision == FRM_PREC_SOE;
    const bool mf = s->precision == FRM_PREC_MFMA_BF16;
    const int J = soe ? kSoeBlock : mf ? kMidBlock : kHistBlock;
    const int N0 = n / J * J, j = n - N0;
    a.near.hist = s->hist->data;
    a.near.ld = hld;
    a.near.s0 = soe ? std::max(0, N0 - 1) : N0;
    a.near.cnt = n - a.near.s0;
    a.near.mask = s->ring ? s->ring - 1 : -1;
    a.near.w = s->w;
    a.near.ldw = s->ldw;
    a.near.f0 = far ? s->far + (int64_t)j * hld : nullptr;
    a.near.f1 = far ? s->far + (int64_t)(J + j) * hld : nullptr;
    a.near.m0 = a.near.m1 = nullptr;
    if (mf) {
        // the 64-step block's far rows (by block parity), the sub-block's mid rows
        const int b = n / kBlockSteps, q = n % kBlockSteps;
        const float* F = s->F + (size_t)(b & 1) * 2 * kBlockSteps * hld;
        a.near.f0 = far ? F + (int64_t)q * hld : nullptr;
        a.near.f1 = far ? F + (int64_t)(kBlockSteps + q) * hld : nullptr;
        a.near.m0 = mid ? s->G + (int64_t)j * hld : nullptr;
        a.near.m1 = mid ? s->G + (int64_t)(kMidBlock + j) * hld : nullptr;
    }
    a.coef = s->rcoef;
    a.same = s->rsame;
    a.part = s->hist->part;
    a.ldh = s->hist->ld;
    a.nch = nch;
    a.ld = s->ld;
    a.lines = s->M - 1;
    a.n = s->NX;
    a.NX = s->NX;
    a.negsk = -s->sg * s->kr0;
    a.S_half = s->S * 0.5;
    a.sg = s->sg;
    a.col_negsk = -s->sg * s->kc0;
    a.kch = s->kch;
    a.b0 = s->C1;
    a.al1 = 0.0;
    return a;
}

static ColArgs col_args(frm_lod2d* s, int n) {
    const bool f32 = s->precision == FRM_PREC_MFMA_BF16 || s->precision == FRM_PREC_F32C;
    ColArgs a;
    a.C = s->C;
    a.rhs = s->crhs;
    a.slot = (double*)s->hist->data +
             (int64_t)(s->ring ? (n % s->ring) : s->hist->depth) * s->hist->ld;
    a.slotf = f32 ? (float*)s->hist->data + (int64_t)s->hist->depth * s->hist->ld : nullptr;
    a.coef = s->ccoef;
    a.same = s->csame;
    a.ld = s->ld;
    a.lines = s->sN - 1;
    a.n = s->NY;
    a.NX = s->NX;
    a.b0 = 0.0;
    a.al1 = 1.0;
    a.groups = (a.lines + s->csh.lw - 1) / s->csh.lw;
    return a;
}

// Lays a direction's coefficients ([3][lines][n] in plain) out for a shape.
static hipError_t layout_coefs(frm_lod2d* s, bool rows, SweepShape sh, const double* plain) {
    const int lines = rows ? s->M - 1 : s->sN - 1, n = rows ? s->NX : s->NY;
    const int stored = (rows ? s->rsame : s->csame) ? 1 : lines, nl = kWave * sh.w;
    const int64_t total = (int64_t)stored * 3 * sh.cm * nl;
    hipLaunchKernelGGL(k_layout_coefs, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                       s->ctx->stream, plain, lines, stored, n, sh.cm, nl,
                       rows ? s->rcoef : s->ccoef);
    return hipGetLastError();
}

// Whether a grid takes the one-workgroup path (k_lod_small): full history with
// lag-only weights, no sweep shape asked for, and what the kernel holds.
static bool takes_small(const frm_lod2d* s, const frm_lod2d_desc* d) {
    const bool f32 = s->precision == FRM_PREC_F32C;
    const bool full = f32 || (s->precision == FRM_PREC_F64 && s->g_func == 0);
    return full && !d->sweep_w && std::max(s->NX, s->NY) <= kSmallLine &&
           (int64_t)s->NX * s->NY <= 2 * kSmallThreads &&
           small_bytes(s->NX, s->NY, f32 ? sizeof(float) : sizeof(double)) <= kSmallLds;
}

static hipError_t launch_small(frm_lod2d* s, int n, int ks, bool far) {
    SmallArgs a;
    a.C = s->C;
    a.rcoef = s->rcoef;
    a.ccoef = s->ccoef;
    a.hist = s->hist->data;
    a.ldh = s->hist->ld;
    a.far = far ? s->far : nullptr;
    a.w = s->w;
    a.ldw = s->ldw;
    a.ld = s->ld;
    a.NX = s->NX;
    a.NY = s->NY;
    a.N0 = n / kHistBlock * kHistBlock;
    a.n0 = n;
    a.ks = ks;
    a.r_negsk = -s->sg * s->kr0;
    a.c_negsk = -s->sg * s->kc0;
    a.S_half = s->S * 0.5;
    a.sg = s->sg;
    a.kch = s->kch;
    a.C1 = s->C1;
    const dim3 g(1), t(kSmallThreads);
    const bool f32 = s->precision == FRM_PREC_F32C;
    auto launch = [&](auto kern) {
        hipLaunchKernelGGL(kern, g, t, 0, s->ctx->stream, a);
        return hipGetLastError();
    };
    const bool one = s->NX * s->NY <= kSmallThreads;
    const int cx = s->NX <= 32 ? 2 : 4, cy = s->NY <= 32 ? 2 : 4;
#define X(CX, CY)                                                                                \
    if (cx == CX && cy == CY)                                                                    \
        return f32 ? launch(one ? k_lod_small<float, 1, CX, CY> : k_lod_small<float, 2, CX, CY>) \
                   : launch(one ? k_lod_small<double, 1, CX, CY> : k_lod_small<double, 2, CX, CY>);
    X(2, 2) X(2, 4) X(4, 2) X(4, 4)
#undef X
    return hipErrorInvalidValue;
}

// Autotuner of the sweep launch shape: for every wavefronts-per-line count
// W in {1, 2, 4} that fits the line (or only `force`) and every column width,
// lay the coefficients out for it and time steps' two sweeps on the solver's own
// buffers (zero state, a block's steps in turn with their far sums, which then
// come from memory as they do in a run), with the other direction's shape held;
// then keep the fastest of each.  Runs at creation, before the initial state is set; the state and the
// history slot it writes are overwritten by frm_lod2d_set_state and the first
// step.  (Timed on one step of a block, alone or not, a sweep finds its data closer than
// a run does: 1531 x 1531 rows ran in 36.8 us in the shape chosen that way, 33.7
// in another.)  rplain, cplain: the rows' and the columns' coefficients on the
// device, [3][lines][n].
static int tune_sweeps(frm_lod2d* s, int force, const double* rplain, const double* cplain) {
    frm_ctx* ctx = s->ctx;
    // the one chunk of partials the timed sweeps read: zeros
    FRM_HIP(ctx, hipMemsetAsync(s->hist->part, 0, sizeof(double) * 2 * s->hist->ld, ctx->stream));
    hipEvent_t e0, e1;
    FRM_HIP(ctx, hipEventCreate(&e0));
    FRM_HIP(ctx, hipEventCreate(&e1));
    constexpr int kWarm = 4, kReps = kHistBlock;
    const int block = std::min(kHistBlock, s->capacity);
    const bool far = s->far || s->F;
    int rc = FRM_OK;
    // a first shape of the columns, for the rows' turn
    for (int W : {4, 2, 1})
        if ((!force || W == force) && pick_cm(s->NY, W))
            for (int lw : kColWidths)
                if (!s->csh.cm && col_fits(pick_cm(s->NY, W), W, lw))
                    s->csh = SweepShape{pick_cm(s->NY, W), W, lw};
    hipError_t e = layout_coefs(s, false, s->csh, cplain);
    if (e != hipSuccess) rc = check_hip(ctx, e, "sweep coefficients");
    for (int pass = 0; pass < 2 && rc == FRM_OK; ++pass) {
        const bool rows = pass == 0;
        const int n = rows ? s->NX : s->NY;
        SweepShape& cur = rows ? s->rsh : s->csh;
        const double* plain = rows ? rplain : cplain;
        float best = 1e30f;
        SweepShape pick;
        for (int W : {1, 2, 4}) {
            const int cm = pick_cm(n, W);
            if ((force && W != force) || !cm) continue;
            e = layout_coefs(s, rows, SweepShape{cm, W}, plain);
            for (int lw : kColWidths) {
                if (rows ? lw > 1 : !col_fits(cm, W, lw)) continue;
                cur = SweepShape{cm, W, rows ? 0 : lw};
                float ms = 0.f;
                for (int it = 0; it < kWarm + kReps && e == hipSuccess; ++it) {
                    if (it == kWarm) e = hipEventRecord(e0, ctx->stream);
                    if (e == hipSuccess)
                        e = launch_rows(s, ctx->stream, row_args(s, 1, it % block, far, far && s->G));
                    if (e == hipSuccess) e = launch_cols(s->csh, ctx->stream, col_args(s, it % block));
                }
                if (e == hipSuccess) e = hipEventRecord(e1, ctx->stream);
                if (e == hipSuccess) e = hipEventSynchronize(e1);
                if (e == hipSuccess) e = hipEventElapsedTime(&ms, e0, e1);
                if (e != hipSuccess) break;
                if (ms < best) {
                    best = ms;
                    pick = cur;
                }
            }
            if (e != hipSuccess) {
                rc = check_hip(ctx, e, "sweep autotuning");
                break;
            }
        }
        if (rc == FRM_OK) {
            cur = pick;
            e = layout_coefs(s, rows, pick, plain);
            if (e != hipSuccess) rc = check_hip(ctx, e, "sweep coefficients");
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return rc;
}

// g(t) = t^p: the current-step weights of step n on the host -- rows
// kb(n, 1/2, 0, 1/2), columns kb(n, 1, 1/2, 1/2), the column half-step term
// kb(n, 1, 0, 1/2) -- as TG_solver::kb computes them (int_alg 1)
static void gpow_current(const frm_lod2d* s, int n, double* kr, double* kc, double* kh,
                         bool* capped) {
    const double a = s->alpha, t = s->tau, p = s->g_pow, ie = s->int_err;
    *kr = s->Da * kb_pow(a, t, p, ie, n, n, 0.5, 0.0, 0.5, capped);
    *kc = s->Da * kb_pow(a, t, p, ie, n, n, 1.0, 0.5, 0.5, capped);
    *kh = s->Da * kb_pow(a, t, p, ie, n, n, 1.0, 0.0, 0.5, capped);
}

// g(t) = t^p: the history weights of step n (GPU) and both directions'
// Thomas coefficients for its current weights
static int gpow_prepare(frm_lod2d* s, int n) {
    frm_ctx* ctx = s->ctx;
    bool capped = false;
    gpow_current(s, n, &s->kr0, &s->kc0, &s->kch, &capped);
    if (capped)
        return set_error(ctx, FRM_E_STATE, "frm_lod2d_step: kb series did not reach int_err at step %d", n);
    if (n > 0) {
        LaunchTimer t(ctx, FRM_K_OTHER, 0.0);
        hipLaunchKernelGGL(k_gpow_weights, dim3((unsigned)((2 * n + 255) / 256)), dim3(256), 0,
                           ctx->stream, n, s->alpha, s->tau, s->g_pow, s->int_err, s->Da,
                           s->ldw, s->w, s->flag);
        FRM_HIP(ctx, hipGetLastError());
    }
    const int64_t nr = (int64_t)(s->M - 1) * s->NX, nc = (int64_t)(s->sN - 1) * s->NY;
    LaunchTimer t(ctx, FRM_K_OTHER, 0.0);
    const int lr = s->rsame ? 1 : s->M - 1, lc = s->csame ? 1 : s->sN - 1;
    hipLaunchKernelGGL(k_line_coefs, dim3((unsigned)((lr + 63) / 64)), dim3(64), 0,
                       ctx->stream, s->lineAB, s->lineAB + nr, lr, s->NX, s->sg * s->kr0,
                       0.0, s->rsh.cm, kWave * s->rsh.w, s->rcoef);
    FRM_HIP(ctx, hipGetLastError());
    hipLaunchKernelGGL(k_line_coefs, dim3((unsigned)((lc + 63) / 64)), dim3(64), 0,
                       ctx->stream, s->lineAB + 2 * nr, s->lineAB + 2 * nr + nc, lc, s->NY,
                       s->sg * s->kc0, 1.0, s->csh.cm, kWave * s->csh.w, s->ccoef);
    FRM_HIP(ctx, hipGetLastError());
    return FRM_OK;
}

static void lod_free(frm_lod2d* s) {
    if (!s) return;
    if (s->hist) frm_hist_destroy(s->hist);
    (void)hipFree(s->C);
    (void)hipFree(s->crhs);
    (void)hipFree(s->w);
    (void)hipFree(s->far);
    (void)hipFree(s->rcoef);
    (void)hipFree(s->ccoef);
    (void)hipFree(s->soe_H);
    (void)hipFree(s->soe_q);
    (void)hipFree(s->soe_c);
    (void)hipFree(s->soe_tab);
    (void)hipFree(s->bin_H);
    (void)hipFree(s->bin_upd);
    (void)hipFree(s->bin_er);
    (void)hipFree(s->bin_ec);
    (void)hipFree(s->bin_cnt);
    (void)hipFree(s->atab);
    (void)hipFree(s->F);
    (void)hipFree(s->G);
    (void)hipFree(s->lineAB);
    (void)hipFree(s->flag);
    (void)hipFree(s->ia_H);
    for (int t = 0; t < 2; ++t) {
        (void)hipFree(s->ia_ops[t]);
        (void)hipFree(s->ia_vals[t]);
    }
    delete s;
}

}  // namespace frm

using namespace frm;

extern "C" {

int frm_lod2d_create(frm_ctx* ctx, const frm_lod2d_desc* d, frm_lod2d** out) {
    FRM_REQUIRE(ctx, ctx && d && out, "frm_lod2d_create: null argument");
    *out = nullptr;
    FRM_REQUIRE(ctx, d->sN >= 2 && d->M >= 2, "frm_lod2d_create: grid %dx%d too small", d->sN,
                d->M);
    FRM_REQUIRE(ctx, d->capacity >= 1, "frm_lod2d_create: capacity %d", d->capacity);
    FRM_REQUIRE(ctx, d->alpha > 0 && d->alpha < 1 && d->tau > 0,
                "frm_lod2d_create: need 0 < alpha < 1 and tau > 0");
    FRM_REQUIRE(ctx, d->rowA && d->rowB && d->colA && d->colB,
                "frm_lod2d_create: coefficient arrays missing");
    FRM_REQUIRE(ctx,
                d->precision == FRM_PREC_F64 || d->precision == FRM_PREC_F32C ||
                    d->precision == FRM_PREC_SOE || d->precision == FRM_PREC_MFMA_BF16 ||
                    d->precision == FRM_PREC_BINOMIAL || d->precision == FRM_PREC_IAIBK,
                "frm_lod2d_create: precision %d not built", d->precision);
    FRM_REQUIRE(ctx,
                d->trunc_eps == 0 ||
                    (d->trunc_eps > 0 && d->precision == FRM_PREC_F64 && d->kernel == FRM_KERNEL_CAPUTO),
                "frm_lod2d_create: trunc_eps takes FRM_PREC_F64 and the Caputo kernel");
    FRM_REQUIRE(ctx,
                d->precision != FRM_PREC_BINOMIAL ||
                    (d->kernel == FRM_KERNEL_CAPUTO && d->series_terms >= 0 &&
                     d->series_terms <= 1000 && d->series_tol >= 0),
                "frm_lod2d_create: FRM_PREC_BINOMIAL takes the Caputo kernel and 0..1000 terms");
    FRM_REQUIRE(ctx, d->soe_terms >= 0 && d->soe_terms <= 64, "frm_lod2d_create: soe_terms %d",
                d->soe_terms);
    FRM_REQUIRE(ctx, d->mfma_parts == 0 || d->mfma_parts == 2 || d->mfma_parts == 3,
                "frm_lod2d_create: mfma_parts %d (2 or 3)", d->mfma_parts);
    FRM_REQUIRE(ctx, d->kernel == FRM_KERNEL_CAPUTO || d->kernel == FRM_KERNEL_AB,
                "frm_lod2d_create: kernel %d", d->kernel);
    FRM_REQUIRE(ctx, d->g_func == 0 || d->g_func == 3, "frm_lod2d_create: g_func %d (0 or 3)",
                d->g_func);
    FRM_REQUIRE(ctx,
                d->precision != FRM_PREC_IAIBK ||
                    (d->kernel == FRM_KERNEL_CAPUTO && d->g_func == 0 && d->trunc_eps == 0),
                "frm_lod2d_create: FRM_PREC_IAIBK takes the Caputo kernel with g(t) = t");
    FRM_REQUIRE(ctx,
                d->g_func == 0 ||
                    (d->precision == FRM_PREC_F64 && d->kernel == FRM_KERNEL_CAPUTO &&
                     d->trunc_eps == 0 && d->g_pow > 0 && d->g_pow <= 4 && d->int_err >= 0),
                "frm_lod2d_create: g_func 3 takes FRM_PREC_F64, the Caputo kernel, the full "
                "history, 0 < g_pow <= 4 and int_err >= 0");
    FRM_REQUIRE(ctx, pick_cm(d->sN - 1, 4) && pick_cm(d->M - 1, 4),
                "frm_lod2d_create: lines longer than %d unknowns", 4 * 64 * 32);
    FRM_REQUIRE(ctx, d->sweep_w == 0 || d->sweep_w == 1 || d->sweep_w == 2 || d->sweep_w == 4,
                "frm_lod2d_create: sweep_w %d (0, 1, 2 or 4)", d->sweep_w);
    FRM_REQUIRE(ctx, d->sweep_w == 0 || (pick_cm(d->sN - 1, d->sweep_w) && pick_cm(d->M - 1, d->sweep_w)),
                "frm_lod2d_create: lines too long for sweep_w %d", d->sweep_w);
    FRM_HIP(ctx, hipSetDevice(ctx->device));

    frm_lod2d* s = new frm_lod2d();
    s->ctx = ctx;
    s->sN = d->sN;
    s->M = d->M;
    s->ld = d->sN + 2;
    s->NX = d->sN - 1;
    s->NY = d->M - 1;
    s->capacity = d->capacity;
    s->alpha = d->alpha;
    s->tau = d->tau;
    s->sigma = d->sigma;
    s->C1 = d->C1;
    s->S = d->S;
    s->sg = d->sigma / d->tau;
    s->g_func = d->g_func;
    s->g_pow = d->g_func == 3 ? d->g_pow : 1.0;
    s->int_err = d->int_err > 0 ? d->int_err : 1e-6;
    s->Da = 1.0 / frm::gamma_cody(1.0 - d->alpha);
    // Caputo: the kernel's integrals over the LOD sub-intervals, as
    // TG_solver::kb (rows target t_{n+1/2}, columns t_{n+1}).
    // Atangana-Baleanu: the kernel is bounded, so a half-interval current
    // weight is smaller than the first history weight and the constant mode
    // of the zero-gradient columns would grow; both half-steps therefore take
    // the full-step weights of MF_intF_simple, I(d) = MF_int_choice(d tau,
    // tau, 0)/(1-alpha), current I(1), with half of the memory term each, so
    // that the two half-steps add up to the full-step AB discretisation.
    frm::AbIntegrator ab(d->alpha, d->ab_maxl > 0 ? d->ab_maxl : 50,
                         d->ab_maxkiter > 0 ? d->ab_maxkiter : 1000,
                         d->ab_eps > 0 ? d->ab_eps : 1e-10);
    const bool is_ab = d->kernel == FRM_KERNEL_AB;
    std::vector<double> abx;
    if (is_ab && d->ab_exact) {
        abx.resize(d->capacity + 2);
        frm::ab_exact_weights(d->alpha, d->tau, d->capacity + 2, abx.data());
    }
    auto abI = [&](int dd) {
        if (!abx.empty()) return abx[dd - 1] / (1.0 - d->alpha);
        return ab.integral(dd * d->tau, d->tau, 0.0) / (1.0 - d->alpha);
    };
    // current-step weights: kb(n,1/2,0,1/2), kb(n,1,1/2,1/2), kb(n,1,0,1/2)
    s->kr0 = is_ab ? abI(1) : caputo_kb(d->alpha, d->tau, 0.5, 0.5);
    s->kc0 = is_ab ? abI(1) : caputo_kb(d->alpha, d->tau, 0.5, 0.5);
    s->kch = is_ab ? 0.0 : caputo_kb(d->alpha, d->tau, 1.0, 0.5);
    if (s->g_func == 3) {
        bool capped = false;
        gpow_current(s, 0, &s->kr0, &s->kc0, &s->kch, &capped);
        if (capped) {
            lod_free(s);
            return set_error(ctx, FRM_E_INVALID, "frm_lod2d_create: kb series did not reach int_err");
        }
    }
    const int64_t nodes = (int64_t)s->NX * s->NY;
    const size_t nn = (size_t)s->ld * (d->M + 2);
    s->precision = d->precision;
    // the SOE, binomial and ia/ibk forms keep only a ring of increments (two
    // slots, or a block's with FP64 mode states), the blocked MFMA and
    // compensated FP32 forms FP32 increments
    const bool mf = d->precision == FRM_PREC_MFMA_BF16;
    s->soe_f32 = d->precision == FRM_PREC_SOE && d->soe_f32;
    if (d->precision == FRM_PREC_SOE && !s->soe_f32)
        s->ring = kSoeRing;
    else if (d->precision == FRM_PREC_SOE || d->precision == FRM_PREC_BINOMIAL ||
             d->precision == FRM_PREC_IAIBK)
        s->ring = kSoeLag0;
    int rc = hist_alloc(ctx, nodes, s->ring ? s->ring : d->capacity,
                        mf || d->precision == FRM_PREC_F32C ? d->precision : FRM_PREC_F64,
                        &s->hist);
    if (rc) {
        lod_free(s);
        return rc;
    }
    hipError_t e = hipMalloc(&s->C, nn * sizeof(double));
    if (e == hipSuccess) e = hipMalloc(&s->crhs, nodes * sizeof(double));
    s->ldw = d->capacity + kHistBlock;
    if (e == hipSuccess) e = hipMalloc(&s->w, (size_t)2 * s->ldw * sizeof(double));
    // far sums: a block past the first needs them (the MFMA form has its own)
    const int block = d->precision == FRM_PREC_SOE ? kSoeBlock : kHistBlock;
    if (e == hipSuccess && row_src(s) != kRowPart && !mf && d->capacity > block)
        e = hipMalloc(&s->far, sizeof(double) * 2 * block * s->hist->ld);
    if (e != hipSuccess) {
        lod_free(s);
        return check_hip(ctx, e, "hipMalloc(lod2d)");
    }
    // lag-indexed history weights: rows kb(s,1/2,0,1) at lag k = n-s is
    // d = k+1/2, l = 1; columns kb(s,1,0,1) is d = k+1, l = 1
    std::vector<double> w(2 * (size_t)d->capacity);
    for (int k = 1; k <= d->capacity && s->g_func == 0; ++k) {
        if (is_ab) {
            w[k - 1] = w[d->capacity + k - 1] = 0.5 * abI(k + 1);
        } else {
            w[k - 1] = caputo_kb(d->alpha, d->tau, k + 0.5, 1.0);
            w[d->capacity + k - 1] = caputo_kb(d->alpha, d->tau, k + 1.0, 1.0);
        }
    }
    // restricted summation (dt_alg = 2): the sums run newest first and stop
    // at the first |kb| < trunc_eps; the Caputo weights fall with the lag,
    // so each direction keeps its leading lags and the kernel reads the
    // newest trunc_L = max of the two
    s->trunc_L = d->capacity;
    if (d->trunc_eps > 0) {
        int keep[2] = {0, 0};
        for (int t = 0; t < 2; ++t) {
            double* wt = w.data() + (size_t)t * d->capacity;
            int k = 0;
            while (k < d->capacity && !(std::fabs(wt[k]) < d->trunc_eps)) ++k;
            keep[t] = k;
            for (; k < d->capacity; ++k) wt[k] = 0.0;
        }
        s->trunc_L = std::max(keep[0], keep[1]);
    }
    // line coefficients
    std::vector<double> rc3((size_t)3 * (d->M - 1) * s->NX), cc3((size_t)3 * (d->sN - 1) * s->NY);
    const int64_t lrows = d->M - 1, lcols = d->sN - 1;
    for (int j = 1; j < d->M; ++j) {
        const int64_t base = (int64_t)j * s->ld + 1;
        double* oa = rc3.data() + (int64_t)(j - 1) * s->NX;
        line_coefs(s->NX, d->rowA + base, d->rowB + base, 1, s->sg * s->kr0, 0.0, oa,
                   oa + lrows * s->NX, oa + 2 * lrows * s->NX);
    }
    for (int i = 1; i < d->sN; ++i) {
        const int64_t base = (int64_t)1 * s->ld + i;
        double* oa = cc3.data() + (int64_t)(i - 1) * s->NY;
        line_coefs(s->NY, d->colA + base, d->colB + base, s->ld, s->sg * s->kc0, 1.0, oa,
                   oa + lcols * s->NY, oa + 2 * lcols * s->NY);
    }
    // all lines alike: one is stored (the small path keeps its own layout)
    s->small = takes_small(s, d);
    s->rsame = !s->small && same_lines(rc3.data(), 3, d->M - 1, s->NX);
    s->csame = !s->small && same_lines(cc3.data(), 3, d->sN - 1, s->NY);
    if (s->g_func == 3) {
        // the lines' off-diagonals for the per-step coefficient kernel
        const int64_t nr = lrows * s->NX, nc = lcols * s->NY;
        std::vector<double> ab((size_t)2 * (nr + nc));
        for (int j = 1; j < d->M; ++j)
            for (int i = 1; i < d->sN; ++i) {
                const int64_t q = (int64_t)j * s->ld + i;
                ab[(j - 1) * s->NX + (i - 1)] = d->rowA[q];
                ab[nr + (j - 1) * s->NX + (i - 1)] = d->rowB[q];
                ab[2 * nr + (i - 1) * s->NY + (j - 1)] = d->colA[q];
                ab[2 * nr + nc + (i - 1) * s->NY + (j - 1)] = d->colB[q];
            }
        s->rsame = same_lines(ab.data(), 2, d->M - 1, s->NX);
        s->csame = same_lines(ab.data() + 2 * nr, 2, d->sN - 1, s->NY);
        e = hipMalloc(&s->lineAB, ab.size() * sizeof(double));
        if (e == hipSuccess) e = hipMalloc(&s->flag, sizeof(int));
        if (e == hipSuccess)
            e = hipMemcpy(s->lineAB, ab.data(), ab.size() * sizeof(double), hipMemcpyHostToDevice);
        if (e == hipSuccess) e = hipMemset(s->flag, 0, sizeof(int));
        if (e != hipSuccess) {
            lod_free(s);
            return check_hip(ctx, e, "hipMalloc(lod2d g = t^p)");
        }
    }
    // coefficient buffers sized for the longest padded line of any shape
    auto padded = [](int n) {
        int mx = 0;
        for (int W : {1, 2, 4})
            if (pick_cm(n, W)) mx = std::max(mx, pick_cm(n, W) * kWave * W);
        return mx;
    };
    e = hipMalloc(&s->rcoef,
                  (size_t)3 * (s->rsame ? 1 : d->M - 1) * padded(s->NX) * sizeof(double));
    if (e == hipSuccess)
        e = hipMalloc(&s->ccoef,
                      (size_t)3 * (s->csame ? 1 : d->sN - 1) * padded(s->NY) * sizeof(double));
    if (e != hipSuccess) {
        lod_free(s);
        return check_hip(ctx, e, "hipMalloc(lod2d coefficients)");
    }
    s->hw.assign({s->kr0, s->kc0, s->kch});
    s->hw.insert(s->hw.end(), w.begin(), w.end());
    std::vector<double> near_w;  // SOE with FP64 states: [2][kSoeBlock] weights by lag
    if (d->precision == FRM_PREC_SOE) {
        s->soe_L = d->soe_terms > 0 ? d->soe_terms : 32;
        s->soe_w1r = w[0];
        s->soe_w1c = w[d->capacity];
        frm::SoeFit fit = frm::soe_fit({w.data(), w.data() + d->capacity}, d->capacity, kSoeLag0,
                                       s->soe_L, d->tau);
        s->soe_err = fit.max_rel;
        // a fit that misses the weights by more than the chosen forms' error
        // bar (or is not finite) is refused rather than run
        if (!(fit.max_rel <= kSoeFitTol)) {
            lod_free(s);
            return set_error(ctx, FRM_E_INVALID,
                             "frm_lod2d_create: the %d-term exponential sum fits the history "
                             "weights to %.3g relative (limit %.0e)%s",
                             d->soe_terms > 0 ? d->soe_terms : 32, fit.max_rel, kSoeFitTol,
                             is_ab && !d->ab_exact ? "; truncated AB weights: set ab_exact" : "");
        }
        const size_t hsz = (s->soe_f32 ? sizeof(float) : sizeof(double)) * (size_t)s->soe_L * s->hist->ld;
        e = hipMalloc(&s->soe_H, hsz);
        if (s->soe_f32) {
            if (e == hipSuccess) e = hipMalloc(&s->soe_q, sizeof(double) * s->soe_L);
            if (e == hipSuccess) e = hipMalloc(&s->soe_c, sizeof(double) * 2 * s->soe_L);
            if (e == hipSuccess) e = hipMemcpy(s->soe_q, fit.q.data(), sizeof(double) * s->soe_L, hipMemcpyHostToDevice);
            if (e == hipSuccess) e = hipMemcpy(s->soe_c, fit.c.data(), sizeof(double) * 2 * s->soe_L, hipMemcpyHostToDevice);
        } else {
            // a block's factors per mode, and the near weights: the exact one
            // at lag 1, then the fitted sum's
            constexpr int J = kSoeBlock;
            const int L = s->soe_L;
            std::vector<double> tab((size_t)L * kSoeTab);
            near_w.assign(2 * J, 0.0);
            for (int l = 0; l < L; ++l) {
                double* f = tab.data() + (size_t)l * kSoeTab;
                const double q = fit.q[l];
                for (int k = 0; k < J - 1; ++k) f[k] = std::pow(q, J - 1 - k);
                f[J - 1] = std::pow(q, J);
                for (int t = 0; t < 2; ++t)
                    for (int j = 0; j < J; ++j) {
                        f[(1 + t) * J + j] = fit.c[(size_t)t * L + l] * std::pow(q, j);
                        if (j + 2 <= J) near_w[t * J + j + 1] += f[(1 + t) * J + j];
                    }
            }
            near_w[0] = s->soe_w1r;
            near_w[J] = s->soe_w1c;
            if (e == hipSuccess) e = hipMalloc(&s->soe_tab, sizeof(double) * tab.size());
            if (e == hipSuccess)
                e = hipMemcpy(s->soe_tab, tab.data(), sizeof(double) * tab.size(), hipMemcpyHostToDevice);
        }
        if (e == hipSuccess) e = hipMemset(s->soe_H, 0, hsz);
        if (e != hipSuccess) {
            lod_free(s);
            return check_hip(ctx, e, "hipMalloc(lod2d SOE)");
        }
    }
    if (d->precision == FRM_PREC_BINOMIAL) {
        s->bin_terms = d->series_terms > 0 ? d->series_terms : 25;
        s->bin_Da = 1.0 / gamma_cody(1.0 - d->alpha);
        const frm::BinomialTables bt = frm::binomial_tables(
            d->alpha, d->tau, d->series_tol > 0 ? d->series_tol : 1e-5, s->bin_terms, d->capacity);
        const size_t hsz = sizeof(double) * 2 * (size_t)s->bin_terms * s->hist->ld;
        const size_t tsz = std::max<size_t>(1, bt.upd.size());
        e = hipMalloc(&s->bin_H, hsz);
        if (e == hipSuccess) e = hipMalloc(&s->bin_upd, sizeof(double) * tsz);
        if (e == hipSuccess) e = hipMalloc(&s->bin_er, sizeof(double) * tsz);
        if (e == hipSuccess) e = hipMalloc(&s->bin_ec, sizeof(double) * tsz);
        if (e == hipSuccess) e = hipMalloc(&s->bin_cnt, sizeof(int) * std::max<size_t>(1, bt.cnt.size()));
        if (e == hipSuccess && !bt.upd.empty()) {
            e = hipMemcpy(s->bin_upd, bt.upd.data(), sizeof(double) * bt.upd.size(), hipMemcpyHostToDevice);
            if (e == hipSuccess) e = hipMemcpy(s->bin_er, bt.er.data(), sizeof(double) * bt.er.size(), hipMemcpyHostToDevice);
            if (e == hipSuccess) e = hipMemcpy(s->bin_ec, bt.ec.data(), sizeof(double) * bt.ec.size(), hipMemcpyHostToDevice);
            if (e == hipSuccess) e = hipMemcpy(s->bin_cnt, bt.cnt.data(), sizeof(int) * bt.cnt.size(), hipMemcpyHostToDevice);
        }
        if (e == hipSuccess) e = hipMemset(s->bin_H, 0, hsz);
        if (e != hipSuccess) {
            lod_free(s);
            return check_hip(ctx, e, "hipMalloc(lod2d binomial)");
        }
    }
    if (d->precision == FRM_PREC_IAIBK) {
        // both directions' plans for the whole capacity, (a, b) = (3/2, 1/2)
        // for rows and (2, 1) for columns (Om1, fr_d_t_g_2d.cpp:3443-3458)
        const double A = 1.0 - d->alpha;
        frm::IaPlan pl[2] = {frm::iaibk_plan(A, 1.5, 0.5, d->capacity),
                             frm::iaibk_plan(A, 2.0, 1.0, d->capacity)};
        s->ia_slots = std::max(1, std::max(pl[0].nslots, pl[1].nslots));
        for (int k = 0; k < frm::kIaMaxAk; ++k) s->ia_ak[k] = pl[0].ak[k];
        s->ia_scale = (1.0 / gamma_cody(1.0 - d->alpha)) * (std::pow(d->tau, 1.0 - d->alpha) / (1.0 - d->alpha));
        e = hipMalloc(&s->ia_H, sizeof(double) * 2 * (size_t)s->ia_slots * frm::kIaMaxAk * s->hist->ld);
        for (int t = 0; t < 2 && e == hipSuccess; ++t) {
            s->ia_off[t] = pl[t].step_off;
            e = hipMalloc(&s->ia_ops[t], sizeof(frm::IaOp) * std::max<size_t>(1, pl[t].ops.size()));
            if (e == hipSuccess) e = hipMalloc(&s->ia_vals[t], sizeof(double) * std::max<size_t>(1, pl[t].vals.size()));
            if (e == hipSuccess && !pl[t].ops.empty())
                e = hipMemcpy(s->ia_ops[t], pl[t].ops.data(), sizeof(frm::IaOp) * pl[t].ops.size(),
                              hipMemcpyHostToDevice);
            if (e == hipSuccess && !pl[t].vals.empty())
                e = hipMemcpy(s->ia_vals[t], pl[t].vals.data(), sizeof(double) * pl[t].vals.size(),
                              hipMemcpyHostToDevice);
        }
        if (e != hipSuccess) {
            lod_free(s);
            return check_hip(ctx, e, "hipMalloc(lod2d ia/ibk)");
        }
    }
    if (mf) {
        // BF16 parts of the FP64 weights: w = p0 + p1 + p2 + O(2^-24 w)
        // default parts: two for the Caputo weights (whose products are
        // dominated by the few large recent lags), three for the bounded AB
        // kernel, whose slowly decaying weights make the far part a large
        // share of the memory term
        const int nparts = d->mfma_parts ? d->mfma_parts : (is_ab ? 3 : 2);
        s->mfma_nprod = nparts == 2 ? 3 : 6;
        std::vector<float> parts(3 * w.size());
        for (size_t k = 0; k < w.size(); ++k) {
            double r = w[k];
            for (int p = 0; p < 3; ++p) {
                parts[p * w.size() + k] = bf16_round(r);
                r -= (double)parts[p * w.size() + k];
            }
        }
        // d = 32 .. N0 + 32 for the largest block start N0 below the capacity
        s->atab_chunks = std::max(1, (d->capacity - 1) / kBlockSteps * kBlockSteps / kFarChunk) + 1;
        // slices of about one round of far-product workgroups (two per CU:
        // a launch of whole rounds keeps every CU busy to its end), at most
        // one per step
        {
            const int groups = block_far_groups(s->hist->ld);
            const int round = block_far_round(ctx->device);
            if (round <= 0) {
                lod_free(s);
                return set_error(ctx, FRM_E_HIP, "frm_lod2d_create: CU count of device %d",
                                 ctx->device);
            }
            s->far_slices = std::max(1, std::min(kBlockSteps, (groups + round - 1) / round));
        }
        const std::vector<uint16_t> tab = atab_build(parts.data(), d->capacity, s->atab_chunks);
        e = hipMalloc(&s->atab, tab.size() * sizeof(uint16_t));
        // two far buffers: the current block's and the next one's, formed in slices
        if (e == hipSuccess) e = hipMalloc(&s->F, sizeof(float) * 2 * 2 * kBlockSteps * s->hist->ld);
        if (e == hipSuccess) e = hipMalloc(&s->G, sizeof(float) * 2 * kMidBlock * s->hist->ld);
        if (e == hipSuccess)
            e = hipMemcpy(s->atab, tab.data(), tab.size() * sizeof(uint16_t), hipMemcpyHostToDevice);
        if (e != hipSuccess) {
            lod_free(s);
            return check_hip(ctx, e, "hipMalloc(lod2d MFMA)");
        }
    }
    {
        std::vector<double> wp((size_t)2 * s->ldw, 0.0);
        for (int t = 0; t < 2 && !near_w.empty(); ++t)
            std::copy(near_w.begin() + t * kSoeBlock, near_w.begin() + (t + 1) * kSoeBlock,
                      wp.begin() + (size_t)t * s->ldw);
        for (int t = 0; t < 2 && near_w.empty(); ++t)
            std::copy(w.begin() + (size_t)t * d->capacity, w.begin() + (size_t)(t + 1) * d->capacity,
                      wp.begin() + (size_t)t * s->ldw);
        // FP32 increments go with FP32 weights; the sums over both are FP64
        if (s->precision == FRM_PREC_F32C)
            for (double& q : wp) q = (double)(float)q;
        e = hipMemcpy(s->w, wp.data(), wp.size() * sizeof(double), hipMemcpyHostToDevice);
    }
    if (e == hipSuccess) e = hipMemset(s->C, 0, nn * sizeof(double));
    if (e != hipSuccess) {
        lod_free(s);
        return check_hip(ctx, e, "hipMemcpy(lod2d setup)");
    }
    double *rplain = s->rcoef, *cplain = s->ccoef;  // the small path reads them as they are
    if (!s->small) {
        rplain = cplain = nullptr;
        e = hipMalloc(&rplain, rc3.size() * sizeof(double));
        if (e == hipSuccess) e = hipMalloc(&cplain, cc3.size() * sizeof(double));
    }
    if (e == hipSuccess)
        e = hipMemcpy(rplain, rc3.data(), rc3.size() * sizeof(double), hipMemcpyHostToDevice);
    if (e == hipSuccess)
        e = hipMemcpy(cplain, cc3.data(), cc3.size() * sizeof(double), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        rc = check_hip(ctx, e, "sweep coefficients");
    } else if (s->small) {
        s->rsh = SweepShape{pick_cm(s->NX, 1), 1};
        s->csh = SweepShape{pick_cm(s->NY, 1), 1};
    } else {
        rc = tune_sweeps(s, d->sweep_w, rplain, cplain);
    }
    if (!s->small) {
        (void)hipStreamSynchronize(ctx->stream);
        (void)hipFree(rplain);
        (void)hipFree(cplain);
    }
    if (rc) {
        lod_free(s);
        return rc;
    }
    // leave no trace of the tuning runs: zero state, right-hand sides and history slots
    {
        const size_t hb = (s->precision == FRM_PREC_MFMA_BF16 || s->precision == FRM_PREC_F32C
                               ? sizeof(float)
                               : sizeof(double)) *
                          (size_t)std::min(s->hist->capacity, std::max(s->ring, 1)) * s->hist->ld;
        e = hipMemset(s->C, 0, nn * sizeof(double));
        if (e == hipSuccess) e = hipMemset(s->crhs, 0, nodes * sizeof(double));
        if (e == hipSuccess) e = hipMemset(s->hist->data, 0, hb);
        if (e != hipSuccess) {
            lod_free(s);
            return check_hip(ctx, e, "hipMemset(lod2d after tuning)");
        }
    }
    *out = s;
    return FRM_OK;
}

int frm_lod2d_destroy(frm_lod2d* s) {
    if (!s) return FRM_OK;
    (void)hipStreamSynchronize(s->ctx->stream);
    lod_free(s);
    return FRM_OK;
}

int frm_lod2d_set_state(frm_lod2d* s, const double* h_C) {
    if (!s || !h_C) return set_error(s ? s->ctx : nullptr, FRM_E_INVALID, "frm_lod2d_set_state: null");
    frm_ctx* ctx = s->ctx;
    FRM_HIP(ctx, hipMemcpyAsync(s->C, h_C, (size_t)s->ld * (s->M + 2) * sizeof(double),
                                hipMemcpyHostToDevice, ctx->stream));
    FRM_HIP(ctx, hipStreamSynchronize(ctx->stream));
    s->tstep = 0;
    s->hist->depth = 0;
    if (s->soe_H) {
        const size_t hsz = (s->soe_f32 ? sizeof(float) : sizeof(double)) * (size_t)s->soe_L * s->hist->ld;
        FRM_HIP(ctx, hipMemsetAsync(s->soe_H, 0, hsz, ctx->stream));
        FRM_HIP(ctx, hipStreamSynchronize(ctx->stream));
    }
    if (s->bin_H) {
        const size_t hsz = sizeof(double) * 2 * (size_t)s->bin_terms * s->hist->ld;
        FRM_HIP(ctx, hipMemsetAsync(s->bin_H, 0, hsz, ctx->stream));
        FRM_HIP(ctx, hipStreamSynchronize(ctx->stream));
    }
    return FRM_OK;
}

int frm_lod2d_step(frm_lod2d* s, int32_t nsteps) {
    if (!s) return set_error(nullptr, FRM_E_INVALID, "frm_lod2d_step: null solver");
    frm_ctx* ctx = s->ctx;
    FRM_REQUIRE(ctx, nsteps >= 0, "frm_lod2d_step: nsteps %d", nsteps);
    const bool soe = s->precision == FRM_PREC_SOE;
    const bool mf = s->precision == FRM_PREC_MFMA_BF16;
    const bool bin = s->precision == FRM_PREC_BINOMIAL;
    const bool iab = s->precision == FRM_PREC_IAIBK;
    if (s->tstep + nsteps > s->capacity)
        return set_error(ctx, FRM_E_RANGE, "frm_lod2d_step: %d steps exceed capacity %d",
                         s->tstep + nsteps, s->capacity);
    for (const int goal = s->tstep + nsteps; s->tstep < goal;) {
        const int n = s->tstep;
        int nch = 0;
        bool far = false, mid = false;
        if (s->g_func == 3) {
            const int rc = gpow_prepare(s, n);
            if (rc) return rc;
        }
        if (soe && s->soe_f32) {
            nch = 1;
            const int64_t ld = s->hist->ld;
            LaunchTimer t(ctx, FRM_K_MEMTERM, (double)ld * (2.0 * s->soe_L * 4 + 2 * 8 + 2 * 8));
            const dim3 grid((unsigned)((ld + 255) / 256));
            auto kern = (double)ld * s->soe_L * 4 >= kStreamBypassBytes ? k_soe_memterm<true>
                                                                       : k_soe_memterm<false>;
            hipLaunchKernelGGL(kern, grid, dim3(256), 0, ctx->stream, (float*)s->soe_H,
                               (const double*)s->hist->data, ld, n, s->soe_L, s->soe_q, s->soe_c,
                               s->soe_w1r, s->soe_w1c, s->hist->part);
            FRM_HIP(ctx, hipGetLastError());
        } else if (soe) {
            // the modes advance, and the block's far sums are formed, once per block
            nch = 1;
            const int64_t ld = s->hist->ld;
            far = n >= kSoeBlock;
            if (far && n % kSoeBlock == 0) {
                LaunchTimer t(ctx, FRM_K_MEMTERM,
                              (double)ld * 8 * (2.0 * s->soe_L + 3.0 * kSoeBlock));
                const dim3 grid((unsigned)((ld + 255) / 256));
                auto kern = (double)ld * s->soe_L * 8 >= kStreamBypassBytes ? k_soe_block<true>
                                                                           : k_soe_block<false>;
                hipLaunchKernelGGL(kern, grid, dim3(256), 0, ctx->stream, (double*)s->soe_H,
                                   (const double*)s->hist->data, ld, n, s->soe_L, s->soe_tab, s->far);
                FRM_HIP(ctx, hipGetLastError());
            }
        } else if (iab) {
            // nothing to sum before the first increment
            nch = n > 0 ? 1 : 0;
            if (n > 0) {
                IaArgs a;
                a.H = s->ia_H;
                a.ring = (const double*)s->hist->data;
                a.ld = s->hist->ld;
                a.n = n;
                a.slots = s->ia_slots;
                for (int t = 0; t < 2; ++t) {
                    a.ops[t] = s->ia_ops[t];
                    a.vals[t] = s->ia_vals[t];
                    a.o0[t] = s->ia_off[t][n - 1];
                    a.o1[t] = s->ia_off[t][n];
                }
                for (int k = 0; k < kIaMaxAk; ++k) a.ak[k] = s->ia_ak[k];
                a.scale = s->ia_scale;
                a.part = s->hist->part;
                LaunchTimer t(ctx, FRM_K_MEMTERM, 0.0);
                hipLaunchKernelGGL(k_iaibk_memterm, dim3((unsigned)(a.ld / 256)), dim3(256), 0,
                                   ctx->stream, a);
                FRM_HIP(ctx, hipGetLastError());
            }
        } else if (bin) {
            nch = 1;
            const int64_t ld = s->hist->ld;
            LaunchTimer t(ctx, FRM_K_MEMTERM, (double)ld * (2.0 * s->bin_terms * 16 + 8 + 2 * 8));
            hipLaunchKernelGGL(k_binomial_memterm, dim3((unsigned)((ld + 255) / 256)), dim3(256), 0,
                               ctx->stream, s->bin_H, (const double*)s->hist->data, ld, n,
                               s->bin_terms, s->bin_upd, s->bin_er, s->bin_ec, s->bin_cnt, s->bin_Da,
                               s->hist->part);
            FRM_HIP(ctx, hipGetLastError());
        } else if (mf) {
            // block b = n / 64 uses the far part of the slots before P0 =
            // N0 - 64 (F of parity b), formed during block b - 1; this
            // block's steps N0 + q 64/S form, slice q of S, the next block's
            // far part (slots before N0, all settled) into F of parity b + 1
            const int64_t ld = s->hist->ld;
            const int N0 = n / kBlockSteps * kBlockSteps;
            const int P0 = std::max(0, N0 - kBlockSteps);
            const float* h32 = (const float*)s->hist->data;
            const size_t fsz = (size_t)2 * kBlockSteps * ld;
            float* Fnext = s->F + (size_t)(((N0 / kBlockSteps) + 1) & 1) * fsz;
            const int every = kBlockSteps / s->far_slices;
            const int q = (n - N0) / every;
            if (N0 > 0 && N0 + kBlockSteps < s->capacity && (n - N0) % every == 0) {
                const int groups = block_far_groups(ld);
                const int per = (groups + s->far_slices - 1) / s->far_slices;
                const int wg0 = q * per, nwg = std::min(per, groups - wg0);
                if (nwg > 0) {
                    const double nodes = (double)s->hist->n_nodes * nwg / groups;
                    LaunchTimer t(ctx, FRM_K_BLOCKFAR, nodes * (4.0 * N0 + 4.0 * 2 * kBlockSteps));
                    if (block_far(ctx->stream, h32, ld, N0 + kBlockSteps, N0, s->atab, s->atab_chunks,
                                  s->mfma_nprod, Fnext, wg0, nwg))
                        return check_hip(ctx, hipGetLastError(), "block_far");
                }
            }
            // the slots from P0 up to the sub-block start, once per sub-block,
            // summed in FP64; the row kernel adds the newest ones
            const int N1 = n / kMidBlock * kMidBlock;
            nch = 1;
            far = P0 > 0;
            mid = N1 > P0;
            if (mid && n == N1) {
                LaunchTimer t(ctx, FRM_K_MEMTERM,
                              (double)ld * ((N1 - P0) * 4.0 + 2 * kMidBlock * 4));
                if (hist_far(ctx->stream, h32, ld, P0, N1, s->w, s->ldw, s->G))
                    return check_hip(ctx, hipGetLastError(), "hist_far");
            }
        } else if (s->g_func == 3) {
            int rc = memterm_partials(ctx, s->hist, 2, s->w, s->ldw, &nch);
            if (rc) return rc;
        } else {
            // the far sums of the block that starts here; the row kernel
            // adds the block's own slots.  Restricted sums leave out the
            // slots beyond their longest lag, whose weights are zero.
            nch = 1;
            const int N0 = n / kHistBlock * kHistBlock;
            const int first = std::max(0, N0 - s->trunc_L);
            far = first < N0;
            if (far && n == N0) {
                const bool f32 = s->precision == FRM_PREC_F32C;
                LaunchTimer t(ctx, FRM_K_MEMTERM,
                              (double)s->hist->n_nodes *
                                  ((double)(N0 - first) * (f32 ? 4 : 8) + 2.0 * kHistBlock * 8));
                const int rc = f32 ? hist_far(ctx->stream, (const float*)s->hist->data, s->hist->ld,
                                              first, N0, s->w, s->ldw, s->far)
                                   : hist_far(ctx->stream, (const double*)s->hist->data, s->hist->ld,
                                              first, N0, s->w, s->ldw, s->far);
                if (rc) return check_hip(ctx, hipGetLastError(), "hist_far");
            }
        }
        if (s->small) {
            const int ks = std::min(goal - n, n / kHistBlock * kHistBlock + kHistBlock - n);
            LaunchTimer t(ctx, FRM_K_ROWS, 0.0);
            FRM_HIP(ctx, launch_small(s, n, ks, far));
            s->hist->depth += ks;
            s->tstep = n + ks;
            continue;
        }
        {
            LaunchTimer t(ctx, FRM_K_ROWS, 0.0);
            FRM_HIP(ctx, launch_rows(s, ctx->stream, row_args(s, nch, n, far, mid)));
        }
        {
            LaunchTimer t(ctx, FRM_K_COLS, 0.0);
            FRM_HIP(ctx, launch_cols(s->csh, ctx->stream, col_args(s, n)));
        }
        if (!soe && !bin && !iab) s->hist->depth += 1;
        s->tstep = n + 1;
    }
    return FRM_OK;
}

int frm_lod2d_get_state(frm_lod2d* s, double* h_C) {
    if (!s || !h_C) return set_error(s ? s->ctx : nullptr, FRM_E_INVALID, "frm_lod2d_get_state: null");
    frm_ctx* ctx = s->ctx;
    FRM_HIP(ctx, hipMemcpyAsync(h_C, s->C, (size_t)s->ld * (s->M + 2) * sizeof(double),
                                hipMemcpyDeviceToHost, ctx->stream));
    int flag = 0;
    if (s->flag)
        FRM_HIP(ctx, hipMemcpyAsync(&flag, s->flag, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
    FRM_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (flag)
        return set_error(ctx, FRM_E_STATE,
                         "frm_lod2d_get_state: a history-weight series did not reach int_err");
    return FRM_OK;
}

int frm_lod2d_tstep(const frm_lod2d* s, int32_t* tstep) {
    if (!s || !tstep) return set_error(nullptr, FRM_E_INVALID, "frm_lod2d_tstep: null");
    *tstep = s->tstep;
    return FRM_OK;
}

int frm_lod2d_fit_error(const frm_lod2d* s, double* max_rel) {
    if (!s || !max_rel) return set_error(nullptr, FRM_E_INVALID, "frm_lod2d_fit_error: null");
    *max_rel = s->soe_err;
    return FRM_OK;
}

int frm_lod2d_weights(const frm_lod2d* s, int32_t n, double* out) {
    if (!s || !out || n < 0 || n > s->capacity)
        return set_error(nullptr, FRM_E_INVALID, "frm_lod2d_weights: bad arguments");
    if (s->g_func == 3) {
        // the weights of step n, computed on the host as the step computes them
        bool capped = false;
        gpow_current(s, n, &out[0], &out[1], &out[2], &capped);
        for (int k = 0; k < n; ++k) {
            out[3 + k] = s->Da * kb_pow(s->alpha, s->tau, s->g_pow, s->int_err, n, n - 1 - k, 0.5,
                                        0.0, 1.0, &capped);
            out[3 + n + k] = s->Da * kb_pow(s->alpha, s->tau, s->g_pow, s->int_err, n, n - 1 - k,
                                            1.0, 0.0, 1.0, &capped);
        }
        return capped ? set_error(nullptr, FRM_E_STATE, "frm_lod2d_weights: series bound") : FRM_OK;
    }
    out[0] = s->hw[0];
    out[1] = s->hw[1];
    out[2] = s->hw[2];
    for (int k = 0; k < n; ++k) {
        out[3 + k] = s->hw[3 + k];
        out[3 + n + k] = s->hw[3 + s->capacity + k];
    }
    return FRM_OK;
}

int frm_lod2d_far_slices(const frm_lod2d* s, int32_t* slices) {
    if (!s || !slices) return set_error(nullptr, FRM_E_INVALID, "frm_lod2d_far_slices: null");
    *slices = s->precision == FRM_PREC_MFMA_BF16 ? s->far_slices : 0;
    return FRM_OK;
}

int frm_lod2d_sweep_shape(const frm_lod2d* s, int32_t* out) {
    if (!s || !out) return set_error(nullptr, FRM_E_INVALID, "frm_lod2d_sweep_shape: null");
    out[0] = s->rsh.cm;
    out[1] = s->rsh.w;
    out[2] = s->csh.cm;
    out[3] = s->csh.w;
    return FRM_OK;
}

int frm_lod2d_state_ptr(frm_lod2d* s, double** d_C) {
    if (!s || !d_C) return set_error(nullptr, FRM_E_INVALID, "frm_lod2d_state_ptr: null");
    *d_C = s->C;
    return FRM_OK;
}

}  // extern "C"
