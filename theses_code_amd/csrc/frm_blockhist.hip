// Blocked history sums in FP64 on the matrix cores.
//
// For weights that depend on the lag only, the history sums of the steps
// n = N0 + j, j < J = kHistBlock, of a block share their settled past:
//   S_t(n) = sum_{s < N0} w_t(N0 + j - s) Delta_s + sum_{N0 <= s < n} w_t(n - s) Delta_s.
// The first part, for all J steps and both targets of the LOD scheme, is one
// dense FP64 product W (2 J x N0) times Delta (N0 x nodes), formed once when
// the block starts; the step's own kernel adds the at most J - 1 newer slots.
// The history is then read once per J steps instead of every step; the
// multiplications are the same ones, rounded in FP64 as before and summed in
// another order.  The reference forms every step's sum from scratch
// (fr_d_t_g_2d.cpp:3340-3437).
//
// Measured (512 x 512 FP64, 1000 steps): the pass over the history went from
// 150 us per step (7.0 TB/s) to 177 us per 16 steps plus 4 us per step for the
// newest slots in the row kernel, the run from 166 to 25.8 ms; 1024 x 1024
// with FP32 increments, 500 steps: from 110 to 26.7 ms.  J = 16 makes each
// target one 16-row tile: 64 multiply-adds per FP64 value read, 16 per byte
// and target pair, so the product takes about as long on the matrix cores
// (70 TFLOP/s) as its read from memory.
//
// FP32 sums (the MFMA form's mid sums) are rounded, and where a block ends decides
// what is rounded: they keep blocks of kMidBlock = 8 steps, both targets in one
// 16-row tile (1024 x 1024, 64 to 120 slots: 90 us, 5.0 TB/s).  Blocks of 16 took
// 116 us for twice the steps but 4 us more per step in the rows, and moved that
// form's results by up to 3e-9 of themselves.
#include "frm_blockhist.hpp"

#include <type_traits>

namespace frm {

typedef double f64x4 __attribute__((ext_vector_type(4)));

// Nodes of a wavefront's tile: column tile c (16 columns, one per lane % 16)
// holds nodes i0 + node_of<NC, HT>(c, lane % 16), chosen so that a lane's
// nodes come in contiguous loads of up to 16 bytes.
template <int NC, typename HT>
__device__ __forceinline__ int node_of(int c, int m) {
    if constexpr (NC == 1) return m;
    else if constexpr (sizeof(HT) == 4) return 4 * m + c;
    else return 32 * (c >> 1) + 2 * m + (c & 1);
}

// One slot's values of a lane's NC nodes (`p` points at node i0 of the slot).
template <int NC, typename HT>
__device__ __forceinline__ void load_nodes(const HT* p, int m, double (&x)[NC]) {
    if constexpr (NC == 1) {
        x[0] = (double)__builtin_nontemporal_load(p + m);
    } else if constexpr (sizeof(HT) == 4) {
        typedef float v4 __attribute__((ext_vector_type(4)));
        const v4 v = __builtin_nontemporal_load(reinterpret_cast<const v4*>(p + 4 * m));
#pragma unroll
        for (int c = 0; c < 4; ++c) x[c] = (double)v[c];
    } else {
        typedef double v2 __attribute__((ext_vector_type(2)));
#pragma unroll
        for (int h = 0; h < NC / 2; ++h) {
            const v2 v = __builtin_nontemporal_load(reinterpret_cast<const v2*>(p + 32 * h + 2 * m));
            x[2 * h] = v.x;
            x[2 * h + 1] = v.y;
        }
    }
}

// Wavefront tile: 2 targets x 16 steps (one 16-row tile each; FP32 sums: 2 x 8
// steps, one tile) by 16 NC nodes, on v_mfma_f64_16x16x4_f64: per 4 slots a lane
// holds A[i = l%16][k = l/16] = w_t(N0 + i - s0 - k) (w_{i/8}(N0 + i%8 - ...)), B[k = l/16][l%16] = Delta_{s0+k} and, per tile, the
// four rows 4 r + l/16 of D.  Loads run two products ahead (512 x 512 FP64 at
// 500 slots: 238 -> 177 us, 6.3 TB/s; held to three wavefronts per SIMD, the
// sums stay in ordinary registers: 190 us otherwise).  KS wavefronts of a workgroup share a tile's
// slots and add their sums through LDS in wavefront order, so that a small
// grid, which has too few tiles to fill the chip, still uses all of it.
template <typename HT, typename GT, int NC, int KS>
__global__ __launch_bounds__(KS == 1 ? 256 : 64 * KS) __attribute__((amdgpu_waves_per_eu(3, 8))) void k_hist_far(
    const HT* __restrict__ hist, int64_t ld, int first, int N0, const double* __restrict__ w,
    int ldw, GT* __restrict__ G) {
    constexpr int T = sizeof(GT) == 4 ? 1 : 2;  // 16-row tiles
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int m = lane & 15, kg = lane >> 4;
    const int64_t tile = KS == 1 ? (int64_t)blockIdx.x * 4 + wv : blockIdx.x;
    const int64_t i0 = tile * (16 * NC);
    if (i0 >= ld) return;  // KS > 1: the grid is exact, so a whole workgroup or none
    int a = first, b = N0;
    if constexpr (KS > 1) {
        const int per = ((N0 - first) / 4 + KS - 1) / KS * 4;
        a = min(N0, first + wv * per);
        b = min(N0, a + per);
    }
    f64x4 acc[T][NC];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[t][c] = f64x4{0.0, 0.0, 0.0, 0.0};
    const HT* hp = hist + (int64_t)(a + kg) * ld + i0;
    const double* wp =
        w + (N0 - a - 1 - kg) + (T == 1 ? (m >> 3) * ldw + (m & (kMidBlock - 1)) : m);
    // two batches of U 4-slot products: one's loads are in flight during the
    // other's products
    constexpr int U = NC == 1 ? 4 : 2;
    double xa[U][NC], va[U][T], xb[U][NC], vb[U][T];
    auto load = [&](double (&x)[U][NC], double (&v)[U][T]) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            load_nodes<NC, HT>(hp + (int64_t)(4 * u) * ld, m, x[u]);
#pragma unroll
            for (int t = 0; t < T; ++t) v[u][t] = wp[t * ldw - 4 * u];
        }
        hp += (int64_t)(4 * U) * ld;
        wp -= 4 * U;
    };
    auto mul = [&](const double (&x)[U][NC], const double (&v)[U][T]) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int t = 0; t < T; ++t)
                    acc[t][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(v[u][t], x[u][c], acc[t][c], 0, 0, 0);
    };
    const int nb = (b - a) / (4 * U);
    int s = a + nb * 4 * U;
    if (nb > 0) load(xa, va);
    for (int k = 0; k < nb; k += 2) {
        if (k + 1 < nb) load(xb, vb);
        mul(xa, va);
        if (k + 2 < nb) load(xa, va);
        if (k + 1 < nb) mul(xb, vb);
    }
    for (; s < b; s += 4) {
        double x[NC];
        load_nodes<NC, HT>(hp, m, x);
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const double v = wp[t * ldw];
#pragma unroll
            for (int c = 0; c < NC; ++c)
                acc[t][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(v, x[c], acc[t][c], 0, 0, 0);
        }
        hp += 4 * ld;
        wp -= 4;
    }
    if constexpr (KS == 1) {
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                GT* g = G + (int64_t)(16 * t + 4 * r + kg) * ld + i0;
#pragma unroll
                for (int c = 0; c < NC; ++c) g[node_of<NC, HT>(c, m)] = (GT)acc[t][c][r];
            }
    } else {
        __shared__ double part[KS][T * NC * 4][64];
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int r = 0; r < 4; ++r) part[wv][(t * NC + c) * 4 + r][lane] = acc[t][c][r];
        __syncthreads();
        for (int q = wv; q < T * NC * 4; q += KS) {
            double v = 0.0;
#pragma unroll
            for (int p = 0; p < KS; ++p) v += part[p][q][lane];
            const int r = q & 3, c = (q >> 2) % NC, t = (q >> 2) / NC;
            G[(int64_t)(16 * t + 4 * r + kg) * ld + i0 + node_of<NC, HT>(c, m)] = (GT)v;
        }
    }
}

template <typename HT, typename GT>
static int far_launch(hipStream_t st, const HT* hist, int64_t ld, int first, int N0,
                      const double* w, int ldw, GT* G) {
    constexpr int J = sizeof(GT) == 4 ? kMidBlock : kHistBlock;
    if (!hist || !w || !G || ld <= 0 || ld % 1024 || N0 <= 0 || N0 % J || first < 0 ||
        first >= N0 || ldw < N0 + J - 1)
        return -1;
    first = first / 4 * 4;
    if (ld >= 262144) {
        hipLaunchKernelGGL((k_hist_far<HT, GT, 4, 1>), dim3((unsigned)(ld / 256)), dim3(256), 0, st,
                           hist, ld, first, N0, w, ldw, G);
    } else if (ld >= 32768) {
        hipLaunchKernelGGL((k_hist_far<HT, GT, 4, 4>), dim3((unsigned)(ld / 64)), dim3(256), 0, st, hist,
                           ld, first, N0, w, ldw, G);
    } else {
        hipLaunchKernelGGL((k_hist_far<HT, GT, 1, 8>), dim3((unsigned)(ld / 16)), dim3(512), 0, st, hist,
                           ld, first, N0, w, ldw, G);
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int hist_far(hipStream_t st, const double* hist, int64_t ld, int first, int N0, const double* w,
             int ldw, double* G) {
    return far_launch(st, hist, ld, first, N0, w, ldw, G);
}

int hist_far(hipStream_t st, const float* hist, int64_t ld, int first, int N0, const double* w,
             int ldw, double* G) {
    return far_launch(st, hist, ld, first, N0, w, ldw, G);
}

int hist_far(hipStream_t st, const float* hist, int64_t ld, int first, int N0, const double* w,
             int ldw, float* G) {
    return far_launch(st, hist, ld, first, N0, w, ldw, G);
}

}  // namespace frm
