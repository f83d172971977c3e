// cond.hip -- KPM conductivity moments (observable type 1) on the device.
//
// Replaces Locality::computeCondKPM (locality.cpp:6348-6727; real H, target
// starts) and Param_tools::matrixResponseTransform (param_tools.cpp:838-905).
// The reference builds beta_m = T_m(H) e_t (m < M), walks a_n = T_n(H) alpha_0
// with alpha_0 = -dxH e_t, and takes C[n][m] = (dxH a_n) . beta_m one dot
// product at a time: M^2 vector dots per target.  Here both vector sets are
// produced for a block of targets at once, one kernel per Chebyshev index
// writing straight into the [target][m][row] sets; C for every target is then
// an FP64 GEMM on the matrix cores (dgemm.hip) split into row chunks, and the 2D
// Jackson/DCT-III transform is two more GEMMs against the cosine matrix.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.h"
#include "kpm_common.h"

namespace leo2d {
namespace {

constexpr int kCondThreads = 256;

// set[(b * M + m) * n + i] = blk[i * B + b]: one Chebyshev vector block [n][B]
// stored as vector m of every target's set
__global__ __launch_bounds__(kCondThreads) void scatter_kernel(const double* __restrict__ blk, int n, int B, int m, int M,
                                                               double* __restrict__ set)
{
    const size_t total = (size_t)n * B;
    for (size_t t = blockIdx.x * (size_t)kCondThreads + threadIdx.x; t < total; t += (size_t)gridDim.x * kCondThreads) {
        const size_t i = t / B;
        const int b = (int)(t % B);
        set[((size_t)b * M + m) * n + i] = blk[t];
    }
}

// X[t][i][j] = 2 g_i g_j C[t][i][j] with the Jackson g_i / sqrt(2)
// (param_tools.cpp:857-890)
__global__ __launch_bounds__(kCondThreads) void cond_weight_kernel(const double* __restrict__ C, int M, int T,
                                                                   double* __restrict__ X)
{
    const size_t total = (size_t)T * M * M;
    const double pm = M_PI / M;
    for (size_t t = blockIdx.x * (size_t)kCondThreads + threadIdx.x; t < total; t += (size_t)gridDim.x * kCondThreads) {
        const int j = (int)(t % M);
        const int i = (int)((t / M) % M);
        const double gi = ((M - i) * cos(pm * i) + sin(pm * i) / tan(pm)) / (sqrt(2.0) * M);
        const double gj = ((M - j) * cos(pm * j) + sin(pm * j) / tan(pm)) / (sqrt(2.0) * M);
        X[t] = 2 * gi * gj * C[t];
    }
}

// column-major P(k, i) = w_i cos(pi i (k + 1/2) / M), w_0 = 1, w_i = 2 (FFTW
// REDFT01), the angle reduced exactly in integers: i (2k + 1) mod 4M
__global__ __launch_bounds__(kCondThreads) void dct3_matrix_kernel(int M, double* __restrict__ P)
{
    const size_t total = (size_t)M * M;
    const long long P4 = 4LL * M;
    for (size_t t = blockIdx.x * (size_t)kCondThreads + threadIdx.x; t < total; t += (size_t)gridDim.x * kCondThreads) {
        const int k = (int)(t % M);
        const int i = (int)(t / M);
        const long long m = ((long long)i * (2LL * k + 1)) % P4;
        const double c = cos(M_PI * (double)m / (2.0 * M));
        P[t] = i == 0 ? 1.0 : 2.0 * c;
    }
}

// C[b][q] = sum over the S row chunks c of part[b][c][q], in order c = 0, 1, ...
__global__ __launch_bounds__(kCondThreads) void chunk_sum_kernel(const double* __restrict__ part, int S, size_t mm,
                                                                 int B, double* __restrict__ C)
{
    const size_t total = (size_t)B * mm;
    for (size_t t = blockIdx.x * (size_t)kCondThreads + threadIdx.x; t < total; t += (size_t)gridDim.x * kCondThreads) {
        const size_t b = t / mm, q = t % mm;
        const double* p = part + b * S * mm + q;
        double s = 0.0;
        for (int c = 0; c < S; ++c) s += p[(size_t)c * mm];
        C[t] = s;
    }
}

// One Chebyshev index of the conductivity recursion for a block of B real
// vectors x = [n][B] (thread per (row, vector), rows in stored CSR order):
//   yh = alpha H x - (beta ? prev : 0)  -> out   [n][B] (the recursion; out may alias prev)
//   yd = dxH x                           -> dset[b][j][row] (written straight into the set)
// H and dxH share the pattern, so each entry's column and the gathered x are
// read once for both products.  With hx == nullptr only the dxH product is
// formed; with dx == nullptr only the H product, and hset (when given)
// receives yh as vector j of the set.
template <bool HAS_H, bool HAS_D>
__global__ __launch_bounds__(kCondThreads) void dual_step_kernel(const int64_t* __restrict__ rp,
                                                                 const int32_t* __restrict__ col,
                                                                 const double* __restrict__ hv,
                                                                 const double* __restrict__ dv, const double* x,
                                                                 const double* prev, double* out, double alpha, int beta,
                                                                 int n, int B, int j, int M, double* __restrict__ hset,
                                                                 double* __restrict__ dset)
{
    constexpr int U = 8;   // entries whose gathers are in flight together
    const size_t total = (size_t)n * B;
    for (size_t t = blockIdx.x * (size_t)kCondThreads + threadIdx.x; t < total; t += (size_t)gridDim.x * kCondThreads) {
        const int row = (int)(t / B);
        const int b = (int)(t % B);
        double ah = 0.0, ad = 0.0;
        int64_t q = rp[row];
        const int64_t e = rp[row + 1];
        for (; q + U <= e; q += U) {
            double xv[U];
#pragma unroll
            for (int u = 0; u < U; ++u) xv[u] = x[(size_t)col[q + u] * B + b];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (HAS_H) ah += hv[q + u] * xv[u];
                if (HAS_D) ad += dv[q + u] * xv[u];
            }
        }
        for (; q < e; ++q) {
            const double xv = x[(size_t)col[q] * B + b];
            if (HAS_H) ah += hv[q] * xv;
            if (HAS_D) ad += dv[q] * xv;
        }
        if (HAS_H) {
            const double y = alpha * ah - (beta ? prev[t] : 0.0);
            out[t] = y;
            if (hset) hset[((size_t)b * M + j) * n + row] = y;
        }
        if (HAS_D) dset[((size_t)b * M + j) * n + row] = ad;
    }
}

// The same index with 16 lanes per row (B <= 16 vectors, kpm_common.h): a row's
// entries and then its gathers are in flight together, where the kernel above walks
// them eight at a time and reads every column and value once per vector.  The
// gathers serve both products (95 k rows, 4 targets: 34.9 -> 18.2 us with both
// products, 20.4 -> 16.2 us with one; both recursions, us an index: 8 targets on 2.1 k /
// 23.6 k / 94.7 k rows 14.9 -> 8.3 / 24.4 -> 18.8 / 74.4 -> 52.9, 16 targets lanes_grid).
template <bool HAS_H, bool HAS_D, int B>
__global__ __launch_bounds__(kCondThreads) void dual_step_lanes_kernel(const int64_t* __restrict__ rp,
                                                                       const int32_t* __restrict__ col,
                                                                       const double* __restrict__ hv,
                                                                       const double* __restrict__ dv,
                                                                       const double* __restrict__ x, const double* prev,
                                                                       double* out, double alpha, int beta, int n, int j,
                                                                       int M, double* __restrict__ hset,
                                                                       double* __restrict__ dset)
{
    constexpr int DUP = 16 / B;          // lanes that end with the same vector
    constexpr int RPI = kCondThreads / 16;
    const int lane = threadIdx.x & 63;
    const int l = lane & 15;
    const int b = l / DUP;
    // consecutive rows per workgroup, the same at every index
    const int G = gridDim.x;
    const int blk = blockIdx.x;
    const int lb = (blk & 7) * (G >> 3) + (blk >> 3);
    const int iters = (n + RPI - 1) / RPI;
    const int it0 = (int)((int64_t)iters * lb / G), it1 = (int)((int64_t)iters * (lb + 1) / G);
    for (int it = it0; it < it1; ++it) {
        const int row = it * RPI + (int)(threadIdx.x >> 4);
        const bool live = row < n;
        RowExtent e = {0, 0};
        if (live) e = row_extent(rp, row);
        const size_t idx = (size_t)(live ? row : 0) * B + b;
        const double p = HAS_H && beta && live ? prev[idx] : 0.0;
        double ah[B], ad[B];
#pragma unroll
        for (int v = 0; v < B; ++v) ah[v] = ad[v] = 0.0;
        for (int64_t q = e.q0 + kLaneEntries * l; q < e.q1; q += kLaneEntries * 16) {
            // entries past the row's end are loaded with these and not used
            const LaneCols lc = *reinterpret_cast<const LaneCols*>(col + q);
            LaneVals<double> lh, ld;
            if (HAS_H) lh = *reinterpret_cast<const LaneVals<double>*>(hv + q);
            if (HAS_D) ld = *reinterpret_cast<const LaneVals<double>*>(dv + q);
            const int m = (int)min((int64_t)kLaneEntries, e.q1 - q);
            double xv[kLaneEntries][B];
#pragma unroll
            for (int k = 0; k < kLaneEntries; ++k)
                if (k < m) ld_vecs<double, B>(xv[k], x + (size_t)lc.c[k] * B);
#pragma unroll
            for (int k = 0; k < kLaneEntries; ++k)
                if (k < m) {
#pragma unroll
                    for (int v = 0; v < B; ++v) {
                        if (HAS_H) ah[v] = fma(lh.h[k], xv[k][v], ah[v]);
                        if (HAS_D) ad[v] = fma(ld.h[k], xv[k][v], ad[v]);
                    }
                }
        }
        const bool writer = live && l % DUP == 0;
        if (HAS_H) {
            const double y = alpha * fold_row<16>(ah, lane) - p;
            if (writer) {
                out[idx] = y;
                if (hset) hset[((size_t)b * M + j) * n + row] = y;
            }
        }
        if (HAS_D) {
            const double y = fold_row<16>(ad, lane);
            if (writer) dset[((size_t)b * M + j) * n + row] = y;
        }
    }
}

// Both recursions of a block of B <= 4 targets at once: x = [n][2B] holds beta_{j-1}
// and then a_{j-1} of every target, H x gives both next vectors, dxH x the D_{j-1} of
// the alpha half; the new betas go straight into their set (vector j), D into its own
// (vector j - 1).  Each matrix entry and each row's latencies serve both recursions:
// microseconds per index on 95 k rows with 4 targets, H on the betas and both products
// on the alphas one after the other 16.2 + 18.2, together 27.9.  The line lies at four
// targets: apart and together 25.3 and 14.9 with one, 27.0 and 18.6 with two, 52.9 and
// 58.9 with eight, where 16 gathered values a row no longer leave several rounds in
// flight (23.6 k rows: 11.1 and 5.8, 13.9 and 9.7 with four, 18.7 and 21.8 with eight).
template <int B>
__global__ __launch_bounds__(kCondThreads) void pair_step_kernel(const int64_t* __restrict__ rp,
                                                                 const int32_t* __restrict__ col,
                                                                 const double* __restrict__ hv,
                                                                 const double* __restrict__ dv,
                                                                 const double* __restrict__ x, const double* prev,
                                                                 double* out, double alpha, int beta, int n, int j, int M,
                                                                 double* __restrict__ hset, double* __restrict__ dset)
{
    constexpr int V = 2 * B;
    constexpr int RPI = kCondThreads / 16;
    const int lane = threadIdx.x & 63;
    const int l = lane & 15;
    const int v = l / (16 / V), b = l / (16 / B);
    // consecutive rows per workgroup, the same at every index
    const int G = gridDim.x;
    const int blk = blockIdx.x;
    const int lb = (blk & 7) * (G >> 3) + (blk >> 3);
    const int iters = (n + RPI - 1) / RPI;
    const int it0 = (int)((int64_t)iters * lb / G), it1 = (int)((int64_t)iters * (lb + 1) / G);
    for (int it = it0; it < it1; ++it) {
        const int row = it * RPI + (int)(threadIdx.x >> 4);
        const bool live = row < n;
        RowExtent e = {0, 0};
        if (live) e = row_extent(rp, row);
        const size_t idx = (size_t)(live ? row : 0) * V + v;
        const double p = beta && live ? prev[idx] : 0.0;
        double ah[V], ad[B];
#pragma unroll
        for (int u = 0; u < V; ++u) ah[u] = 0.0;
#pragma unroll
        for (int u = 0; u < B; ++u) ad[u] = 0.0;
        for (int64_t q = e.q0 + kLaneEntries * l; q < e.q1; q += kLaneEntries * 16) {
            // entries past the row's end are loaded with these and not used
            const LaneCols lc = *reinterpret_cast<const LaneCols*>(col + q);
            const LaneVals<double> lh = *reinterpret_cast<const LaneVals<double>*>(hv + q);
            const LaneVals<double> ld = *reinterpret_cast<const LaneVals<double>*>(dv + q);
            const int m = (int)min((int64_t)kLaneEntries, e.q1 - q);
            double xv[kLaneEntries][V];
#pragma unroll
            for (int k = 0; k < kLaneEntries; ++k)
                if (k < m) ld_vecs<double, V>(xv[k], x + (size_t)lc.c[k] * V);
#pragma unroll
            for (int k = 0; k < kLaneEntries; ++k)
                if (k < m) {
#pragma unroll
                    for (int u = 0; u < V; ++u) ah[u] = fma(lh.h[k], xv[k][u], ah[u]);
#pragma unroll
                    for (int u = 0; u < B; ++u) ad[u] = fma(ld.h[k], xv[k][B + u], ad[u]);
                }
        }
        const double y = alpha * fold_row<16>(ah, lane) - p;
        const double d = fold_row<16>(ad, lane);
        if (live && l % (16 / V) == 0) {
            out[idx] = y;
            if (v < B) hset[((size_t)v * M + j) * n + row] = y;
        }
        if (live && l % (16 / B) == 0) dset[((size_t)b * M + j - 1) * n + row] = d;
    }
}

// x = [n][2B] and the betas' set at index 0: beta_0 = e_t, a_0 as given ([n][B])
__global__ __launch_bounds__(kCondThreads) void pair_start_kernel(const int32_t* __restrict__ targets,
                                                                  const double* __restrict__ a0, int n, int B, int M,
                                                                  double* __restrict__ x, double* __restrict__ hset)
{
    const size_t total = (size_t)n * B;
    for (size_t t = blockIdx.x * (size_t)kCondThreads + threadIdx.x; t < total; t += (size_t)gridDim.x * kCondThreads) {
        const size_t i = t / B;
        const int b = (int)(t % B);
        const double e = (size_t)targets[b] == i ? 1.0 : 0.0;
        x[i * 2 * B + b] = e;
        x[i * 2 * B + B + b] = a0[t];
        hset[(size_t)b * M * n + i] = e;
    }
}

// the alpha half of x = [n][2B] as a block of its own
__global__ __launch_bounds__(kCondThreads) void pair_alpha_kernel(const double* __restrict__ x, int n, int B,
                                                                  double* __restrict__ a)
{
    const size_t total = (size_t)n * B;
    for (size_t t = blockIdx.x * (size_t)kCondThreads + threadIdx.x; t < total; t += (size_t)gridDim.x * kCondThreads)
        a[t] = x[t / B * 2 * B + B + t % B];
}

// 16 rows per workgroup and iteration, at most four workgroups a CU; with 16 vectors two, as many as
// their registers leave room for at a time (23.6 k rows, both recursions: 43.4 us an index with four,
// 34.7 with two, 39.6 with a thread per row and vector; 94.7 k rows 117, 114 and 123).
dim3 lanes_grid(int n, int B)
{
    constexpr int rpi = kCondThreads / 16;
    return dim3((unsigned)std::min(B < 16 ? 1024 : 512, std::max(8, ((n + rpi - 1) / rpi + 7) / 8 * 8)));
}

template <int B>
hipError_t launch_dual_lanes(const int64_t* rp, const int32_t* col, const double* hv, const double* dv, const double* x,
                             const double* prev, double* out, double alpha, int beta, int n, int j, int M, double* hset,
                             double* dset, hipStream_t s)
{
    const dim3 g = lanes_grid(n, B);
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, g, dim3(kCondThreads), 0, s, rp, col, hv, dv, x, prev, out, alpha, beta, n, j, M, hset,
                           dset);
        return hipGetLastError();
    };
    // both products of up to kCondPair vectors are pair_step_kernel's
    if constexpr (B > kCondPair)
        if (hv && dv) return launch(dual_step_lanes_kernel<true, true, B>);
    if (hv && !dv) return launch(dual_step_lanes_kernel<true, false, B>);
    if (!hv && dv) return launch(dual_step_lanes_kernel<false, true, B>);
    return hipErrorInvalidValue;
}

dim3 grid_for(size_t work) { return dim3((unsigned)std::min<size_t>(4096, (work + kCondThreads - 1) / kCondThreads)); }

}  // namespace

hipError_t launch_cond_scatter(const double* blk, int n, int B, int m, int M, double* set, hipStream_t s)
{
    hipLaunchKernelGGL(scatter_kernel, grid_for((size_t)n * B), dim3(kCondThreads), 0, s, blk, n, B, m, M, set);
    return hipGetLastError();
}

hipError_t launch_cond_chunk_sum(const double* part, int S, size_t mm, int B, double* C, hipStream_t s)
{
    hipLaunchKernelGGL(chunk_sum_kernel, grid_for((size_t)B * mm), dim3(kCondThreads), 0, s, part, S, mm, B, C);
    return hipGetLastError();
}

hipError_t launch_cond_dual_step(const int64_t* rp, const int32_t* col, const double* hv, const double* dv,
                                 const double* x, const double* prev, double* out, double alpha, int beta, int n, int B,
                                 int j, int M, double* hset, double* dset, hipStream_t s)
{
    switch (B) {
    case 1: return launch_dual_lanes<1>(rp, col, hv, dv, x, prev, out, alpha, beta, n, j, M, hset, dset, s);
    case 2: return launch_dual_lanes<2>(rp, col, hv, dv, x, prev, out, alpha, beta, n, j, M, hset, dset, s);
    case 4: return launch_dual_lanes<4>(rp, col, hv, dv, x, prev, out, alpha, beta, n, j, M, hset, dset, s);
    case 8: return launch_dual_lanes<8>(rp, col, hv, dv, x, prev, out, alpha, beta, n, j, M, hset, dset, s);
    case 16: return launch_dual_lanes<16>(rp, col, hv, dv, x, prev, out, alpha, beta, n, j, M, hset, dset, s);
    default: break;
    }
    const size_t work = (size_t)n * B;
    const dim3 g((unsigned)std::min<size_t>(8192, (work + kCondThreads - 1) / kCondThreads));
    if (hv && dv)
        hipLaunchKernelGGL((dual_step_kernel<true, true>), g, dim3(kCondThreads), 0, s, rp, col, hv, dv, x, prev, out,
                           alpha, beta, n, B, j, M, hset, dset);
    else if (hv)
        hipLaunchKernelGGL((dual_step_kernel<true, false>), g, dim3(kCondThreads), 0, s, rp, col, hv, dv, x, prev, out,
                           alpha, beta, n, B, j, M, hset, dset);
    else if (dv)
        hipLaunchKernelGGL((dual_step_kernel<false, true>), g, dim3(kCondThreads), 0, s, rp, col, hv, dv, x, prev, out,
                           alpha, beta, n, B, j, M, hset, dset);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_cond_pair_step(const int64_t* rp, const int32_t* col, const double* hv, const double* dv,
                                 const double* x, const double* prev, double* out, double alpha, int beta, int n, int B,
                                 int j, int M, double* hset, double* dset, hipStream_t s)
{
    const auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, lanes_grid(n, B), dim3(kCondThreads), 0, s, rp, col, hv, dv, x, prev, out, alpha, beta, n,
                           j, M, hset, dset);
        return hipGetLastError();
    };
    if (j < 1) return hipErrorInvalidValue;
    switch (B) {
    case 1: return launch(pair_step_kernel<1>);
    case 2: return launch(pair_step_kernel<2>);
    case 4: return launch(pair_step_kernel<4>);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_cond_pair_start(const int32_t* targets, const double* a0, int n, int B, int M, double* x, double* hset,
                                  hipStream_t s)
{
    hipLaunchKernelGGL(pair_start_kernel, grid_for((size_t)n * B), dim3(kCondThreads), 0, s, targets, a0, n, B, M, x, hset);
    return hipGetLastError();
}

hipError_t launch_cond_pair_alpha(const double* x, int n, int B, double* a, hipStream_t s)
{
    hipLaunchKernelGGL(pair_alpha_kernel, grid_for((size_t)n * B), dim3(kCondThreads), 0, s, x, n, B, a);
    return hipGetLastError();
}

hipError_t launch_cond_weight(const double* C, int M, int T, double* X, hipStream_t s)
{
    hipLaunchKernelGGL(cond_weight_kernel, grid_for((size_t)T * M * M), dim3(kCondThreads), 0, s, C, M, T, X);
    return hipGetLastError();
}

hipError_t launch_dct3_matrix(int M, double* P, hipStream_t s)
{
    hipLaunchKernelGGL(dct3_matrix_kernel, grid_for((size_t)M * M), dim3(kCondThreads), 0, s, M, P);
    return hipGetLastError();
}

}  // namespace leo2d
