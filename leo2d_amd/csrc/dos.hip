// dos.hip -- Jackson-kernel DoS reconstruction and the Gershgorin bound.
//
// DoS: Param_tools::densityTransform{,Trace} (param_tools.cpp:661-768) apply
// the Jackson damping g_n, an FFTW REDFT01 (DCT-III)
//     out_k = in_0 + 2 sum_{n>=1} in_n cos(pi n (k+1/2) / M)
// and divide by pi sqrt(a^2 - (E_k - b)^2).  The DCT-III is a direct sum in FP64
// with exactly reduced phases: cos(pi n (2k+1) / 2M) is entry n (2k+1) mod 4M of
// a cosine table, of which the first quarter is stored.
//
// What bounds it: FP64 multiply-adds, M^2 / 2 per moment row.  Columns k and
// M - 1 - k differ only in the sign of the odd terms, so a lane sums even and
// odd n of one k < M / 2 apart and writes both columns.  A cosine is looked up
// once (LDS, a gather) for kRows moment rows, whose weights arrive as scalar
// loads; the n range is cut over the eight wavefronts of a workgroup, added in
// wavefront order, so one row of few moments still fills several SIMDs.
// (One workgroup per row with one look-up and one 64-bit remainder per term
// took 9055 us for 32 rows of 4096 moments, 143 us for one row of 500.)
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.h"

namespace leo2d {
namespace {

constexpr int kThreads = 256;
constexpr int kRows = 8;               // moment rows that share a cosine look-up
constexpr int kDosWaves = 8;           // wavefronts of a workgroup, each a slice of n
constexpr size_t kDosLds = 160 << 10;  // LDS of a CU

// table entry i of the quarter wave in LDS: one double of padding per 16, so the
// lanes' stride 2n through the table does not fall on one bank for n = 8, 16, ...
__device__ inline int dos_slot(int i) { return i + (i >> 4); }

// wt[group][n][kRows] = g_n mu (twice for n >= 1), rows past T zero; quarter-wave
// cosine table ctab[i] = cos(pi i / 2M), i = 0 .. M; energies
__global__ __launch_bounds__(kThreads) void dos_prepare_kernel(const double* mu, int T, int M, double a, double b,
                                                               double* wt, double* ctab, double* E)
{
    const double pi = 3.14159265358979323846;
    const size_t total = (size_t)((T + kRows - 1) / kRows) * M * kRows;
    for (size_t t = blockIdx.x * (size_t)kThreads + threadIdx.x; t < total || t <= (size_t)M;
         t += (size_t)gridDim.x * kThreads) {
        if (t <= (size_t)M) ctab[t] = cos(pi * (double)t / (2.0 * M));
        if (t < (size_t)M) E[t] = b + a * cos((t * 1.0 + 0.5) * pi / M);
        if (t < total) {
            const int i = (int)(t / kRows % M);
            const size_t row = t / kRows / M * kRows + t % kRows;
            double w = 0.0;
            if (row < (size_t)T) {
                // Jackson coefficients (param_tools.cpp:670-671)
                const double g = ((M - i) * cos((pi * i) / M) + sin((pi * i) / M) / tan(pi / M)) / (M);
                w = g * mu[row * M + i];
                if (i > 0) w = 2.0 * w;
            }
            wt[t] = w;
        }
    }
}

// LDS: the quarter-wave table is copied into LDS (else read from global memory)
template <bool LDS>
__global__ __launch_bounds__(64 * kDosWaves) void dos_kernel(const double* __restrict__ wt,
                                                             const double* __restrict__ ctab,
                                                             const double* __restrict__ E, int T, int M, double a,
                                                             double b, double scale, double* __restrict__ rho)
{
    extern __shared__ double lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int half = (M + 1) / 2;
    const int kblocks = (half + 63) / 64;
    const int group = blockIdx.x / kblocks;
    const int k = blockIdx.x % kblocks * 64 + lane;
    const int P = 4 * M, H = 2 * M;
    if (LDS) {
        for (int i = threadIdx.x; i <= M; i += 64 * kDosWaves) lds[dos_slot(i)] = ctab[i];
        __syncthreads();
    }
    // this wavefront's n, an even start so that the parities alternate from even
    const int per = (M + 2 * kDosWaves - 1) / (2 * kDosWaves) * 2;
    const int n0 = wave * per, n1 = n0 + per < M ? n0 + per : M;
    const int step = 2 * (k < half ? k : half - 1) + 1;
    int m = (int)((long long)n0 * step % P);
    auto look = [&]() {
        int i = m <= H ? m : P - m;                 // cos(2 pi - x) = cos x
        const bool neg = i > M;                     // cos(pi - x) = -cos x
        i = neg ? H - i : i;
        m += step;
        m -= m >= P ? P : 0;
        const double c = LDS ? lds[dos_slot(i)] : ctab[i];
        return neg ? -c : c;
    };
    const double* w = wt + (size_t)group * M * kRows;
    double ev[kRows], od[kRows];
#pragma unroll
    for (int r = 0; r < kRows; ++r) ev[r] = od[r] = 0.0;
    int n = n0;
#pragma unroll 2
    for (; n + 1 < n1; n += 2) {
        const double c0 = look(), c1 = look();
        const double* wn = w + (size_t)n * kRows;
#pragma unroll
        for (int r = 0; r < kRows; ++r) ev[r] = fma(wn[r], c0, ev[r]);
#pragma unroll
        for (int r = 0; r < kRows; ++r) od[r] = fma(wn[kRows + r], c1, od[r]);
    }
    if (n < n1) {
        const double c0 = look();
        const double* wn = w + (size_t)n * kRows;
#pragma unroll
        for (int r = 0; r < kRows; ++r) ev[r] = fma(wn[r], c0, ev[r]);
    }
    if (LDS) __syncthreads();   // the table's space takes the partial sums
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        lds[(wave * 2 * kRows + r) * 64 + lane] = ev[r];
        lds[(wave * 2 * kRows + kRows + r) * 64 + lane] = od[r];
    }
    __syncthreads();
    static_assert(kRows == kDosWaves, "one row per wavefront in the fold");
    const int row = group * kRows + wave;
    if (row >= T || k >= half) return;
    double e = 0.0, o = 0.0;
#pragma unroll
    for (int q = 0; q < kDosWaves; ++q) {
        e += lds[(q * 2 * kRows + wave) * 64 + lane];
        o += lds[(q * 2 * kRows + kRows + wave) * 64 + lane];
    }
    const double pi = 3.14159265358979323846;
    auto density = [&](double s, int c) {
        const double x = E[c] - b;
        rho[(size_t)row * M + c] = scale * s / (pi * sqrt(a * a - x * x));
    };
    density(e + o, k);
    if (M - 1 - k != k) density(e - o, M - 1 - k);
}

__global__ __launch_bounds__(kThreads) void gershgorin_kernel(const int64_t* rp, const int32_t* col, const void* val,
                                                              int is_complex, int n, double* lohi)
{
    __shared__ double slo[kThreads], shi[kThreads];
    double lo = 1e300, hi = -1e300;
    for (int i = blockIdx.x * kThreads + threadIdx.x; i < n; i += gridDim.x * kThreads) {
        double d = 0.0, rsum = 0.0;
        for (int64_t q = rp[i]; q < rp[i + 1]; ++q) {
            double re_v, mag;
            if (is_complex) {
                const double2 h = static_cast<const double2*>(val)[q];
                re_v = h.x;
                mag = sqrt(h.x * h.x + h.y * h.y);
            } else {
                re_v = static_cast<const double*>(val)[q];
                mag = fabs(re_v);
            }
            if (col[q] == i) d += re_v;
            else rsum += mag;
        }
        lo = fmin(lo, d - rsum);
        hi = fmax(hi, d + rsum);
    }
    slo[threadIdx.x] = lo;
    shi[threadIdx.x] = hi;
    __syncthreads();
    for (int w = kThreads / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) {
            slo[threadIdx.x] = fmin(slo[threadIdx.x], slo[threadIdx.x + w]);
            shi[threadIdx.x] = fmax(shi[threadIdx.x], shi[threadIdx.x + w]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        lohi[2 * blockIdx.x] = slo[0];
        lohi[2 * blockIdx.x + 1] = shi[0];
    }
}

}  // namespace

size_t dos_workspace(int T, int M)
{
    return sizeof(double) * ((size_t)((T + kRows - 1) / kRows) * kRows * M + (size_t)M + 1);
}

hipError_t launch_dos(const double* mu, int T, int M, double a, double b, double scale, double* E, double* rho,
                      double* work, hipStream_t s)
{
    if (M > (1 << 28)) return hipErrorInvalidValue;   // 4M + 2M in 32-bit phase arithmetic
    const int groups = (T + kRows - 1) / kRows;
    double* wt = work;
    double* ctab = work + (size_t)groups * kRows * M;
    const size_t items = std::max((size_t)groups * kRows * M, (size_t)M + 1);
    hipLaunchKernelGGL(dos_prepare_kernel, dim3((unsigned)std::min<size_t>(2048, (items + kThreads - 1) / kThreads)),
                       dim3(kThreads), 0, s, mu, T, M, a, b, wt, ctab, E);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const dim3 grid((unsigned)(((M + 1) / 2 + 63) / 64) * (unsigned)groups);
    const size_t fold = sizeof(double) * 64 * 2 * kRows * kDosWaves;
    const size_t table = sizeof(double) * ((size_t)M + 1 + M / 16 + 1);
    // the table in LDS while it fits (M <= 19,000); longer rows read it through the caches
    const size_t shmem = table <= kDosLds ? std::max(fold, table) : fold;
    const bool in_lds = table <= kDosLds;
    const void* f = in_lds ? (const void*)dos_kernel<true> : (const void*)dos_kernel<false>;
    if (shmem > (64u << 10)) {
        e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);
        if (e != hipSuccess) return e;
    }
    if (in_lds)
        hipLaunchKernelGGL(dos_kernel<true>, grid, dim3(64 * kDosWaves), shmem, s, wt, ctab, E, T, M, a, b, scale, rho);
    else
        hipLaunchKernelGGL(dos_kernel<false>, grid, dim3(64 * kDosWaves), shmem, s, wt, ctab, E, T, M, a, b, scale, rho);
    return hipGetLastError();
}

hipError_t launch_gershgorin(const int64_t* rp, const int32_t* col, const void* val, int is_complex, int n,
                             double* lohi, int blocks, hipStream_t s)
{
    hipLaunchKernelGGL(gershgorin_kernel, dim3(blocks), dim3(kThreads), 0, s, rp, col, val, is_complex, n, lohi);
    return hipGetLastError();
}

}  // namespace leo2d
