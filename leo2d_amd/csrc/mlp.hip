// mlp.hip -- BF16 MFMA kernels of the learned local-moment surrogate.
//
// The surrogate is a small multilayer perceptron (64 Fourier features of a
// local stacking configuration -> hidden GELU layers -> local Chebyshev
// moments).  Weights and activations are bfloat16, every product accumulates
// in FP32 on the matrix cores (v_mfma_f32_16x16x32_bf16), and the optimiser
// keeps FP32 master weights.  There is no counterpart in the reference; the
// moments it learns come from the KPM recursion of this library.
//
// Both operands of every product have k contiguous in memory, so a lane's eight k of
// an MFMA operand are one 16-byte load: X W^T reads X and W, the input gradient dZ W
// reads a transposed copy of W, the weight gradient dZ^T X transposed copies of dZ
// and X, which the kernels that make these operands write beside them.
//
// What bounds it: the products are small (a training batch of 512 on 256-wide
// layers), so a launch is a chain of load latencies.  Small products take 32 x 32
// tiles, a 16 x 16 block per wavefront with sixteen loads straight into registers in
// flight: 128 to 512 workgroups where 64 x 64 tiles gave 32, and no barrier per k
// step.  Large products (inference) stage 64 x 64 or 128 x 128 tiles through LDS:
// read straight from memory, an operand row's 64 bytes per k step come at the 16
// bytes a clock of a scattered load.  Every output is one chain of k steps of 32 in
// order in all of them, so the tile does not change a bit of the result.  (k shared
// by the four wavefronts of a workgroup was as fast and changes the rounding.)
// The two products of a layer's backward pass (its weight gradient and the input
// gradient below) go out in one launch, bias gradients and the loss with them: a
// training step on 512 rows of 72 -> 3 x 256 -> 1024 is 10 launches and about 75 us
// on the GPU (19 and 177 us with 64 x 64 tiles, operands transposed through LDS two
// bytes at a time and a kernel each for the loss and the column sums).
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <algorithm>

#include "mlp.h"

namespace leo2d {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef short bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));

constexpr int kT = 256;

__device__ inline uint16_t f2bf(float f)
{
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0;   // NaN stays NaN
    u += 0x7fffu + ((u >> 16) & 1u);                       // round to nearest even
    return (uint16_t)(u >> 16);
}
__device__ inline float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

// GELU, tanh form: 0.5 z (1 + tanh(c (z + 0.044715 z^3))), c = sqrt(2/pi)
__device__ inline float gelu(float z)
{
    const float c = 0.7978845608028654f;
    return 0.5f * z * (1.0f + tanhf(c * (z + 0.044715f * z * z * z)));
}
__device__ inline float gelu_grad(float z)
{
    const float c = 0.7978845608028654f;
    const float u = c * (z + 0.044715f * z * z * z);
    const float t = tanhf(u);
    return 0.5f * (1.0f + t) + 0.5f * z * (1.0f - t * t) * c * (1.0f + 3.0f * 0.044715f * z * z);
}

// eight k of an operand row from k on, zero past K
__device__ inline bf16x8 ld_frag(const uint16_t* row, int k, int K)
{
    bf16x8 v = {0, 0, 0, 0, 0, 0, 0, 0};
    if (k < K) {
        v = *reinterpret_cast<const bf16x8*>(row + k);
        if (k + 8 > K) {
#pragma unroll
            for (int t = 0; t < 8; ++t)
                if (k + t >= K) v[t] = 0;
        }
    }
    return v;
}

struct GemmBatch {
    GemmArgs g[2];
    int tiles[2];       // workgroups of each product
    SumArgs sums;
    int sum_blocks;
    LossArgs loss;
};

// the epilogue EPI of four rows of one column (rows row .. row + 3, those below M)
template <int EPI>
__device__ inline void gemm_store(const GemmArgs& g, const floatx4& v, int row, int col, int lane)
{
    const bool in = col < g.N;
    const int rows = in ? min(4, g.M - row) : 0;
    const float bias = in && (EPI == EPI_BIAS_F32 || EPI == EPI_BIAS_GELU || EPI == EPI_MSE) ? g.bias[col] : 0.f;
    uint16_t h[4] = {0, 0, 0, 0};
    double sq[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        if (t < rows) {
            const int64_t o = (int64_t)(row + t) * g.ldc + col;
            if (EPI == EPI_STORE_F32) {
                g.C32[o] = v[t];
            } else if (EPI == EPI_BIAS_F32) {
                g.C32[o] = v[t] + bias;
            } else if (EPI == EPI_BIAS_GELU) {
                const float z = v[t] + bias;
                if (g.Z) g.Z[o] = z;
                h[t] = f2bf(gelu(z));
            } else if (EPI == EPI_GELU_BWD) {
                h[t] = f2bf(v[t] * gelu_grad(g.Z[o]));
            } else {
                const float d = (v[t] + bias) - g.T[o];
                h[t] = f2bf(g.scale * d);
                sq[t] = (double)d * (double)d;
            }
            if (EPI != EPI_STORE_F32 && EPI != EPI_BIAS_F32) g.C16[(int64_t)(row + t) * g.ld16 + col] = h[t];
        }
    }
    if (EPI == EPI_STORE_F32 || EPI == EPI_BIAS_F32) return;
    if (g.C16T && rows > 0) {
        uint16_t* p = g.C16T + (int64_t)col * g.ld16t + row;   // row is a multiple of 4, ld16t of 8
        if (rows == 4) {
            *reinterpret_cast<u16x4*>(p) = u16x4{h[0], h[1], h[2], h[3]};
        } else {
#pragma unroll
            for (int t = 0; t < 4; ++t)
                if (t < rows) p[t] = h[t];
        }
    }
    if (EPI == EPI_MSE) {
        // the 16 columns of this block (their lanes hold the same four rows)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
#pragma unroll
            for (int off = 8; off > 0; off >>= 1) sq[t] += __shfl_xor(sq[t], off);
            if ((lane & 15) == 0 && row + t < g.M && col < g.N)
                g.loss[(int64_t)(row + t) * ((g.N + 15) / 16) + col / 16] = sq[t];
        }
    }
}
// the same, the epilogue known at run time only
__device__ inline void gemm_store(const GemmArgs& g, const floatx4& v, int row, int col, int lane)
{
    switch (g.epi) {
    case EPI_STORE_F32: gemm_store<EPI_STORE_F32>(g, v, row, col, lane); break;
    case EPI_BIAS_F32: gemm_store<EPI_BIAS_F32>(g, v, row, col, lane); break;
    case EPI_BIAS_GELU: gemm_store<EPI_BIAS_GELU>(g, v, row, col, lane); break;
    case EPI_GELU_BWD: gemm_store<EPI_GELU_BWD>(g, v, row, col, lane); break;
    default: gemm_store<EPI_MSE>(g, v, row, col, lane); break;
    }
}

// out[c] = sum_k A[c][k].  A workgroup owns kSumRows rows of A (outputs c); kSumGroups
// threads each add a contiguous slice of k in order, and the slices are added in order.
constexpr int kSumRows = 16;
constexpr int kSumGroups = kT / kSumRows;
__device__ inline void row_sums(const SumArgs& a, int block, float (*part)[kSumRows])
{
    const int cx = threadIdx.x / kSumGroups, g = threadIdx.x % kSumGroups;
    const int c = block * kSumRows + cx;
    const int per = (a.K + kSumGroups - 1) / kSumGroups;
    const int k0 = min(a.K, g * per), k1 = min(a.K, k0 + per);
    float s = 0.f;
    if (c < a.rows) {
        const uint16_t* p = a.A + (int64_t)c * a.lda;
        int k = k0;
        for (; k + 8 <= k1; k += 8) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = bf2f(p[k + u]);
#pragma unroll
            for (int u = 0; u < 8; ++u) s += v[u];
        }
        for (; k < k1; ++k) s += bf2f(p[k]);
    }
    part[g][cx] = s;
    __syncthreads();
    if (g == 0 && c < a.rows) {
        float t = part[0][cx];
        for (int q = 1; q < kSumGroups; ++q) t += part[q][cx];
        a.out[c] = t;
    }
}

// the product and tile of a workgroup of a batch; false for the workgroups of the sums
__device__ inline bool gemm_tile(const GemmBatch& p, int tile, bool& second, int& m0, int& n0)
{
    __shared__ float part[kSumGroups][kSumRows];
    int t = blockIdx.x;
    const int products = p.tiles[0] + p.tiles[1];
    if (t >= products + p.sum_blocks) {
        const int r = (t - products - p.sum_blocks) * kT + threadIdx.x;
        if (r < p.loss.rows) {
            const double* q = p.loss.part + (int64_t)r * p.loss.parts;
            double s = 0.0;
            for (int c = 0; c < p.loss.parts; ++c) s += q[c];
            p.loss.row_loss[r] = s;
        }
        return false;
    }
    if (t >= products) {
        row_sums(p.sums, t - products, part);
        return false;
    }
    second = t >= p.tiles[0];
    if (second) t -= p.tiles[0];
    const int tiles_n = (p.g[second].N + tile - 1) / tile;
    m0 = t / tiles_n * tile;
    n0 = t % tiles_n * tile;
    return true;
}

// a 32 x 32 tile, a 16 x 16 block per wavefront, operands straight into registers: the
// next U k steps load while the current U are multiplied
__global__ __launch_bounds__(kT) void mlp_gemm_small_kernel(GemmBatch p)
{
    constexpr int U = 4;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    bool second;
    int m0, n0;
    if (!gemm_tile(p, 32, second, m0, n0)) return;
    const GemmArgs& g = second ? p.g[1] : p.g[0];
    const int r = lane & 15, kg = lane >> 4;
    m0 += (wave >> 1) * 16;
    n0 += (wave & 1) * 16;
    const uint16_t* a = g.A + (int64_t)min(m0 + r, g.M - 1) * g.lda;
    const uint16_t* b = g.B + (int64_t)min(n0 + r, g.N - 1) * g.ldb;
    const int K = g.K;
    bf16x8 fa[2][U], fb[2][U];
    auto load = [&](bf16x8 (&va)[U], bf16x8 (&vb)[U], int k) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            va[u] = ld_frag(a, k + 32 * u + 8 * kg, K);
            vb[u] = ld_frag(b, k + 32 * u + 8 * kg, K);
        }
    };
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
    auto mul = [&](const bf16x8 (&va)[U], const bf16x8 (&vb)[U]) {
        // steps past K multiply zeros
#pragma unroll
        for (int u = 0; u < U; ++u) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va[u], vb[u], acc, 0, 0, 0);
    };
    load(fa[0], fb[0], 0);
    for (int k = 0; k < K; k += 64 * U) {
        load(fa[1], fb[1], k + 32 * U);
        mul(fa[0], fb[0]);
        load(fa[0], fb[0], k + 64 * U);
        mul(fa[1], fb[1]);
    }
    // a lane holds C[row0 + t][col], t = 0..3
    gemm_store(g, acc, m0 + 4 * kg, n0 + r, lane);
}

// TILE x TILE outputs through LDS, a (TILE / 2)^2 quarter per wavefront; k in steps of
// 64, the next step's rows in registers during the products of this one
template <int TILE, int EPI>
__global__ __launch_bounds__(kT) void mlp_gemm_tile_kernel(GemmBatch p)
{
    constexpr int BK = 64, LD = BK + 8;        // padded rows: 16 lanes of a read start in 16 different banks
    constexpr int NB = TILE / 32;              // 16 x 16 blocks per side of a wavefront's quarter
    constexpr int NL = TILE * BK / (8 * kT);   // 16-byte runs per thread and operand
    __shared__ __align__(16) uint16_t As[TILE * LD], Bs[TILE * LD];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    bool second;
    int m0, n0;
    if (!gemm_tile(p, TILE, second, m0, n0)) return;
    const GemmArgs& g = p.g[0];
    const int r = lane & 15, kg = lane >> 4;
    const int wm = (wave >> 1) * (TILE / 2), wn = (wave & 1) * (TILE / 2);
    const int K = g.K;
    bf16x8 ra[NL], rb[NL];
    auto load = [&](int k) {
#pragma unroll
        for (int q = 0; q < NL; ++q) {
            const int row = (q * kT + tid) / 8, kk = k + (tid & 7) * 8;
            ra[q] = ld_frag(g.A + (int64_t)min(m0 + row, g.M - 1) * g.lda, kk, K);
            rb[q] = ld_frag(g.B + (int64_t)min(n0 + row, g.N - 1) * g.ldb, kk, K);
        }
    };
    floatx4 acc[NB][NB];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    load(0);
    for (int k = 0; k < K; k += BK) {
        __syncthreads();
#pragma unroll
        for (int q = 0; q < NL; ++q) {
            const int at = (q * kT + tid) / 8 * LD + (tid & 7) * 8;
            *reinterpret_cast<bf16x8*>(&As[at]) = ra[q];
            *reinterpret_cast<bf16x8*>(&Bs[at]) = rb[q];
        }
        __syncthreads();
        if (k + BK < K) load(k + BK);
#pragma unroll
        for (int ks = 0; ks < BK; ks += 32) {
            bf16x8 fa[NB], fb[NB];
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                fa[i] = *reinterpret_cast<const bf16x8*>(&As[(wm + 16 * i + r) * LD + ks + 8 * kg]);
                fb[i] = *reinterpret_cast<const bf16x8*>(&Bs[(wn + 16 * i + r) * LD + ks + 8 * kg]);
            }
#pragma unroll
            for (int i = 0; i < NB; ++i)
#pragma unroll
                for (int j = 0; j < NB; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
        }
    }
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) gemm_store<EPI>(g, acc[i][j], m0 + wm + 16 * i + 4 * kg, n0 + wn + 16 * j + r, lane);
}

// rows of X (FP32; row b is idx[b], or b without idx) -> bf16 batch and its transpose; rows of T -> FP32 batch
__global__ __launch_bounds__(kT) void gather_kernel(const float* X, int in, const float* T, int out, const int64_t* idx,
                                                    int rows, uint16_t* Xb, int64_t ldx, uint16_t* XbT, int64_t ldxt,
                                                    float* Tb, int* ctr)
{
    const int b = blockIdx.x;
    if (b >= rows) return;
    if (ctr && b == 0 && threadIdx.x == 0) *ctr += 1;
    const int64_t src = idx ? idx[b] : b;
    for (int c = threadIdx.x; c < in; c += kT) {
        const uint16_t h = f2bf(X[src * in + c]);
        Xb[(int64_t)b * ldx + c] = h;
        if (XbT) XbT[(int64_t)c * ldxt + b] = h;
    }
    if (T)
        for (int c = threadIdx.x; c < out; c += kT) Tb[(int64_t)b * out + c] = T[src * out + c];
}

// Adam with bias correction on one parameter, and its bf16 rounding
__device__ inline uint16_t param_step(const ParamArgs& a, float c1, float c2, int64_t i)
{
    float pn = a.p[i];
    if (a.grad) {
        const float gr = a.grad[i];
        const float mi = a.b1 * a.m[i] + (1.f - a.b1) * gr;
        const float vi = a.b2 * a.v[i] + (1.f - a.b2) * gr * gr;
        a.m[i] = mi;
        a.v[i] = vi;
        const float upd = a.lr * (mi / c1) / (sqrtf(vi / c2) + a.eps);
        pn = pn - upd;
        a.p[i] = pn;
    }
    return f2bf(pn);
}

// A workgroup owns a 32 x 32 block of one layer's W (or 256 biases): the update runs
// along the rows of W, the transposed copy leaves through LDS.
__global__ __launch_bounds__(kT) void params_kernel(ParamArgs a)
{
    __shared__ uint16_t tile[kParamTile][kParamTile + 1];
    int l = 0;
    while (l + 1 < a.nlayers && a.layers[l + 1].tile0 <= (int)blockIdx.x) ++l;
    const LayerDesc d = a.layers[l];
    const int t = blockIdx.x - d.tile0;
    float c1 = a.c1, c2 = a.c2;
    if (a.corr) {
        const int64_t k = *a.ctr;
        c1 = a.corr[2 * k];
        c2 = a.corr[2 * k + 1];
    }
    const int tiles_i = (d.din + kParamTile - 1) / kParamTile, tiles_o = (d.dout + kParamTile - 1) / kParamTile;
    if (t >= tiles_i * tiles_o) {
        const int o = (t - tiles_i * tiles_o) * kT + threadIdx.x;
        if (o < d.dout) (void)param_step(a, c1, c2, d.boff + o);
        return;
    }
    const int i0 = t % tiles_i * kParamTile, o0 = t / tiles_i * kParamTile;
    const int x = threadIdx.x % kParamTile, y = threadIdx.x / kParamTile;
    constexpr int RY = kT / kParamTile;
    for (int q = y; q < kParamTile; q += RY) {
        const int o = o0 + q, i = i0 + x;
        if (o < d.dout && i < d.din) {
            const uint16_t h = param_step(a, c1, c2, d.woff + (int64_t)o * d.din + i);
            a.p16[d.w16 + (int64_t)o * d.ldw + i] = h;
            tile[q][x] = h;
        }
    }
    __syncthreads();
    for (int q = y; q < kParamTile; q += RY) {
        const int i = i0 + q, o = o0 + x;
        if (o < d.dout && i < d.din) a.pt16[d.wt16 + (int64_t)i * d.ldwt + o] = tile[x][q];
    }
}

// per row: mean over the E ensemble members and, for each of nblk equal blocks
// of the outputs, the root mean square over the block of the ensemble standard
// deviation (block grid: blockIdx.y)
__global__ __launch_bounds__(kT) void ensemble_stats_kernel(const float* Ys, int E, int64_t estride, int rows, int cols,
                                                            int nblk, float* mean, float* spread)
{
    const int r = blockIdx.x, b = blockIdx.y;
    if (r >= rows || b >= nblk) return;
    const int bw = cols / nblk;
    __shared__ float s[kT];
    float acc = 0.f;
    for (int c = b * bw + threadIdx.x; c < (b + 1) * bw; c += kT) {
        const int64_t o = (int64_t)r * cols + c;
        float mu = 0.f;
        for (int e = 0; e < E; ++e) mu += Ys[e * estride + o];
        mu /= (float)E;
        float var = 0.f;
        for (int e = 0; e < E; ++e) {
            const float d = Ys[e * estride + o] - mu;
            var += d * d;
        }
        if (mean) mean[o] = mu;
        acc += var / (float)E;
    }
    s[threadIdx.x] = acc;
    __syncthreads();
    for (int w = kT / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) spread[(int64_t)r * nblk + b] = sqrtf(s[0] / (float)bw);
}

}  // namespace

namespace {

template <int TILE>
void launch_tile(const GemmBatch& p, dim3 grid, hipStream_t s)
{
    switch (p.g[0].epi) {
    case EPI_STORE_F32: hipLaunchKernelGGL((mlp_gemm_tile_kernel<TILE, EPI_STORE_F32>), grid, dim3(kT), 0, s, p); break;
    case EPI_BIAS_F32: hipLaunchKernelGGL((mlp_gemm_tile_kernel<TILE, EPI_BIAS_F32>), grid, dim3(kT), 0, s, p); break;
    case EPI_BIAS_GELU: hipLaunchKernelGGL((mlp_gemm_tile_kernel<TILE, EPI_BIAS_GELU>), grid, dim3(kT), 0, s, p); break;
    case EPI_GELU_BWD: hipLaunchKernelGGL((mlp_gemm_tile_kernel<TILE, EPI_GELU_BWD>), grid, dim3(kT), 0, s, p); break;
    default: hipLaunchKernelGGL((mlp_gemm_tile_kernel<TILE, EPI_MSE>), grid, dim3(kT), 0, s, p); break;
    }
}

}  // namespace

hipError_t launch_gemm_bf16(const GemmArgs& a, const GemmArgs* b, const SumArgs& sums, const LossArgs& loss,
                            hipStream_t s)
{
    auto bad = [](const GemmArgs& g) {
        return g.M <= 0 || g.N <= 0 || g.K <= 0 || g.lda % 8 != 0 || g.ldb % 8 != 0 || g.ld16t % 8 != 0 ||
               ((uintptr_t)g.A | (uintptr_t)g.B) % 16 != 0 || (uintptr_t)g.C16T % 8 != 0;
    };
    if (bad(a) || (b && bad(*b))) return hipErrorInvalidValue;
    auto tiles = [](const GemmArgs& g, int t) { return (int64_t)((g.M + t - 1) / t) * ((g.N + t - 1) / t); };
    // the widest tile that still gives each of the 256 CUs a workgroup
    auto width = [&](const GemmArgs& g) { return tiles(g, 128) >= 256 ? 128 : (tiles(g, 64) >= 256 ? 64 : 32); };
    if (b && (width(a) != 32 || width(*b) != 32)) {
        const hipError_t e = launch_gemm_bf16(a, nullptr, sums, loss, s);
        return e != hipSuccess ? e : launch_gemm_bf16(*b, nullptr, SumArgs{}, LossArgs{}, s);
    }
    const int t = width(a);
    GemmBatch p{};
    p.g[0] = a;
    if (b) p.g[1] = *b;
    p.sums = sums;
    p.sum_blocks = (sums.rows + kSumRows - 1) / kSumRows;
    p.loss = loss;
    const int64_t na = tiles(a, t), nb = b ? tiles(*b, t) : 0;
    const int64_t blocks = na + nb + p.sum_blocks + (loss.rows + kT - 1) / kT;
    if (blocks > 0x7fffff) return hipErrorInvalidValue;   // grid x block below 2^32
    p.tiles[0] = (int)na;
    p.tiles[1] = (int)nb;
    const dim3 grid((unsigned)blocks);
    if (t == 128) launch_tile<128>(p, grid, s);
    else if (t == 64) launch_tile<64>(p, grid, s);
    else hipLaunchKernelGGL(mlp_gemm_small_kernel, grid, dim3(kT), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_gather(const float* X, int in, const float* T, int out, const int64_t* idx, int rows, uint16_t* Xb,
                         int64_t ldx, uint16_t* XbT, int64_t ldxt, float* Tb, int* ctr, hipStream_t s)
{
    hipLaunchKernelGGL(gather_kernel, dim3(rows), dim3(kT), 0, s, X, in, T, out, idx, rows, Xb, ldx, XbT, ldxt, Tb, ctr);
    return hipGetLastError();
}

hipError_t launch_cast_rows(const float* X, int in, int rows, uint16_t* Xb, int64_t ldx, uint16_t* XbT, int64_t ldxt,
                            hipStream_t s)
{
    return launch_gather(X, in, nullptr, 0, nullptr, rows, Xb, ldx, XbT, ldxt, nullptr, nullptr, s);
}

hipError_t launch_params(const ParamArgs& a, hipStream_t s)
{
    hipLaunchKernelGGL(params_kernel, dim3(a.blocks), dim3(kT), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_ensemble_stats(const float* Ys, int E, int64_t estride, int rows, int cols, int nblk, float* mean,
                                 float* spread, hipStream_t s)
{
    if (rows <= 0) return hipSuccess;
    if (nblk <= 0 || cols % nblk != 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(ensemble_stats_kernel, dim3(rows, nblk), dim3(kT), 0, s, Ys, E, estride, rows, cols, nblk, mean,
                       spread);
    return hipGetLastError();
}

void adam_corrections(float b1, float b2, int step, float* c1, float* c2)
{
    *c1 = 1.f - powf(b1, (float)step);
    *c2 = 1.f - powf(b2, (float)step);
}

}  // namespace leo2d
