// mlp.h -- launchers of the surrogate's BF16 MFMA kernels (mlp.hip).
// Internal to libleo2d; the public boundary is include/leo2d.h.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace leo2d {

// bf16 operands are stored as uint16_t with k contiguous: rows on 16-byte boundaries, leading
// dimensions multiples of 8 (elements past K are never used, only allocated)
inline int64_t pad8(int64_t n) { return (n + 7) / 8 * 8; }

// C[m][n] = sum_k A[m*lda + k] B[n*ldb + k] (FP32 accumulation), then the epilogue:
enum GemmEpilogue {
    EPI_STORE_F32 = 0,   // C32[m*ldc + n] = C
    EPI_BIAS_F32 = 1,    // C32 = C + bias[n]
    EPI_BIAS_GELU = 2,   // C16 = bf16(gelu(C + bias[n])); Z = C + bias[n] when Z is given
    EPI_GELU_BWD = 3,    // C16 = bf16(C * gelu'(Z))
    EPI_MSE = 4,         // d = C + bias[n] - T; C16 = bf16(scale d); loss[m][n / 16] = sum of d^2 over 16 n
};
struct GemmArgs {
    int epi;
    const uint16_t* A;
    int64_t lda;
    const uint16_t* B;
    int64_t ldb;
    int M, N, K;
    const float* bias;
    float* C32;
    int64_t ldc;         // of C32, Z and T
    float* Z;
    uint16_t* C16;       // [m][n], leading dimension ld16
    int64_t ld16;
    uint16_t* C16T;      // [n][m], leading dimension ld16t (nullptr: not written)
    int64_t ld16t;
    const float* T;
    float scale;
    double* loss;        // [M][(N + 15) / 16]
};
// out[c] = sum_k A[c*lda + k], c < rows (rows = 0: nothing)
struct SumArgs {
    const uint16_t* A;
    int64_t lda;
    int rows, K;
    float* out;
};
// row_loss[r] = sum over the parts of row r, in order (rows = 0: nothing)
struct LossArgs {
    const double* part;
    int rows, parts;
    double* row_loss;
};
// one or two independent products (b may be nullptr), row sums and the loss sums in one launch
hipError_t launch_gemm_bf16(const GemmArgs& a, const GemmArgs* b, const SumArgs& sums, const LossArgs& loss,
                            hipStream_t s);

// Rows idx[b] of X as bf16, [b][in] and transposed, and of T (T may be null).  ctr (may be null)
// is advanced by one: the step count of a replayed training epoch.
hipError_t launch_gather(const float* X, int in, const float* T, int out, const int64_t* idx, int rows, uint16_t* Xb,
                         int64_t ldx, uint16_t* XbT, int64_t ldxt, float* Tb, int* ctr, hipStream_t s);
// Xb[b][in] = bf16(X[b][in]); XbT as above (may be null)
hipError_t launch_cast_rows(const float* X, int in, int rows, uint16_t* Xb, int64_t ldx, uint16_t* XbT, int64_t ldxt,
                            hipStream_t s);
// mean[r][c] (may be null) over E outputs Ys[e*estride + r*cols + c]; spread[r][b] = RMS over the
// outputs of block b (cols / nblk each) of the ensemble standard deviation
hipError_t launch_ensemble_stats(const float* Ys, int E, int64_t estride, int rows, int cols, int nblk, float* mean,
                                 float* spread, hipStream_t s);

// One layer of a network's parameters: FP32 W[dout][din] at woff and biases at boff of the flat
// vector, bf16 copies W[dout][ldw] at w16 and W^T[din][ldwt] at wt16; tiles: 32 x 32 blocks of W
struct LayerDesc {
    int64_t woff, boff, w16, wt16;
    int din, dout;
    int64_t ldw, ldwt;
    int tile0;           // first workgroup of the layer in a parameter launch
};
constexpr int kParamTile = 32;
inline int param_tiles(int din, int dout)
{
    const int t = kParamTile;
    return ((din + t - 1) / t) * ((dout + t - 1) / t) + (dout + 255) / 256;   // and the biases
}
struct ParamArgs {
    const LayerDesc* layers;   // device, [nlayers]
    int nlayers, blocks;       // workgroups of all layers
    float* p;
    uint16_t *p16, *pt16;
    // Adam (grad != nullptr): moments m, v and the bias corrections c1, c2, or those of step
    // *ctr in corr[2 *ctr], corr[2 *ctr + 1] when corr is given
    const float* grad;
    float *m, *v;
    float lr, b1, b2, eps, c1, c2;
    const float* corr;
    const int* ctr;
};
// refreshes the bf16 copies from the FP32 parameters, after an Adam step on them when grad is given
hipError_t launch_params(const ParamArgs& a, hipStream_t s);
// Adam's bias corrections 1 - b1^step, 1 - b2^step
void adam_corrections(float b1, float b2, int step, float* c1, float* c2);

}  // namespace leo2d
