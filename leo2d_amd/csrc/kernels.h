// kernels.h -- launchers for the HIP kernels (kpm.hip, dos.hip, assemble.hip).
// Internal to libleo2d; the public boundary is include/leo2d.h.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace leo2d {

// element types of a KPM launch
enum MatType { MAT_REAL_F64 = 0, MAT_CPX_F64 = 1, MAT_REAL_F32 = 2, MAT_CPX_F32 = 3 };
enum VecType { VEC_REAL_F64 = 0, VEC_CPX_F64 = 1, VEC_CPX_F32 = 2, VEC_REAL_F32 = 3 };

inline size_t vec_bytes(int vt) { return vt == VEC_CPX_F64 ? 16 : (vt == VEC_REAL_F32 ? 4 : 8); }

// One Chebyshev step over a block of R vectors stored row-major [n][R]:
//   out = alpha * H * cur - (beta ? prev : 0)        (out may alias prev)
// and per-vector partial sums for the moment reductions:
//   part[g][r][0] = sum_i |cur_ir|^2
//   part[g][r][1] = sum_i Re(conj(out_ir) cur_ir)
//   part[g][r][2] = sum_i Re(conj(v_ir) cur_ir)      (only when v != nullptr)
struct StepArgs {
    const int64_t* row_ptr;
    const int32_t* col;
    const void* val;
    int n;
    int R;
    const void* cur;
    const void* prev;
    void* out;
    const void* v;
    double alpha;
    int beta;
    double* part;   // [grid][R][3]
    const int32_t* targets;   // with tval: the row of each vector's unit start vector
    double* tval;             // tval[r tstride] <- Re cur[targets[r]][r] (nullptr: not wanted)
    int tstride;
    int grid;       // number of workgroups (multiple of 8)
    int variant;    // 0 = lane per vector (any R), 1 = wavefront per row (R >= 64), 2 = group of lanes per row
                    // (FP64, R <= 8), 14 = vector chunks split
                    // over the XCDs (R = 16, 32, 64, 128), 15 = two rows per wavefront, 16-byte FP32 gathers
                    // (complex FP32, R = 64)
    int long_rows;  // variant 2: 1 = a wavefront per row instead of 16 lanes
    int xcd_rows;   // variant 1: rows per XCD slice (0 = interleave rows over the grid)
};

// entries allocated after nnz in every device CSR, so kernels may load whole chunks of a row
// (column 0 and value 0 in the spatially ordered CSR, unset elsewhere)
constexpr int kCsrPad = 16;
hipError_t launch_kpm_step(int mat_type, int vec_type, const StepArgs& a, hipStream_t s);

// ---- SELL-4-sigma step with LDS-staged row tiles (sell.hip) -----------------
// Tiles of at most kSellMaxRows consecutive rows whose distinct columns (the
// union, own rows first) fit `ucap` LDS rows of 256 B; each tile's rows sorted
// by length into groups of 4 (SELL-C-sigma with C = 4, sigma = the tile).
constexpr int kSellMaxRows = 64;    // rows per tile (8 wavefronts x 2 groups x 4 rows)
constexpr int kSellMaxLen = 64;     // longest row a group can hold
constexpr int kSellUcap = 288;      // staged rows per LDS buffer (two buffers of 288 x 256 B)
constexpr int kSellUcapTiled = 256; // the same with per-tile partials (their LDS takes the difference)
constexpr int kSellWaves = 8;       // wavefronts per workgroup (one workgroup per CU)
constexpr int kSellCwWaves = 7;     // compute wavefronts beside the copy wavefront (copy_wave)
constexpr int kSellCwRows = 56;     // rows per tile with a copy wavefront (7 wavefronts x 2 groups x 4 rows)
struct SellStepArgs {
    int n;
    int R;
    const void* cur;
    const void* prev;
    void* out;
    const void* v;
    double alpha;
    int beta;
    double* part;               // [grid][R][3], or [ntiles][R][2] with tile_part
    int grid;
    int tile_part;              // 1: partial sums per tile (stacked jobs), at most kSellUcapTiled union rows
    int ucap;                   // union rows the tiles were cut to
    int ntiles;
    const int32_t* tile_row0;   // [ntiles + 1]
    const int64_t* tile_u0;     // [ntiles + 1] offsets into ucols
    const int32_t* ucols;       // union rows of every tile (own rows first)
    const int32_t* tile_g0;     // [ntiles + 1] first group of each tile
    const int32_t* grow;        // [groups][4] row of each group slot (-1: empty)
    const int32_t* glen;        // [groups] steps of the group (multiple of 4, <= kSellMaxLen)
    const int64_t* goff;        // [groups] first entry of the group; entry e of slot s at goff + 4 e + s
    const uint16_t* eu;         // [entries] union index of the entry's column
    const void* ev;             // [entries] value (matrix element type)
    int tile_rows;              // most rows in a tile (<= kSellMaxRows)
    int max_len;                // most steps in a group (<= kSellMaxLen)
    int sliced;                 // 1: XCD x walks its own contiguous eighth of the tiles
    int reverse;                // 1: every workgroup walks its tiles last to first (alternate steps)
    int copy_wave;              // 1: staging copies issued by a wavefront of their own (tiles <= kSellCwRows)
};
// copy_wave: 16 complex FP32 vectors (128-byte row chunks) need the copy-wavefront kernel
bool sell_supported(int mat_type, int vec_type, int R, bool copy_wave);
hipError_t launch_kpm_step_sell(int mat_type, int vec_type, const SellStepArgs& a, hipStream_t s);
// Their layout, built on the device (sell_build.hip).  Segments of rows are cut into tiles on
// their own (a tile never crosses a segment); then the tiles are listed and measured, and after
// the scans of their union rows, groups and entries written.
constexpr int kSegTiles = 48;   // full tiles in a segment, at most
hipError_t launch_sell_cut(const int64_t* rp, const int32_t* col, const int32_t* seg_row0, int nseg, int ucap, int tmax,
                           int32_t* cut_row, int32_t* cut_u, int64_t* seg_tiles, int32_t* flag, hipStream_t s);
// most[0], most[1] (zero before): most rows of a tile, most steps of a group; job_tile0[j] = first
// tile of segment job_seg[j], j < njobs1
hipError_t launch_sell_list(const int64_t* rp, const int32_t* seg_row0, const int64_t* seg_off, int nseg, int ntiles,
                            const int32_t* cut_row, const int32_t* cut_u, int32_t* row0, int64_t* ucount, int64_t* gcount,
                            int64_t* ecount, int32_t* most, const int32_t* job_seg, int njobs1, int32_t* job_tile0,
                            hipStream_t s);
hipError_t launch_sell_write(const int64_t* rp, const int32_t* col, int ntiles, const int32_t* row0, const int64_t* u0,
                             const int64_t* g0, const int64_t* e0, int32_t* g0_out, int32_t* ucols, int32_t* grow,
                             int32_t* glen, int64_t* goff, uint16_t* eu, hipStream_t s);
// the stored values of every group from the CSR values (elements of 4, 8 or 16 bytes)
hipError_t launch_sell_fill(const int64_t* rp, const int32_t* grow, const int32_t* glen, const int64_t* goff, int ngroups,
                            const void* src, void* dst, int elem_bytes, hipStream_t s);

// Deterministic reduction of the partials of `steps` consecutive steps from j0 on
// into moments (step 0 in a launch of its own: the others read its moments).
//   scheme 0 (reference, target starts): mu_j = Re T_j[target_r][r] for j < M/2 is
//            written by the steps themselves (tval = mu + j); dots for j >= M/4
//            (locality.cpp:6002-6034)
//   scheme 1 (doubling from j = 1): mu_{2j}, mu_{2j+1} from the dots
//   scheme 2 (reference, vector starts): mu_j = part[..][2] for j < M/2
struct ReduceArgs {
    const double* part;      // [steps][grid][R][3]
    int grid;
    int R;
    int M;
    int j0;                  // first step (step 0 = the product T1 = H T0)
    int steps;
    int scheme;
    double* mu;              // [R][M] device
};
// steps whose partials a recursion collects before it reduces them, for partials of step_bytes
// a step in `space` bytes
inline int reduce_every(size_t step_bytes, size_t space, int M)
{
    const size_t k = space / (step_bytes ? step_bytes : 1);
    const size_t most = (size_t)(M / 2);
    return (int)(k < 1 ? 1 : (k < most ? k : most));
}
// Partials kept before a reduction: 10 to 20 steps of a full grid, so a reduction's launch is a
// small part of a step.  (32 MiB allocated and freed by every call cost as much as it saved.)
constexpr size_t kPartialSpace = size_t(4) << 20;
// The same for a batch, whose buffers stay with the handle between calls.
constexpr size_t kBatchPartialSpace = size_t(32) << 20;
hipError_t launch_kpm_reduce(const ReduceArgs& a, hipStream_t s);
// tval[r tstride] <- Re cur[targets[r]][r], for steps that do not write it themselves (the SELL step)
hipError_t launch_target_values(const void* cur, int vec_type, const int32_t* targets, int R, double* tval, int tstride,
                                hipStream_t s);

// ---- batched recursion over many stacked Hamiltonians (batch.hip) ----------
// One step for every job of a block-diagonal stack: out = alpha*H*cur - (beta ?
// out : 0) with per-tile partials part[t][r][0] = sum |cur|^2,
// part[t][r][1] = sum Re(conj(out) cur) over the rows of tile t.
struct BatchStepArgs {
    const int64_t* row_ptr;
    const int32_t* col;
    const void* val;
    const void* cur;
    void* out;                 // T_{j-1} in, T_{j+1} out
    double alpha;
    int beta;
    int R;                     // vectors per job: 4, 8, 16 or 32
    const int32_t* tile_row0;  // [ntiles + 1]; tiles never cross a job boundary
    int ntiles;
    double* part;              // [ntiles][R][2]
    int grid;                  // workgroups (multiple of 8)
    int mode;                  // 0 = row groups, 1 = entry slots, 2 = row chunks (R = 16, 32)
};
hipError_t launch_batch_step(int mat_type, int vec_type, const BatchStepArgs& a, hipStream_t s);
// mu[p][r][M] of job p from its tiles [job_tile0[p], job_tile0[p+1]) (doubling identity), for `steps`
// steps from j0 on with partials part[step][ntiles][R][2]; step 0 in a launch of its own
hipError_t launch_batch_reduce(const double* part, const int32_t* job_tile0, int ntiles, int P, int R, int M, int j0,
                               int steps, double* mu, hipStream_t s);
// start vectors: random phases (vector r of job p = global vector p*R + r), or,
// when targets != nullptr, the unit vector on orbital targets[p*R + r] of job p
hipError_t launch_batch_init(void* x, int vec_type, const int64_t* job_row0, int P, int64_t nrows, int R, uint64_t seed,
                             const int32_t* targets, hipStream_t s);
hipError_t launch_batch_offset(const int32_t* col_in, int64_t nnz, int32_t row_off, int32_t* col_out,
                               const int64_t* rp_in, int n, int64_t nnz_off, int64_t* rp_out, hipStream_t s);

// start vectors
hipError_t launch_init_targets(void* x, int vec_type, int n, int R, const int32_t* targets, hipStream_t s);
hipError_t launch_init_random_phase(void* x, int vec_type, int n, int R, uint64_t seed, int r0, hipStream_t s);
hipError_t launch_init_from_host_layout(void* x, int vec_type, const double* src, int src_complex, int n, int R,
                                        hipStream_t s);
hipError_t launch_convert_f64_to_f32(const double* in, float* out, int64_t count, hipStream_t s);

// spatial permutation support (q = new row, i = iperm[q] = original row)
hipError_t launch_init_random_phase_perm(void* x, int vec_type, int n, int R, uint64_t seed, int r0,
                                        const int32_t* iperm, hipStream_t s);
hipError_t launch_init_from_host_layout_perm(void* x, int vec_type, const double* src, int src_complex, int n, int R,
                                             const int32_t* iperm, hipStream_t s);
hipError_t launch_perm_len(const int64_t* rp, const int32_t* iperm, int n, int64_t* len, hipStream_t s);
hipError_t launch_perm_fill(const int64_t* rp, const int32_t* col, const void* val, int val_bytes, const int32_t* iperm,
                            const int32_t* perm, int n, const int64_t* prp, int32_t* pcol, void* pval, hipStream_t s);
hipError_t scan_exclusive_i64(const int64_t* cnt, int64_t* out, int n, hipStream_t s);

// KPM conductivity (cond.hip): blk [n][B] -> set[b][m][n]; X = 2 g_i g_j C
// (Jackson g / sqrt 2); column-major DCT-III matrix P(k, i) = w_i cos(pi i (k+1/2)/M)
hipError_t launch_cond_scatter(const double* blk, int n, int B, int m, int M, double* set, hipStream_t s);
// one index of the conductivity recursion on a real [n][B] block: out = alpha H x - (beta ? prev : 0)
// (hset[b][j][.] = out when hset != nullptr) and dset[b][j][.] = dxH x; hv or dv may be nullptr
hipError_t launch_cond_dual_step(const int64_t* rp, const int32_t* col, const double* hv, const double* dv,
                                 const double* x, const double* prev, double* out, double alpha, int beta, int n, int B,
                                 int j, int M, double* hset, double* dset, hipStream_t s);
// both recursions of up to kCondPair targets on x = [n][2B], betas first: x_j = alpha H x - (beta ? prev : 0),
// its beta half into hset as vector j >= 1, dxH times the alpha half of x into dset as vector j - 1
constexpr int kCondPair = 4;
hipError_t launch_cond_pair_step(const int64_t* rp, const int32_t* col, const double* hv, const double* dv,
                                 const double* x, const double* prev, double* out, double alpha, int beta, int n, int B,
                                 int j, int M, double* hset, double* dset, hipStream_t s);
// x_0 from the targets' unit vectors (also into hset as vector 0) and a0 = [n][B]; the alpha half of x
hipError_t launch_cond_pair_start(const int32_t* targets, const double* a0, int n, int B, int M, double* x, double* hset,
                                  hipStream_t s);
hipError_t launch_cond_pair_alpha(const double* x, int n, int B, double* a, hipStream_t s);
hipError_t launch_cond_weight(const double* C, int M, int T, double* X, hipStream_t s);
// C[b] = sum_c part[b][c] (c = 0 .. S-1, fixed order), blocks of mm values
hipError_t launch_cond_chunk_sum(const double* part, int S, size_t mm, int B, double* C, hipStream_t s);
hipError_t launch_dct3_matrix(int M, double* P, hipStream_t s);

// FP64 GEMM on the matrix cores (dgemm.hip), batched and split along k:
//   C[b][s](m, n) = sum_{k in split s} A_b(m, k) B_b(k, n)
//   A_b(m, k) = A[b sab + m sam + k sak], B_b(k, n) = B[b sbb + n sbn + k sbk],
//   C[b][s](m, n) at C[b scb + s scs + m scm + n scn]
// split s covers k in [s kc, (s+1) kc), kc = ceil(K / splits) rounded up to 16
struct DgemmArgs {
    int M, N, K;
    int batch;
    int splits;
    int kchunk;     // set by the launcher
    const double* A;
    int64_t sam, sak, sab;
    const double* B;
    int64_t sbn, sbk, sbb;
    double* C;
    int64_t scm, scn, scb, scs;
};
hipError_t launch_dgemm(const DgemmArgs& a, hipStream_t s);

// Jackson-kernel DoS: rho[t][k] = DCT-III(g * mu[t]) / (pi sqrt(a^2 - (E_k - b)^2)) * scale;
// work: dos_workspace(T, M) bytes of device scratch
size_t dos_workspace(int T, int M);
hipError_t launch_dos(const double* mu, int T, int M, double a, double b, double scale, double* E, double* rho,
                      double* work, hipStream_t s);

// Static device workspace of the allocation-free KPM entry point (scratch.hip).
// scratch_init(d) looks up device d's address of the array (d must be current);
// scratch_ptr(d) returns it (nullptr before scratch_init succeeded).
constexpr size_t kScratchBytes = size_t(64) << 20;
hipError_t scratch_init(int device);
void* scratch_ptr(int device);
hipError_t launch_zero_f64(double* p, int64_t count, hipStream_t s);

// Gershgorin interval of a CSR matrix: lo = min_i (Re H_ii - R_i), hi = max_i (Re H_ii + R_i)
hipError_t launch_gershgorin(const int64_t* rp, const int32_t* col, const void* val, int is_complex, int n,
                             double* lohi /*[2*blocks]*/, int blocks, hipStream_t s);

}  // namespace leo2d
