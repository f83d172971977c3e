// sell_build.hip -- SELL-4-sigma row tiles (sell.hip) built on the device.
//
// Every Hamiltonian a worker assembles (a k-point, a shift, a batch of cells) needs
// the tiles of its pattern before its first step.  The rows are cut into segments;
// one wavefront walks a segment's rows and cuts tiles greedily, counting a tile's
// distinct columns in a hash set in LDS; then a workgroup per tile lists the union,
// sorts the rows by length into groups of four and writes the entries' union
// indices.  Nothing but three totals comes back to the host.
// (Host threads over a copy of the pattern took 355 ms for the 24.6 million entries
// of 762 k rows and 10 ms for 24 k rows of a flake; these kernels take 2.0 and 0.2 ms.)
//
// What bounds it: the walk of a segment, row after row (about 0.5 us each,
// LDS latency), so segments are short while that fills the GPU, and at most kSegTiles
// full tiles.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.h"
#include "kpm_common.h"

namespace leo2d {
namespace {

constexpr int kSlots = 1024;          // hash set of a tile's columns: at most kSellUcap + kSellMaxLen + 1 of them
constexpr int kWalkWaves = 4;         // segments (wavefronts) per workgroup of the walk
constexpr int kTileThreads = 256;
static_assert(kSellUcap + kSellMaxLen + 1 < kSlots / 2, "the sets stay less than half full");
static_assert(kSellMaxRows <= 64 && kSellMaxLen <= 64, "a row's entries and a tile's rows fit a wavefront");

// insert c (c < 0: nothing) into the set; true in the lane whose insertion was the first
__device__ inline bool set_insert(int* table, int c)
{
    if (c < 0) return false;
    unsigned h = ((unsigned)c * 2654435761u) >> 22;
    static_assert(kSlots == 1 << 10, "hash of ten bits");
    for (;;) {
        const int old = atomicCAS(&table[h], -1, c);
        if (old == -1) return true;
        if (old == c) return false;
        h = (h + 1) & (kSlots - 1);
    }
}

// Tiles of the rows [seg_row0[g], seg_row0[g + 1]): first rows and union sizes at
// cut_row / cut_u from the segment's first row on, their number in seg_tiles[g].
// *flag is set when a row has more than kSellMaxLen entries or more columns than ucap.
__global__ __launch_bounds__(64 * kWalkWaves) void sell_cut_kernel(const int64_t* __restrict__ rp,
                                                                   const int32_t* __restrict__ col,
                                                                   const int32_t* __restrict__ seg_row0, int nseg,
                                                                   int ucap, int tmax, int32_t* cut_row, int32_t* cut_u,
                                                                   int64_t* seg_tiles, int32_t* flag)
{
    __shared__ int sets[kWalkWaves][kSlots];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = blockIdx.x * kWalkWaves + wave;
    if (g >= nseg) return;
    int* const set = sets[wave];
    const int lo = seg_row0[g], hi = seg_row0[g + 1];
    // the set is this wavefront's own: its LDS accesses stay in order
    auto clear = [&]() {
        for (int i = lane; i < kSlots; i += 64) set[i] = -1;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    };
    // a row's columns and the row itself: in the first lane without a column, while there is one
    auto insert = [&](int row, int c, int len) {
        int added = __popcll(__ballot(set_insert(set, lane == len ? row : c)));
        if (len >= 64) added += __popcll(__ballot(set_insert(set, lane == 0 ? row : -1)));
        return added;
    };
    int tiles = 0, start = lo, size = 0;
    auto close = [&](int next) {
        if (lane == 0) {
            cut_row[lo + tiles] = start;
            cut_u[lo + tiles] = size;
        }
        ++tiles;
        start = next;
        size = 0;
    };
    clear();
    // the columns of the next kAhead rows are on their way while a row's are inserted
    // (a row ahead the walk took 0.9 us a row, most of it the load)
    constexpr int kAhead = 8;
    int lens[kAhead], cols[kAhead];
    auto load = [&](int row, int& len, int& c) {
        len = 0;
        c = -1;
        if (row < hi) {
            const int64_t q0 = rp[row];
            len = (int)(rp[row + 1] - q0);
            c = lane < len ? col[q0 + lane] : -1;
        }
    };
#pragma unroll
    for (int i = 0; i < kAhead; ++i) load(lo + i, lens[i], cols[i]);
    bool fits = true;
    for (int base = lo; base < hi && fits; base += kAhead) {
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            const int r = base + i;
            const int len = lens[i], c = cols[i];
            load(r + kAhead, lens[i], cols[i]);
            if (r >= hi || !fits) continue;
            if (r - start == tmax) {
                close(r);
                clear();
            }
            int added = insert(r, c, len);
            if (size + added > ucap && r > start) {
                close(r);
                clear();
                added = insert(r, c, len);
            }
            size += added;
            fits = len <= kSellMaxLen && size <= ucap;
        }
    }
    if (!fits) {
        if (lane == 0) *flag = 1;
        return;
    }
    if (start < hi) close(hi);
    if (lane == 0) seg_tiles[g] = tiles;
}

// first rows and union sizes of all tiles, in order; the jobs' first tiles
__global__ __launch_bounds__(64) void sell_list_kernel(const int32_t* __restrict__ seg_row0,
                                                       const int64_t* __restrict__ seg_off, int nseg,
                                                       const int32_t* __restrict__ cut_row,
                                                       const int32_t* __restrict__ cut_u, int32_t* row0, int64_t* ucount,
                                                       const int32_t* __restrict__ job_seg, int njobs1, int32_t* job_tile0)
{
    const int g = blockIdx.x;
    const int64_t t0 = seg_off[g];
    const int tiles = (int)(seg_off[g + 1] - t0);
    for (int k = threadIdx.x; k < tiles; k += 64) {
        row0[t0 + k] = cut_row[seg_row0[g] + k];
        ucount[t0 + k] = cut_u[seg_row0[g] + k];
    }
    if (g == nseg - 1 && threadIdx.x == 0) row0[t0 + tiles] = seg_row0[nseg];
    if (g == 0)
        for (int j = threadIdx.x; j < njobs1; j += 64) job_tile0[j] = (int32_t)seg_off[job_seg[j]];
}

// place of each lane's row in the tile's order (longest first, ties by row)
__device__ inline int length_rank(int len, int rows, int lane)
{
    int rank = 0;
    for (int j = 0; j < rows; ++j) {
        const int other = __shfl(len, j);
        rank += other > len || (other == len && j < lane);
    }
    return rank;
}

// groups and stored entries of every tile (a wavefront each); most rows and steps of any
__global__ __launch_bounds__(64 * kWalkWaves) void sell_shape_kernel(const int64_t* __restrict__ rp,
                                                                     const int32_t* __restrict__ row0, int ntiles,
                                                                     int64_t* gcount, int64_t* ecount, int32_t* most)
{
    const int lane = threadIdx.x & 63;
    const int t = blockIdx.x * kWalkWaves + (int)(threadIdx.x >> 6);
    if (t >= ntiles) return;
    const int r0 = row0[t], rows = row0[t + 1] - r0;
    const int len = lane < rows ? (int)(rp[r0 + lane + 1] - rp[r0 + lane]) : -1;
    const int rank = length_rank(len, rows, lane);
    // a group's steps are its first row's length, rounded up to four
    const int steps = lane < rows && rank % 4 == 0 ? (len + 3) / 4 * 4 : 0;
    int sum = steps, top = steps;
    for (int off = 32; off > 0; off >>= 1) {
        sum += __shfl_xor(sum, off);
        top = max(top, __shfl_xor(top, off));
    }
    if (lane == 0) {
        gcount[t] = (rows + 3) / 4;
        ecount[t] = 4 * (int64_t)sum;
        atomicMax(&most[0], rows);
        atomicMax(&most[1], top);
    }
}

// one tile: union (own rows, then the other columns in increasing order), groups, entries
__global__ __launch_bounds__(kTileThreads) void sell_write_kernel(const int64_t* __restrict__ rp,
                                                                  const int32_t* __restrict__ col, int ntiles,
                                                                  const int32_t* __restrict__ row0,
                                                                  const int64_t* __restrict__ u0,
                                                                  const int64_t* __restrict__ g0,
                                                                  const int64_t* __restrict__ e0, int32_t* g0_out,
                                                                  int32_t* ucols, int32_t* grow, int32_t* glen,
                                                                  int64_t* goff, uint16_t* eu)
{
    __shared__ int set[kSlots];
    __shared__ int found[kSellUcap], halo[kSellUcap];
    __shared__ int order[64], glens[16];
    __shared__ int64_t goffs[16];
    __shared__ int nfound;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    constexpr int NW = kTileThreads / 64;
    const int t = blockIdx.x;
    const int r0 = row0[t], rows = row0[t + 1] - r0;
    const int64_t ub = u0[t], gb = g0[t];
    const int nhalo = (int)(u0[t + 1] - ub) - rows, groups = (int)(g0[t + 1] - gb);
    for (int i = tid; i < kSlots; i += kTileThreads) set[i] = -1;
    if (tid == 0) {
        nfound = 0;
        g0_out[t] = (int32_t)gb;
        if (t == ntiles - 1) g0_out[ntiles] = (int32_t)g0[ntiles];
    }
    __syncthreads();
    for (int i = wave; i < rows; i += NW) {
        const int64_t q0 = rp[r0 + i];
        const int len = (int)(rp[r0 + i + 1] - q0);
        const int c = lane < len ? col[q0 + lane] : -1;
        const bool fresh = set_insert(set, c >= r0 && c < r0 + rows ? -1 : c);
        if (fresh) {
            const int k = atomicAdd(&nfound, 1);
            if (k < kSellUcap) found[k] = c;
        }
    }
    if (wave == 0) {
        const int len = lane < rows ? (int)(rp[r0 + lane + 1] - rp[r0 + lane]) : -1;
        const int rank = length_rank(len, rows, lane);
        if (lane < rows) {
            order[rank] = r0 + lane;
            if (rank % 4 == 0) glens[rank / 4] = (len + 3) / 4 * 4;
        }
    }
    __syncthreads();
    // the columns in increasing order: each one's rank is the number of smaller ones
    for (int k = tid; k < nhalo; k += kTileThreads) {
        const int c = found[k];
        int rank = 0;
        for (int j = 0; j < nhalo; ++j) rank += found[j] < c;
        halo[rank] = c;
        ucols[ub + rows + rank] = c;
    }
    for (int i = tid; i < rows; i += kTileThreads) ucols[ub + i] = r0 + i;
    if (tid == 0) {
        int64_t off = e0[t];
        for (int g = 0; g < groups; ++g) {
            goffs[g] = off;
            off += 4 * glens[g];
        }
    }
    __syncthreads();
    if (tid < groups) {
        glen[gb + tid] = glens[tid];
        goff[gb + tid] = goffs[tid];
    }
    const int s = lane >> 4, k = lane & 15;
    for (int g = wave; g < groups; g += NW) {
        const int at = 4 * g + s;
        const int row = at < rows ? order[at] : -1;
        if (k == 0) grow[4 * gb + at] = row;
        const int64_t q0 = row >= 0 ? rp[row] : 0;
        const int len = row >= 0 ? (int)(rp[row + 1] - q0) : 0;
        for (int e = k; e < glens[g]; e += 16) {
            int u = 0;
            if (e < len) {
                const int c = col[q0 + e];
                if (c >= r0 && c < r0 + rows) {
                    u = c - r0;
                } else {
                    int a = 0, b = nhalo - 1;   // c is one of them
                    while (a < b) {
                        const int m = (a + b) >> 1;
                        if (halo[m] < c) a = m + 1;
                        else b = m;
                    }
                    u = rows + a;
                }
            }
            eu[goffs[g] + 4 * e + s] = (uint16_t)u;
        }
    }
}

// stored values of every group (a wavefront each) from the CSR values, zero in the padding
template <typename E>
__global__ __launch_bounds__(kTileThreads) void sell_fill_kernel(const int64_t* __restrict__ rp,
                                                                 const int32_t* __restrict__ grow,
                                                                 const int32_t* __restrict__ glen,
                                                                 const int64_t* __restrict__ goff, int ngroups,
                                                                 const E* __restrict__ src, E* __restrict__ dst)
{
    const int lane = threadIdx.x & 63;
    const int s = lane >> 4, k = lane & 15;
    const int stride = gridDim.x * (kTileThreads / 64);
    for (int g = blockIdx.x * (kTileThreads / 64) + (int)(threadIdx.x >> 6); g < ngroups; g += stride) {
        const int row = grow[4 * (int64_t)g + s];
        const int64_t q0 = row >= 0 ? rp[row] : 0;
        const int len = row >= 0 ? (int)(rp[row + 1] - q0) : 0;
        const int steps = glen[g];
        const int64_t o = goff[g];
        for (int e = k; e < steps; e += 16) {
            E v;
            zero(v);
            if (e < len) v = src[q0 + e];
            dst[o + 4 * e + s] = v;
        }
    }
}

}  // namespace

hipError_t launch_sell_cut(const int64_t* rp, const int32_t* col, const int32_t* seg_row0, int nseg, int ucap, int tmax,
                           int32_t* cut_row, int32_t* cut_u, int64_t* seg_tiles, int32_t* flag, hipStream_t s)
{
    if (ucap > kSellUcap || tmax > kSellMaxRows || tmax < 1 || nseg < 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL(sell_cut_kernel, dim3((nseg + kWalkWaves - 1) / kWalkWaves), dim3(64 * kWalkWaves), 0, s, rp, col,
                       seg_row0, nseg, ucap, tmax, cut_row, cut_u, seg_tiles, flag);
    return hipGetLastError();
}

hipError_t launch_sell_list(const int64_t* rp, const int32_t* seg_row0, const int64_t* seg_off, int nseg, int ntiles,
                            const int32_t* cut_row, const int32_t* cut_u, int32_t* row0, int64_t* ucount, int64_t* gcount,
                            int64_t* ecount, int32_t* most, const int32_t* job_seg, int njobs1, int32_t* job_tile0,
                            hipStream_t s)
{
    hipLaunchKernelGGL(sell_list_kernel, dim3(nseg), dim3(64), 0, s, seg_row0, seg_off, nseg, cut_row, cut_u, row0, ucount,
                       job_seg, njobs1, job_tile0);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(sell_shape_kernel, dim3((ntiles + kWalkWaves - 1) / kWalkWaves), dim3(64 * kWalkWaves), 0, s, rp,
                       row0, ntiles, gcount, ecount, most);
    return hipGetLastError();
}

hipError_t launch_sell_write(const int64_t* rp, const int32_t* col, int ntiles, const int32_t* row0, const int64_t* u0,
                             const int64_t* g0, const int64_t* e0, int32_t* g0_out, int32_t* ucols, int32_t* grow,
                             int32_t* glen, int64_t* goff, uint16_t* eu, hipStream_t s)
{
    hipLaunchKernelGGL(sell_write_kernel, dim3(ntiles), dim3(kTileThreads), 0, s, rp, col, ntiles, row0, u0, g0, e0,
                       g0_out, ucols, grow, glen, goff, eu);
    return hipGetLastError();
}

hipError_t launch_sell_fill(const int64_t* rp, const int32_t* grow, const int32_t* glen, const int64_t* goff, int ngroups,
                            const void* src, void* dst, int elem_bytes, hipStream_t s)
{
    if (ngroups <= 0) return hipSuccess;
    const dim3 grid((unsigned)std::min(8192, (ngroups + 3) / 4)), block(kTileThreads);
    switch (elem_bytes) {
    case 4:
        hipLaunchKernelGGL(sell_fill_kernel<float>, grid, block, 0, s, rp, grow, glen, goff, ngroups, (const float*)src,
                           (float*)dst);
        break;
    case 8:
        hipLaunchKernelGGL(sell_fill_kernel<double>, grid, block, 0, s, rp, grow, glen, goff, ngroups,
                           (const double*)src, (double*)dst);
        break;
    case 16:
        hipLaunchKernelGGL(sell_fill_kernel<double2>, grid, block, 0, s, rp, grow, glen, goff, ngroups,
                           (const double2*)src, (double2*)dst);
        break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace leo2d
