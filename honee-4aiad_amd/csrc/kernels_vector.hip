// Vector and restriction kernels of the MI355X backend (CeedVector arithmetic, norms, multiplicity, restriction apply).
// All are bandwidth-bound streaming kernels with grid-stride loops.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.hpp"

namespace {

constexpr int kBlock = 256;

inline int grid_for(long long n) {
  long long g = (n + kBlock - 1) / kBlock;
  if (g > 65536) g = 65536;
  if (g < 1) g = 1;
  return (int)g;
}

__global__ void k_fill(double *x, double v, long long n) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) x[i] = v;
}
__global__ void k_axpby(double *y, double a, double b, const double *x, long long n) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) y[i] = a * x[i] + b * y[i];
}
__global__ void k_scale(double *x, double a, long long n) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) x[i] *= a;
}
__global__ void k_pmult(double *w, const double *x, const double *y, long long n) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) w[i] = x[i] * y[i];
}
__global__ void k_recip(double *x, long long n) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    if (fabs(x[i]) > 1e-300) x[i] = 1.0 / x[i];
}

// Per-block partial: 0 -> sum|x|, 1 -> sum x^2, 2 -> max|x|; npartial blocks, results in partial[block]
__global__ void k_norm(const double *x, long long n, int type, double *partial) {
  __shared__ double red[kBlock];
  double            acc = 0;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const double v = x[i];
    if (type == 0) acc += fabs(v);
    else if (type == 1) acc += v * v;
    else acc = fmax(acc, fabs(v));
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = kBlock / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] = (type == 2) ? fmax(red[threadIdx.x], red[threadIdx.x + s]) : red[threadIdx.x] + red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

__global__ void k_multiplicity(const int *off, long long n, int ncomp, int cs, double *mult) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    for (int c = 0; c < ncomp; c++) atomicAdd(&mult[off[i] + c * cs], 1.0);
}

// E-vector layout [elem][comp][node] (libCEED's offset-restriction E-vector ordering)
__global__ void k_rstr_n(const int *off, int nelem, int esize, int ncomp, int cs, const double *u, double *e) {
  const long long n = (long long)nelem * esize;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const long long el = i / esize, node = i % esize;
    for (int c = 0; c < ncomp; c++) e[(el * ncomp + c) * esize + node] = u[off[i] + c * cs];
  }
}
__global__ void k_rstr_t(const int *off, int nelem, int esize, int ncomp, int cs, const double *e, double *u) {
  const long long n = (long long)nelem * esize;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const long long el = i / esize, node = i % esize;
    for (int c = 0; c < ncomp; c++) atomicAdd(&u[off[i] + c * cs], e[(el * ncomp + c) * esize + node]);
  }
}

// Deterministic second scatter pass: one thread per (L-vector node, component) item.  Row k's contributions are the
// E-vector slots t_rowptr[k] .. t_rowptr[k+1]-1 (node-sorted E-vector); they are summed in ascending order.  Each thread
// handles NPT items a grid stride apart and issues all their row-pointer loads, then all their contribution loads (up to 8
// per row, the most a hexahedral mesh node has), so a thread waits on two memory round trips for NPT items.
template <int NPT>
__global__ void __launch_bounds__(256) k_node_gather(int nrows, int ncomp, int cs, const int *__restrict__ rowptr, const int *__restrict__ toff,
                                                     const double *__restrict__ ev, double *__restrict__ v, bool overwrite) {
  const long long n      = (long long)nrows * ncomp;
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long i0 = (long long)blockIdx.x * blockDim.x + threadIdx.x; i0 < n; i0 += stride * NPT) {
    int row[NPT], c[NPT], b[NPT], m[NPT];
#pragma unroll
    for (int j = 0; j < NPT; j++) {
      const long long i = i0 + j * stride;
      row[j]            = i < n ? (int)(i / ncomp) : 0;
      c[j]              = i < n ? (int)(i % ncomp) : 0;
      b[j]              = rowptr[row[j]];
      m[j]              = i < n ? rowptr[row[j] + 1] - b[j] : 0;
    }
    double acc[NPT];
#pragma unroll
    for (int j = 0; j < NPT; j++) acc[j] = 0;
    bool more = false;
#pragma unroll
    for (int j = 0; j < NPT; j++) more |= m[j] > 8;
    if (!more) {  // every row has at most 8 contributions: one batch of loads
      double x[NPT][8];
#pragma unroll
      for (int j = 0; j < NPT; j++)
#pragma unroll
        for (int k = 0; k < 8; k++) {
          x[j][k] = 0;
          if (k < m[j]) x[j][k] = ev[(long long)(b[j] + k) * ncomp + c[j]];
        }
#pragma unroll
      for (int j = 0; j < NPT; j++)
#pragma unroll
        for (int k = 0; k < 8; k++)
          if (k < m[j]) acc[j] += x[j][k];
    } else {
#pragma unroll
      for (int j = 0; j < NPT; j++)
        for (int k = 0; k < m[j]; k++) acc[j] += ev[(long long)(b[j] + k) * ncomp + c[j]];
    }
#pragma unroll
    for (int j = 0; j < NPT; j++) {
      if (i0 + j * stride < n) {
        double *dst = &v[toff[row[j]] + (long long)c[j] * cs];
        *dst        = overwrite ? acc[j] : *dst + acc[j];
      }
    }
  }
}

__global__ void __launch_bounds__(256) k_inverse_permutation(const int *__restrict__ index, long long n, int *__restrict__ perm) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) perm[index[i]] = (int)i;
}

// Slots of a tile in ascending order and the place there of each, by counting the smaller ones (they differ); a block per tile.
// Run once per restriction.
__global__ void __launch_bounds__(256) k_layout_tiles(GatherTiles g, const int *__restrict__ index, int *__restrict__ slot,
                                                      unsigned short *__restrict__ pos) {
  __shared__ int s[kGatherSlots];
  const int      r0 = g.tile_row[blockIdx.x], j0 = g.rowptr[r0], m = g.rowptr[g.tile_row[blockIdx.x + 1]] - j0;
  if (m > kGatherSlots) {  // one row, ascending as it is; its places are not read
    for (int j = threadIdx.x; j < m; j += 256) slot[j0 + j] = index[j0 + j];
    return;
  }
  for (int j = threadIdx.x; j < m; j += 256) s[j] = index[j0 + j];
  __syncthreads();
  for (int j = threadIdx.x; j < m; j += 256) {
    int rank = 0;
    for (int i = 0; i < m; i++) rank += s[i] < s[j] ? 1 : 0;
    slot[j0 + rank] = s[j];
    pos[j0 + j]     = (unsigned short)rank;
  }
}

// The same sum for the element-ordered E-vector of 5 components, a tile of consecutive rows per block.  The block loads the
// tile's slots in ascending address order, lanes along the 40 bytes of a slot and on to the next, so that each line is asked
// for by one or two wave loads; it then sums each (row, component) from LDS over the row's slots in ascending order, as in
// k_node_gather (identical results).  A thread per row that reads its slots straight from memory asks for each line 5 to 10
// times and spends the time on requests that wait for a line already on its way (measured: 0.9 of the cycles, and L2 to L1
// traffic of 4.7 times the E-vector at p=2).
// Tiles hold at most kGatherSlots slots (23.6 KB of LDS with the places and row starts: 6 blocks a CU) and as many rows; a row with more slots is a tile by
// itself, summed straight from memory.  The tiles are split into 8 contiguous ranges, one per XCD (block b runs on XCD
// b % 8; the grid is a multiple of 8), so that a range's E-vector lines go to one L2.
// Measured against a thread per row: 64^3 p=2 177 -> 122 us (3.4 TB/s), 40^3 p=4 196 -> 158 us, 32^3 p=3 50 -> 44 us.
// E is the E-vector's type: double, or float for the FP32 Jacobian's contributions (summed in FP64 here).
template <typename E>
__global__ void __launch_bounds__(256) k_node_gather_tiles(GatherTiles g, int cs, const E *__restrict__ ev, double *__restrict__ v, bool overwrite) {
  constexpr int NC = 5, NT = 256, NL = kGatherSlots * NC / NT;
  __shared__ E              buf[kGatherSlots * NC];
  __shared__ unsigned short pos[kGatherSlots];
  __shared__ int            first[kGatherSlots + 1];
  const int per = (g.ntile + 7) / 8, tile = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  if ((int)(blockIdx.x / 8) >= per || tile >= g.ntile) return;
  const int r0 = g.tile_row[tile], nr = g.tile_row[tile + 1] - r0, j0 = g.rowptr[r0], m = g.rowptr[r0 + nr] - j0, tid = threadIdx.x;
  auto store = [&](int row, int c, double acc) {
    const long long o = (g.stride ? (long long)row * g.stride : (long long)g.toff[row]) + (long long)c * cs;
    v[o]              = overwrite ? acc : v[o] + acc;
  };
  if (m > kGatherSlots) {  // one row
    if (tid < NC) {
      double acc = 0;
      for (int k = 0; k < m; k++) acc += (double)ev[(long long)g.slot[j0 + k] * NC + tid];
      store(r0, tid, acc);
    }
    return;
  }
  int s[NL];
  E   x[NL];
#pragma unroll
  for (int u = 0; u < NL; u++) {
    const int i = tid + u * NT;
    s[u]        = i < m * NC ? g.slot[j0 + i / NC] : 0;
  }
#pragma unroll
  for (int u = 0; u < NL; u++) {
    const int i = tid + u * NT;
    x[u]        = i < m * NC ? ev[(long long)s[u] * NC + i % NC] : (E)0;
  }
  for (int i = tid; i <= nr; i += NT) first[i] = g.rowptr[r0 + i] - j0;
  for (int i = tid; i < m; i += NT) pos[i] = (unsigned short)(g.pos[j0 + i] * NC);
#pragma unroll
  for (int u = 0; u < NL; u++)
    if (tid + u * NT < m * NC) buf[tid + u * NT] = x[u];
  __syncthreads();
  for (int i = tid; i < nr * NC; i += NT) {
    const int row = i / NC, c = i % NC, end = first[row + 1];
    double    acc = 0;
    for (int k = first[row]; k < end; k++) acc += (double)buf[pos[k] + c];
    store(r0 + row, c, acc);
  }
}

// The point-block form of the element-ordered gather: the E-vector holds a 5 x 5 block [c_out][c_in] per element node
// (25 consecutive values), the output a block per node at 25 * (offset / 5) (the L-vector offsets of an interleaved
// 5-component field are 5 * node).  One thread per (node, c_out) row of the block sums its 5 values over the node's
// contributions in ascending slot order and writes them to the output, or adds them.
__global__ void __launch_bounds__(256) k_node_gather_blocks(int nrows, const int *__restrict__ rowptr, const int *__restrict__ index,
                                                            const int *__restrict__ toff, const double *__restrict__ ev, double *__restrict__ v,
                                                            bool overwrite) {
  const long long n = (long long)nrows * 5;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const int row = (int)(i / 5), co = (int)(i % 5);
    const int b = rowptr[row], m = rowptr[row + 1] - b;
    double    acc[5] = {0, 0, 0, 0, 0};
    for (int k = 0; k < m; k++) {
      const double *src = ev + (long long)index[b + k] * 25 + co * 5;
#pragma unroll
      for (int c = 0; c < 5; c++) acc[c] += src[c];
    }
    double *dst = v + (long long)toff[row] * 5 + co * 5;
#pragma unroll
    for (int c = 0; c < 5; c++) dst[c] = overwrite ? acc[c] : dst[c] + acc[c];
  }
}

// Per-block partial sums of x . y over a fixed grid (deterministic for a given n and npartial)
__global__ void k_dot(const double *x, const double *y, long long n, double *partial) {
  __shared__ double red[kBlock];
  double            acc = 0;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) acc += x[i] * y[i];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = kBlock / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// ---- Conjugate gradients ----
// Streaming kernels over the vectors of one iteration, bound by their bytes: 2 vectors read for p.Ap, 5 read and 2 written
// by the update, 3 read and 1 written by the direction, against 21 by separate dot, axpy and multiply calls.  A kernel that
// needs a scalar sums the block partials before it itself (4 KB per block, out of L2), which costs no launch and no host read.
// Measured at 2.9 M entries: 53 us an iteration (dot 9.0, residual 29.2, direction 15.1), 142 us before (with the fill and the
// reads' synchronizations).
constexpr int kCgThreads = 512;

__device__ __forceinline__ double cg_block_sum(double v, double *s) {  // s: one value per wave
#pragma unroll
  for (int w = 32; w > 0; w >>= 1) v += __shfl_down(v, w);
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = v;
  __syncthreads();
  double r = 0;
#pragma unroll
  for (int i = 0; i < kCgThreads / 64; i++) r += s[i];
  __syncthreads();
  return r;
}
// Sum of the nb <= kCgThreads partials, in every block alike
__device__ __forceinline__ double cg_total(const double *partial, int nb, double *s) {
  return cg_block_sum((int)threadIdx.x < nb ? partial[threadIdx.x] : 0.0, s);
}
// f(i) over the thread's entries
template <class F>
__device__ __forceinline__ void cg_each(long long n, F &&f) {
  const long long stride = (long long)gridDim.x * kCgThreads;
  for (long long i = (long long)blockIdx.x * kCgThreads + threadIdx.x; i < n; i += stride) f(i);
}
__device__ __forceinline__ void cg_publish(const CgArgs &a, double v) {
  a.h[0] = v;
  __threadfence_system();
  __hip_atomic_store(a.flag, a.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ void __launch_bounds__(kCgThreads) k_cg_start(CgArgs a) {
  __shared__ double s[kCgThreads / 64];
  double            acc = 0;
  cg_each(a.n, [&](long long i) {
    const double r = a.rhs[i], z = a.dinv[i] * r;
    a.x[i] = 0.0;
    a.r[i] = r;
    a.p[i] = z;
    acc += r * z;
  });
  acc = cg_block_sum(acc, s);
  if (threadIdx.x == 0) a.scratch[blockIdx.x] = acc;
}
__global__ void __launch_bounds__(kCgThreads) k_cg_start_total(CgArgs a, int nb) {
  __shared__ double s[kCgThreads / 64];
  const double      rz = cg_total(a.scratch, nb, s);
  if (threadIdx.x == 0) {
    a.scratch[2 * kCgBlocks] = rz;
    cg_publish(a, rz);
  }
}
__global__ void __launch_bounds__(kCgThreads) k_cg_dot(CgArgs a) {
  __shared__ double s[kCgThreads / 64];
  double            acc = 0;
  cg_each(a.n, [&](long long i) { acc += a.p[i] * a.ap[i]; });
  acc = cg_block_sum(acc, s);
  if (threadIdx.x == 0) a.scratch[kCgBlocks + blockIdx.x] = acc;
}
__global__ void __launch_bounds__(kCgThreads) k_cg_residual(CgArgs a, int nb) {
  __shared__ double s[kCgThreads / 64];
  const double      alpha = a.scratch[2 * kCgBlocks + a.odd] / cg_total(a.scratch + kCgBlocks, nb, s);
  double            acc   = 0;
  cg_each(a.n, [&](long long i) {
    a.x[i] += alpha * a.p[i];
    const double r = a.r[i] - alpha * a.ap[i];
    a.r[i]         = r;
    acc += r * (a.dinv[i] * r);
  });
  acc = cg_block_sum(acc, s);
  if (threadIdx.x == 0) a.scratch[blockIdx.x] = acc;
}
__global__ void __launch_bounds__(kCgThreads) k_cg_direction(CgArgs a, int nb) {
  __shared__ double s[kCgThreads / 64];
  const double      rz = cg_total(a.scratch, nb, s), beta = rz / a.scratch[2 * kCgBlocks + a.odd];
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    a.scratch[2 * kCgBlocks + (a.odd ^ 1)] = rz;
    cg_publish(a, rz);
  }
  cg_each(a.n, [&](long long i) { a.p[i] = a.dinv[i] * a.r[i] + beta * a.p[i]; });
}

int cg_blocks(long long n) { return (int)std::min<long long>(kCgBlocks, std::max<long long>(1, (n + kCgThreads - 1) / kCgThreads)); }

}  // namespace

hipError_t launch_cg_start(const CgArgs &a, hipStream_t s) {
  const int nb = cg_blocks(a.n);
  hipLaunchKernelGGL(k_cg_start, dim3(nb), dim3(kCgThreads), 0, s, a);
  hipLaunchKernelGGL(k_cg_start_total, dim3(1), dim3(kCgThreads), 0, s, a, nb);
  return hipGetLastError();
}
hipError_t launch_cg_dot(const CgArgs &a, hipStream_t s) {
  hipLaunchKernelGGL(k_cg_dot, dim3(cg_blocks(a.n)), dim3(kCgThreads), 0, s, a);
  return hipGetLastError();
}
hipError_t launch_cg_update(const CgArgs &a, hipStream_t s) {
  const int nb = cg_blocks(a.n);
  hipLaunchKernelGGL(k_cg_residual, dim3(nb), dim3(kCgThreads), 0, s, a, nb);
  hipLaunchKernelGGL(k_cg_direction, dim3(nb), dim3(kCgThreads), 0, s, a, nb);
  return hipGetLastError();
}

hipError_t launch_node_gather(int nrows, int ncomp, int comp_stride, const int *t_rowptr, const int *t_offset, const double *ev, double *v,
                              bool overwrite, hipStream_t s) {
  constexpr int   NPT = 2;  // measured: 2 items per thread 31.8 us against 39.1 us (1) and 39.0 us (4) at 884,736 rows
  const long long n   = (long long)nrows * ncomp;
  if (n <= 0) return hipSuccess;
  const int grid = grid_for((n + NPT - 1) / NPT);
  hipLaunchKernelGGL((k_node_gather<NPT>), dim3(grid), dim3(kBlock), 0, s, nrows, ncomp, comp_stride, t_rowptr, t_offset, ev, v, overwrite);
  return hipGetLastError();
}

hipError_t launch_inverse_permutation(const int *index, long long n, int *perm, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_inverse_permutation, dim3(grid_for(n)), dim3(kBlock), 0, s, index, n, perm);
  return hipGetLastError();
}

hipError_t launch_layout_tiles(const GatherTiles &g, const int *index, int *slot, unsigned short *pos, hipStream_t s) {
  if (g.ntile <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_layout_tiles, dim3(g.ntile), dim3(256), 0, s, g, index, slot, pos);
  return hipGetLastError();
}

hipError_t launch_node_gather_tiles(const GatherTiles &g, int comp_stride, const double *ev, const float *ev32, double *v, bool overwrite,
                                    hipStream_t s) {
  if (g.ntile <= 0) return hipSuccess;
  const dim3 grid((g.ntile + 7) / 8 * 8);
  if (ev32)
    hipLaunchKernelGGL((k_node_gather_tiles<float>), grid, dim3(256), 0, s, g, comp_stride, ev32, v, overwrite);
  else
    hipLaunchKernelGGL((k_node_gather_tiles<double>), grid, dim3(256), 0, s, g, comp_stride, ev, v, overwrite);
  return hipGetLastError();
}

hipError_t launch_node_gather_blocks(int nrows, const int *t_rowptr, const int *t_index, const int *t_offset, const double *ev, double *v,
                                     bool overwrite, hipStream_t s) {
  const long long n = (long long)nrows * 5;
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_node_gather_blocks, dim3(grid_for(n)), dim3(kBlock), 0, s, nrows, t_rowptr, t_index, t_offset, ev, v, overwrite);
  return hipGetLastError();
}

hipError_t launch_fill(double *x, double value, long long n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill, dim3(grid_for(n)), dim3(kBlock), 0, s, x, value, n);
  return hipGetLastError();
}
hipError_t launch_axpby(double *y, double alpha, double beta, const double *x, long long n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_axpby, dim3(grid_for(n)), dim3(kBlock), 0, s, y, alpha, beta, x, n);
  return hipGetLastError();
}
hipError_t launch_scale(double *x, double alpha, long long n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_scale, dim3(grid_for(n)), dim3(kBlock), 0, s, x, alpha, n);
  return hipGetLastError();
}
hipError_t launch_pointwise_mult(double *w, const double *x, const double *y, long long n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_pmult, dim3(grid_for(n)), dim3(kBlock), 0, s, w, x, y, n);
  return hipGetLastError();
}
hipError_t launch_reciprocal(double *x, long long n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_recip, dim3(grid_for(n)), dim3(kBlock), 0, s, x, n);
  return hipGetLastError();
}
hipError_t launch_dot(const double *x, const double *y, long long n, double *d_partial, int npartial, hipStream_t s) {
  hipLaunchKernelGGL(k_dot, dim3(npartial), dim3(kBlock), 0, s, x, y, n, d_partial);
  return hipGetLastError();
}
hipError_t launch_norm(const double *x, long long n, int type, double *d_partial, int npartial, hipStream_t s) {
  hipLaunchKernelGGL(k_norm, dim3(npartial), dim3(kBlock), 0, s, x, n, type, d_partial);
  return hipGetLastError();
}
hipError_t launch_multiplicity(const int *offsets, long long n_offsets, int ncomp, int comp_stride, double *mult, hipStream_t s) {
  if (n_offsets <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_multiplicity, dim3(grid_for(n_offsets)), dim3(kBlock), 0, s, offsets, n_offsets, ncomp, comp_stride, mult);
  return hipGetLastError();
}
hipError_t launch_restriction_notranspose(const int *offsets, int nelem, int elemsize, int ncomp, int comp_stride, const double *u, double *e,
                                          hipStream_t s) {
  const long long n = (long long)nelem * elemsize;
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_rstr_n, dim3(grid_for(n)), dim3(kBlock), 0, s, offsets, nelem, elemsize, ncomp, comp_stride, u, e);
  return hipGetLastError();
}
hipError_t launch_restriction_transpose(const int *offsets, int nelem, int elemsize, int ncomp, int comp_stride, const double *e, double *u,
                                        hipStream_t s) {
  const long long n = (long long)nelem * elemsize;
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_rstr_t, dim3(grid_for(n)), dim3(kBlock), 0, s, offsets, nelem, elemsize, ncomp, comp_stride, e, u);
  return hipGetLastError();
}
