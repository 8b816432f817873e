// Vector kernels of the time integrator and its Krylov solvers (GMRES with point-Jacobi, Newton, explicit RK).
//
// Reductions are deterministic: a grid of fixed size (a function of the length only) reduces contiguous grid-stride
// slices per block in a fixed tree order into partials[slot][block] (slot-major, so that a consumer reads each slot's
// partials contiguously).  The kernel that needs a sum adds the at most 256 partials itself, every block alike and in the
// same order (2 KB per sum out of L2), which costs no launch between; a sum that only the host needs has a last kernel.  The
// same inputs give bitwise identical results from run to run.
//
// One Arnoldi step is three launches: the dots of w with all basis vectors, w -= sum_j h_j V_j with the partial sums of
// ||w||^2, and w /= ||w||, whose first block also stores (h_0..h_k, ||w||^2) into mapped host memory (Publish) for the
// step's single host read.
#include <hip/hip_runtime.h>

#include "krylov.hpp"

namespace {

constexpr int kThreads = 256, kRed = 512;  // threads of an elementwise kernel's block, of a reduction's

__device__ __forceinline__ double wave_sum(double v) {  // to all lanes
#pragma unroll
  for (int w = 32; w > 0; w >>= 1) v += __shfl_xor(v, w);
  return v;
}
// Sum over the block in thread 0; s holds a value per wave
__device__ __forceinline__ double block_sum(double v, double *s) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = v;
  __syncthreads();
  double r = 0;
  if (threadIdx.x == 0)
    for (int i = 0; i < (int)blockDim.x / 64; i++) r += s[i];
  return r;
}
// A slot's total, in every wave that asks alike
__device__ __forceinline__ double slot_total(const double *__restrict__ partial, int slot, int nb) {
  double x[kMaxReductionBlocks / 64];
#pragma unroll
  for (int i = 0; i < kMaxReductionBlocks / 64; i++) {
    const int b = i * 64 + (int)(threadIdx.x & 63);
    x[i]        = b < nb ? partial[(long long)slot * kMaxReductionBlocks + b] : 0.0;
  }
  double v = 0;
#pragma unroll
  for (int i = 0; i < kMaxReductionBlocks / 64; i++) v += x[i];
  return wave_sum(v);
}
// The 8 sums over the wave of a[0..7]: lane l returns that of a[l >> 3].  At each of the first three steps a lane keeps half of
// its sums and gives the others away: 10 exchanges instead of 48.
__device__ __forceinline__ double wave_sum8(const double (&a)[8]) {
  const bool b5 = threadIdx.x & 32, b4 = threadIdx.x & 16, b3 = threadIdx.x & 8;
  double     x[4], y[2];
#pragma unroll
  for (int j = 0; j < 4; j++) x[j] = (b5 ? a[j + 4] : a[j]) + __shfl_xor(b5 ? a[j] : a[j + 4], 32);
#pragma unroll
  for (int j = 0; j < 2; j++) y[j] = (b4 ? x[j + 2] : x[j]) + __shfl_xor(b4 ? x[j] : x[j + 2], 16);
  double z = (b3 ? y[1] : y[0]) + __shfl_xor(b3 ? y[0] : y[1], 8);
#pragma unroll
  for (int w = 4; w > 0; w >>= 1) z += __shfl_xor(z, w);
  return z;
}
// Store out[0 .. count) into mapped host memory, slot's value being r, then the sequence number; one block of >= count threads
__device__ __forceinline__ void publish(const Publish &pub, const double *out, int slot, double r) {
  const int i = threadIdx.x;
  if (i < pub.count) pub.h[i] = i == slot ? r : out[i];  // the other slots come from earlier launches
  __threadfence_system();  // each thread's value reaches host memory before the sequence number
  __syncthreads();
  if (i == 0) __hip_atomic_store(pub.flag, pub.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// acc[j] += w[i] V[j ldv + i] over the thread's slice, j < NJ: the loads of several entries in flight (a count of vectors that is
// known only at run time has every product wait for its own load)
template <int NJ>
__device__ __forceinline__ void dots(const double *__restrict__ w, const double *__restrict__ V, long long ldv, long long n, long long i0,
                                     long long stride, double (&acc)[8]) {
#pragma unroll(NJ <= 2 ? 4 : 2)
  for (long long i = i0; i < n; i += stride) {
    const double wi = w[i];
#pragma unroll
    for (int j = 0; j < NJ; j++) acc[j] += wi * V[(long long)j * ldv + i];
  }
}

// partial[j][block] = sum over this block's slice of w[i] V[j ldv + i], j < k, 8 vectors to a row of blocks (w is read once per
// row, 1/8 of the bytes, and the rows share the latency).
// Bound by the basis vectors' bytes (L2 and the memory-side cache hold those of a small problem).  Measured at 553 k entries: 6.1 us
// for 7 vectors, 11.2 us for 12 (in a GMRES solve with 10.5 on average 10.5 us); with a launch for every 8 vectors, a tree of barriers for every sum and a kernel that adds the
// partials, 15.3 and 27.7 us.  At 10.6 M entries 117 and 202 us (5.8 TB/s), with that 166 and 287 us, and 271 and 279 us where the
// vectors of a row that is not full were counted at run time.
__global__ void __launch_bounds__(kRed) k_mdot(const double *__restrict__ w, const double *__restrict__ V, long long ldv, int k, long long n,
                                               double *__restrict__ partial) {
  __shared__ double s[8][kRed / 64];
  const int         j0 = 8 * blockIdx.y, nj = k - j0 < 8 ? k - j0 : 8;
  const long long   stride = (long long)gridDim.x * kRed, i0 = (long long)blockIdx.x * kRed + threadIdx.x;
  double            acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  V += (long long)j0 * ldv;
  switch (nj) {
    case 1: dots<1>(w, V, ldv, n, i0, stride, acc); break;
    case 2: dots<2>(w, V, ldv, n, i0, stride, acc); break;
    case 3: dots<3>(w, V, ldv, n, i0, stride, acc); break;
    case 4: dots<4>(w, V, ldv, n, i0, stride, acc); break;
    case 5: dots<5>(w, V, ldv, n, i0, stride, acc); break;
    case 6: dots<6>(w, V, ldv, n, i0, stride, acc); break;
    case 7: dots<7>(w, V, ldv, n, i0, stride, acc); break;
    default: dots<8>(w, V, ldv, n, i0, stride, acc);
  }
  const double r = wave_sum8(acc);
  if ((threadIdx.x & 7) == 0) s[(threadIdx.x >> 3) % 8][threadIdx.x >> 6] = r;
  __syncthreads();
  if ((int)threadIdx.x < nj) {
    double t = 0;
#pragma unroll
    for (int i = 0; i < kRed / 64; i++) t += s[threadIdx.x][i];
    partial[(long long)(j0 + threadIdx.x) * kMaxReductionBlocks + blockIdx.x] = t;
  }
}

// partial[slot][block] = sum over this block's slice of x[i] y[i]
__global__ void __launch_bounds__(kRed) k_dot(const double *__restrict__ x, const double *__restrict__ y, long long n, int slot,
                                              double *__restrict__ partial) {
  __shared__ double s[kRed / 64];
  double            acc    = 0;
  const long long   stride = (long long)gridDim.x * kRed;
#pragma unroll 4
  for (long long i = (long long)blockIdx.x * kRed + threadIdx.x; i < n; i += stride) acc += x[i] * y[i];
  const double r = block_sum(acc, s);
  if (threadIdx.x == 0) partial[(long long)slot * kMaxReductionBlocks + blockIdx.x] = r;
}

// acc[u] + SIGN sum_{j < k} c[j] V[j ldv + i + u stride] in the order j = 0, 1, ..., the loads of 8 vectors in flight
template <int SIGN, int U>
__device__ __forceinline__ void basis_sum(double (&acc)[U], const double *c, const double *__restrict__ V, long long ldv, int k, long long i,
                                          long long stride) {
  int j = 0;
  for (; j + 8 <= k; j += 8) {
    double v[U][8];
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int l = 0; l < 8; l++) v[u][l] = V[(long long)(j + l) * ldv + i + u * stride];
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int l = 0; l < 8; l++) acc[u] += SIGN * c[j + l] * v[u][l];
  }
  double v[U][8];
#pragma unroll
  for (int u = 0; u < U; u++)
#pragma unroll
    for (int l = 0; l < 8; l++) v[u][l] = j + l < k ? V[(long long)(j + l) * ldv + i + u * stride] : 0.0;
#pragma unroll
  for (int u = 0; u < U; u++)
#pragma unroll
    for (int l = 0; l < 8; l++)
      if (j + l < k) acc[u] += SIGN * c[j + l] * v[u][l];
}

// out[j] = sum of partial[j][0 .. nb), j < k; w[i] -= sum_{j < k} out[j] V[j ldv + i] (in order j = 0, 1, ...);
// partial[slot][block] = sum of the new w[i]^2.  slot >= k: a block may overwrite no partials that another one still reads.
// Bound as k_mdot; measured in that solve 12.4 us and 5.9 us for k_normalize, 11.4 + 3.6 us with a kernel of 4.1 us between them.  A
// whole step (three launches against five) at 4.4 M entries, 7 vectors: 120 -> 95 us, 20 vectors: 350 -> 287 us.
__global__ void __launch_bounds__(kRed) k_project_out(double *__restrict__ w, const double *__restrict__ V, long long ldv, int k, long long n,
                                                      int slot, double *__restrict__ partial, int nb, double *__restrict__ out) {
  __shared__ double s[kRed / 64];
  __shared__ double c[kMaxDots];
  for (int j = threadIdx.x >> 6; j < k; j += kRed / 64) {
    const double h = slot_total(partial, j, nb);
    if ((threadIdx.x & 63) == 0) {
      c[j] = h;
      if (blockIdx.x == 0) out[j] = h;
    }
  }
  __syncthreads();
  double          ss     = 0;
  const long long stride = (long long)gridDim.x * kRed;
  long long       i      = (long long)blockIdx.x * kRed + threadIdx.x;
  for (; i + stride < n; i += 2 * stride) {
    double acc[2] = {w[i], w[i + stride]};
    basis_sum<-1>(acc, c, V, ldv, k, i, stride);
    w[i]          = acc[0];
    w[i + stride] = acc[1];
    ss += acc[0] * acc[0] + acc[1] * acc[1];
  }
  if (i < n) {
    double acc[1] = {w[i]};
    basis_sum<-1>(acc, c, V, ldv, k, i, stride);
    w[i] = acc[0];
    ss += acc[0] * acc[0];
  }
  const double r = block_sum(ss, s);
  if (threadIdx.x == 0) partial[(long long)slot * kMaxReductionBlocks + blockIdx.x] = r;
}

// out[slot] = sum over blocks b (in order) of partial[slot][b] (one wave); with pub.h set out[0 .. pub.count) is then published
__global__ void __launch_bounds__(64) k_reduce_partials(const double *__restrict__ partial, int nb, int slot, double *__restrict__ out, Publish pub) {
  const double r = slot_total(partial, slot, nb);
  if (threadIdx.x == 0) out[slot] = r;
  if (pub.h) publish(pub, out, slot, r);
}

// out[slot] = sum of partial[slot][0 .. nb), published with out[0 .. pub.count); y = y / sqrt(out[slot]) unless that is zero
// (a Krylov vector normalized by its squared norm)
constexpr int kNormalize = 4;  // entries a thread
__global__ void __launch_bounds__(kThreads) k_normalize(double *__restrict__ y, const double *__restrict__ partial, int nb, int slot,
                                                        double *__restrict__ out, long long n, Publish pub) {
  // the first entries are on their way while the partials come
  const long long stride = (long long)gridDim.x * kThreads, i0 = (long long)blockIdx.x * kThreads + threadIdx.x;
  double          x[kNormalize];
#pragma unroll
  for (int u = 0; u < kNormalize; u++) x[u] = i0 + u * stride < n ? y[i0 + u * stride] : 0.0;
  const double h = slot_total(partial, slot, nb);
  if (blockIdx.x == 0) {
    if (threadIdx.x == 0) out[slot] = h;
    if (pub.h) publish(pub, out, slot, h);
  }
  if (h == 0) return;
  const double a = 1.0 / sqrt(h);
#pragma unroll
  for (int u = 0; u < kNormalize; u++)
    if (i0 + u * stride < n) y[i0 + u * stride] = a * x[u];
  for (long long i = i0 + kNormalize * stride; i < n; i += stride) y[i] = a * y[i];
}

// y[i] = a y[i] + sum_{j < m} c_j X_j[i]
__global__ void __launch_bounds__(kThreads) k_lincomb(double *__restrict__ y, double a, LinComb lc, long long n) {
  const long long stride = (long long)gridDim.x * kThreads;
  for (long long i = (long long)blockIdx.x * kThreads + threadIdx.x; i < n; i += stride) {
    double acc = a == 0 ? 0.0 : a * y[i];
    for (int j = 0; j < lc.m; j++) acc += lc.c[j] * lc.x[j][i];
    y[i] = acc;
  }
}

// y[i] = a y[i] + sum_{j < k} c_j V[j ldv + i] with basis-vector coefficients
__global__ void __launch_bounds__(kThreads) k_basis_comb(double *__restrict__ y, const double *__restrict__ V, long long ldv, Coefs cf, long long n) {
  const long long stride = (long long)gridDim.x * kThreads;
  for (long long i = (long long)blockIdx.x * kThreads + threadIdx.x; i < n; i += stride) {
    double acc[1] = {y[i]};
    basis_sum<1>(acc, cf.c, V, ldv, cf.k, i, stride);
    y[i] = acc[0];
  }
}

// z[i] = d[i] (x[i] - y[i]) (y may be null: z = d x)
__global__ void __launch_bounds__(kThreads) k_dscale_diff(double *__restrict__ z, const double *__restrict__ d, const double *__restrict__ x,
                                                          const double *__restrict__ y, long long n) {
  const long long stride = (long long)gridDim.x * kThreads;
  for (long long i = (long long)blockIdx.x * kThreads + threadIdx.x; i < n; i += stride) z[i] = d[i] * (y ? x[i] - y[i] : x[i]);
}

// One Runge-Kutta stage behind its right-hand side: k = d r is the stage derivative, y = q + sum_{j < m} c_j K_j + ck k the
// next stage's state.  LAST: y is the step's result and the non-finite entries of y are counted (partial as k_dot).
// Bound by its bytes: a vector read for each of d, r, q, K_j, one written for k (unless it is not needed again) and for y.
// Measured at 10.6 M entries, SSP33: 79 us a stage (5.9 TB/s) and 96 us the last (5.3 TB/s); as a mass solve, a combination or
// copy and a count 91 us and 111 us.
// The count needs one partial per block, so the last stage has 256 large blocks whose threads keep 4 entries in flight: 8 waves
// a CU with 2 entries a thread reached 3.5 TB/s.
template <bool LAST>
constexpr int kRkThreads = LAST ? 1024 : kThreads;
template <bool LAST>
__global__ void __launch_bounds__(kRkThreads<LAST>) k_rk_stage(RkStage a, long long n, int slot, double *__restrict__ partial) {
  constexpr int   NT = kRkThreads<LAST>, U = LAST ? 4 : 1;
  const long long stride = (long long)gridDim.x * NT;
  double          cnt    = 0;
  for (long long i0 = (long long)blockIdx.x * NT + threadIdx.x; i0 < n; i0 += U * stride) {
    double k[U], y[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const long long i = i0 + u * stride < n ? i0 + u * stride : i0;
      k[u]              = a.d[i] * a.r[i];
      y[u]              = a.q[i];
    }
    for (int j = 0; j < a.lc.m; j++)
#pragma unroll
      for (int u = 0; u < U; u++) y[u] += a.lc.c[j] * a.lc.x[j][i0 + u * stride < n ? i0 + u * stride : i0];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const long long i = i0 + u * stride;
      if (i >= n) break;
      if (a.ck != 0) y[u] += a.ck * k[u];
      if (a.k) a.k[i] = k[u];
      a.y[i] = y[u];
      if constexpr (LAST) cnt += isfinite(y[u]) ? 0.0 : 1.0;
    }
  }
  if constexpr (LAST) {
    __shared__ double s[NT / 64];
    const double      r = block_sum(cnt, s);
    if (threadIdx.x == 0) partial[(long long)slot * kMaxReductionBlocks + blockIdx.x] = r;
  }
}

// d[i] = 1 / d[i], with 1 where d[i] == 0 (PCJACOBI's zero-diagonal rule)
__global__ void __launch_bounds__(kThreads) k_jacobi_invert(double *__restrict__ d, long long n) {
  const long long stride = (long long)gridDim.x * kThreads;
  for (long long i = (long long)blockIdx.x * kThreads + threadIdx.x; i < n; i += stride) d[i] = d[i] != 0 ? 1.0 / d[i] : 1.0;
}

__global__ void __launch_bounds__(kThreads) k_set(double *__restrict__ x, double v, long long n) {
  const long long stride = (long long)gridDim.x * kThreads;
  for (long long i = (long long)blockIdx.x * kThreads + threadIdx.x; i < n; i += stride) x[i] = v;
}

// partial[slot][block] = number of non-finite entries in the block's slice (as a double)
__global__ void __launch_bounds__(kRed) k_count_nonfinite(const double *__restrict__ x, long long n, int slot, double *__restrict__ partial) {
  __shared__ double s[kRed / 64];
  double            cnt    = 0;
  const long long   stride = (long long)gridDim.x * kRed;
#pragma unroll 4
  for (long long i = (long long)blockIdx.x * kRed + threadIdx.x; i < n; i += stride) cnt += isfinite(x[i]) ? 0.0 : 1.0;
  const double r = block_sum(cnt, s);
  if (threadIdx.x == 0) partial[(long long)slot * kMaxReductionBlocks + blockIdx.x] = r;
}

// In-place inverse of each node's 5x5 block (row-major [c_out][c_in]) by Gauss-Jordan elimination with partial
// pivoting on [A | I]; every index is a compile-time constant so the blocks stay in registers.
// partial[slot][block] counts the singular blocks of the block's slice.
__global__ void __launch_bounds__(kThreads) k_pb_invert(double *__restrict__ pb, long long nn, int slot, double *__restrict__ partial) {
  __shared__ double s[kThreads / 64];
  double            bad    = 0;
  const long long   stride = (long long)gridDim.x * kThreads;
  for (long long node = (long long)blockIdx.x * kThreads + threadIdx.x; node < nn; node += stride) {
    double A[5][5], X[5][5];
#pragma unroll
    for (int i = 0; i < 5; i++)
#pragma unroll
      for (int j = 0; j < 5; j++) {
        A[i][j] = pb[node * 25 + i * 5 + j];
        X[i][j] = i == j ? 1.0 : 0.0;
      }
    bool singular = false;
#pragma unroll
    for (int k = 0; k < 5; k++) {
      int    piv  = k;
      double best = fabs(A[k][k]);
#pragma unroll
      for (int i = k + 1; i < 5; i++)
        if (fabs(A[i][k]) > best) {
          best = fabs(A[i][k]);
          piv  = i;
        }
#pragma unroll
      for (int i = k + 1; i < 5; i++)
        if (i == piv)
#pragma unroll
          for (int j = 0; j < 5; j++) {
            double ta = A[k][j], tx = X[k][j];
            A[k][j] = A[i][j], X[k][j] = X[i][j];
            A[i][j] = ta, X[i][j] = tx;
          }
      if (A[k][k] == 0) singular = true;
      const double inv = A[k][k] != 0 ? 1.0 / A[k][k] : 0.0;
#pragma unroll
      for (int j = 0; j < 5; j++) {
        A[k][j] *= inv;
        X[k][j] *= inv;
      }
#pragma unroll
      for (int i = 0; i < 5; i++) {
        if (i == k) continue;
        const double f = A[i][k];
#pragma unroll
        for (int j = 0; j < 5; j++) {
          A[i][j] -= f * A[k][j];
          X[i][j] -= f * X[k][j];
        }
      }
    }
    if (singular) bad += 1.0;
#pragma unroll
    for (int i = 0; i < 5; i++)
#pragma unroll
      for (int j = 0; j < 5; j++) pb[node * 25 + i * 5 + j] = X[i][j];
  }
  const double r = block_sum(bad, s);
  if (threadIdx.x == 0) partial[(long long)slot * kMaxReductionBlocks + blockIdx.x] = r;
}

// z_n = Binv_n (x_n - y_n) per node n (y may be null)
__global__ void __launch_bounds__(kThreads) k_pb_apply(double *__restrict__ z, const double *__restrict__ pbinv, const double *__restrict__ x,
                                                       const double *__restrict__ y, long long nn) {
  const long long stride = (long long)gridDim.x * kThreads;
  for (long long node = (long long)blockIdx.x * kThreads + threadIdx.x; node < nn; node += stride) {
    double r[5];
#pragma unroll
    for (int j = 0; j < 5; j++) r[j] = y ? x[node * 5 + j] - y[node * 5 + j] : x[node * 5 + j];
#pragma unroll
    for (int i = 0; i < 5; i++) {
      double acc = 0;
#pragma unroll
      for (int j = 0; j < 5; j++) acc += pbinv[node * 25 + i * 5 + j] * r[j];
      z[node * 5 + i] = acc;
    }
  }
}

int elementwise_grid(long long n) {
  long long g = (n + kThreads - 1) / kThreads;
  if (g > 4096) g = 4096;
  return g < 1 ? 1 : (int)g;
}

}  // namespace

static int krylov_reduction_blocks(long long n, int threads) {
  long long g = (n + threads - 1) / threads;
  if (g > kMaxReductionBlocks) g = kMaxReductionBlocks;
  return g < 1 ? 1 : (int)g;
}
int krylov_reduction_blocks(long long n) { return krylov_reduction_blocks(n, kRed); }

hipError_t launch_mdot(const double *w, const double *V, long long ldv, int k, long long n, double *partial, hipStream_t s) {
  if (k < 1 || k > kMaxDots) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_mdot, dim3(krylov_reduction_blocks(n), (k + 7) / 8), dim3(kRed), 0, s, w, V, ldv, k, n, partial);
  return hipGetLastError();
}

hipError_t launch_dot_partial(const double *x, const double *y, long long n, int slot, double *partial, hipStream_t s) {
  if (slot < 0 || slot >= kMaxDots) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_dot, dim3(krylov_reduction_blocks(n)), dim3(kRed), 0, s, x, y, n, slot, partial);
  return hipGetLastError();
}

hipError_t launch_dot(const double *x, const double *y, long long n, int slot, double *partial, double *out, hipStream_t s, const Publish &pub) {
  if (slot < 0 || slot >= kMaxDots || pub.count > 64) return hipErrorInvalidValue;
  const int nb = krylov_reduction_blocks(n);
  hipLaunchKernelGGL(k_dot, dim3(nb), dim3(kRed), 0, s, x, y, n, slot, partial);
  hipLaunchKernelGGL(k_reduce_partials, dim3(1), dim3(64), 0, s, partial, nb, slot, out, pub);
  return hipGetLastError();
}

hipError_t launch_project_out(double *w, const double *V, long long ldv, int k, long long n, int slot, double *partial, double *out, hipStream_t s) {
  if (k < 0 || k > kMaxDots || slot < k || slot >= kMaxDots) return hipErrorInvalidValue;
  const int nb = krylov_reduction_blocks(n);
  hipLaunchKernelGGL(k_project_out, dim3(nb), dim3(kRed), 0, s, w, V, ldv, k, n, slot, partial, nb, out);
  return hipGetLastError();
}

hipError_t launch_normalize(double *y, const double *partial, int slot, double *out, long long n, hipStream_t s, const Publish &pub) {
  if (slot < 0 || slot >= kMaxDots || pub.count > kThreads) return hipErrorInvalidValue;
  const int grid = elementwise_grid((n + kNormalize - 1) / kNormalize);
  hipLaunchKernelGGL(k_normalize, dim3(grid), dim3(kThreads), 0, s, y, partial, krylov_reduction_blocks(n), slot, out, n, pub);
  return hipGetLastError();
}

hipError_t launch_lincomb(double *y, double a, const LinComb &lc, long long n, hipStream_t s) {
  if (lc.m < 0 || lc.m > kMaxLinComb) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_lincomb, dim3(elementwise_grid(n)), dim3(kThreads), 0, s, y, a, lc, n);
  return hipGetLastError();
}

hipError_t launch_basis_comb(double *y, const double *V, long long ldv, const Coefs &cf, long long n, hipStream_t s) {
  if (cf.k < 0 || cf.k > kMaxDots) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_basis_comb, dim3(elementwise_grid(n)), dim3(kThreads), 0, s, y, V, ldv, cf, n);
  return hipGetLastError();
}

hipError_t launch_dscale_diff(double *z, const double *d, const double *x, const double *y, long long n, hipStream_t s) {
  hipLaunchKernelGGL(k_dscale_diff, dim3(elementwise_grid(n)), dim3(kThreads), 0, s, z, d, x, y, n);
  return hipGetLastError();
}

hipError_t launch_rk_stage(const RkStage &a, long long n, hipStream_t s) {
  if (a.lc.m < 0 || a.lc.m > kMaxLinComb) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_rk_stage<false>, dim3(elementwise_grid(n)), dim3(kThreads), 0, s, a, n, 0, nullptr);
  return hipGetLastError();
}

hipError_t launch_rk_last(const RkStage &a, long long n, int slot, double *partial, double *out, hipStream_t s, const Publish &pub) {
  if (a.lc.m < 0 || a.lc.m > kMaxLinComb || slot < 0 || slot >= kMaxDots || pub.count > 64) return hipErrorInvalidValue;
  const int nb = krylov_reduction_blocks(n);
  hipLaunchKernelGGL(k_rk_stage<true>, dim3(nb), dim3(kRkThreads<true>), 0, s, a, n, slot, partial);
  hipLaunchKernelGGL(k_reduce_partials, dim3(1), dim3(64), 0, s, partial, nb, slot, out, pub);
  return hipGetLastError();
}

hipError_t launch_jacobi_invert(double *d, long long n, hipStream_t s) {
  hipLaunchKernelGGL(k_jacobi_invert, dim3(elementwise_grid(n)), dim3(kThreads), 0, s, d, n);
  return hipGetLastError();
}

hipError_t launch_set(double *x, double v, long long n, hipStream_t s) {
  hipLaunchKernelGGL(k_set, dim3(elementwise_grid(n)), dim3(kThreads), 0, s, x, v, n);
  return hipGetLastError();
}

hipError_t launch_count_nonfinite(const double *x, long long n, int slot, double *partial, double *out, hipStream_t s, const Publish &pub) {
  if (slot < 0 || slot >= kMaxDots || pub.count > 64) return hipErrorInvalidValue;
  const int nb = krylov_reduction_blocks(n);
  hipLaunchKernelGGL(k_count_nonfinite, dim3(nb), dim3(kRed), 0, s, x, n, slot, partial);
  hipLaunchKernelGGL(k_reduce_partials, dim3(1), dim3(64), 0, s, partial, nb, slot, out, pub);
  return hipGetLastError();
}

hipError_t launch_pb_invert(double *pb, long long nnodes, int slot, double *partial, double *out, hipStream_t s, const Publish &pub) {
  if (slot < 0 || slot >= kMaxDots || pub.count > 64) return hipErrorInvalidValue;
  const int nb = krylov_reduction_blocks(nnodes, kThreads);  // a node a thread as long as the grid allows it
  hipLaunchKernelGGL(k_pb_invert, dim3(nb), dim3(kThreads), 0, s, pb, nnodes, slot, partial);
  hipLaunchKernelGGL(k_reduce_partials, dim3(1), dim3(64), 0, s, partial, nb, slot, out, pub);
  return hipGetLastError();
}

hipError_t launch_pb_apply(double *z, const double *pbinv, const double *x, const double *y, long long nnodes, hipStream_t s) {
  hipLaunchKernelGGL(k_pb_apply, dim3(elementwise_grid(nnodes)), dim3(kThreads), 0, s, z, pbinv, x, y, nnodes);
  return hipGetLastError();
}
