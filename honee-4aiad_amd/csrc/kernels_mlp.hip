// FP32 training kernels of the subgrid-stress MLP (leaky ReLU), the network that the fused FP64 closure evaluates
// (qfunctions/sgs_dd_model.h:37-53): y = W2 lrelu(W1 x + b1) + b2 (the reference's one hidden layer) or, with a second
// hidden layer, y = W3 lrelu(W2 lrelu(W1 x + b1) + b2) + b3; loss = mean over samples and outputs of (y - t)^2.
//
// k_mlp_grad runs the forward pass, the backward pass and the parameter gradients on the FP32 matrix cores, 16 samples per
// wave at a time; k_mlp_reduce_adam sums the per-block partials in a fixed order and applies Adam, so the result does not
// depend on scheduling.
// Parameter layout (floats): see MlpDims.  The layer sizes are compile-time constants (6-20-6 and 6-20-20-6).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels_mlp.hpp"
#include "ns_physics.hpp"
#include "sgs_ops.hpp"

namespace {

constexpr int kTpb = 256;
constexpr int kWaves = kTpb / 64, kGroup = 16;  // k_mlp_grad: waves per block, samples per wave and step
constexpr int kGradBlocks = 512;                // most blocks of k_mlp_grad (two per CU), and so rows of partials

using f32x4 = __attribute__((ext_vector_type(4))) float;
__device__ __forceinline__ f32x4 mfma16(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// Batch gradient of the network with NL hidden layers.  v_mfma_f32_16x16x4: lane l holds A[l & 15][l >> 4],
// B[l >> 4][l & 15] and, in register r, D[4 (l >> 4) + r][l & 15].
//
// Forward and backward: the 16 columns are the wave's samples, the rows neurons.  A hidden layer takes two row tiles:
// neurons 0..15, and neurons 16..19 in the rows 4 g (register 0 of every lane), so a layer's 20 activations are five
// registers per lane that are the next product's B operands as they are; the weights are loaded in the matching order
// once per wave and stay in registers.  The outputs sit in the rows 4 g (0..3) and 4 g + 1 (4, 5).
// Gradients: sums over the samples of products of two activations or errors, so both go through the wave's LDS rows
// [sample][column] and come back with the sample as the contracted index; a column of ones beside each activation gives
// the bias gradients.  The tiles accumulate in registers over all of the wave's steps; the block adds its waves in order.
//
// One batch is bound by the latency of its chain of products and loads, not by arithmetic (17 MFLOP at 4096 samples), so
// it is spread over as many waves as there are groups of 16.  Measured at 4096 samples, 6-20-20-6: 38.8 -> 7.7 us against
// one thread per sample with the gradients as LDS dot products (32 blocks, whose columns all lay in one bank).
template <int NL>
__global__ void __launch_bounds__(kTpb) k_mlp_grad(float alpha, const float *__restrict__ theta, const float *__restrict__ X, const float *__restrict__ T,
                                                   const int *__restrict__ idx, int first, int count, float inv_norm, float *__restrict__ partial) {
  constexpr int NI = 6, NH = 20, NO = 6;
  constexpr int oB1 = NH * NI, oW2 = oB1 + NH, oB2 = oW2 + NH * NH, oWo = NL == 2 ? oB2 + NH : oW2, oBo = oWo + NO * NH, np = oBo + NO;
  // columns of a sample's LDS row: inputs and a one, activations and a one, errors
  constexpr int cX = 0, cA1 = cX + NI + 1, cA2 = cA1 + NH + 1, cD1 = NL == 2 ? cA2 + NH + 1 : cA2, cD2 = cD1 + NH, cDY = NL == 2 ? cD2 + NH : cD2;
  constexpr int kRow = (cDY + NO) | 1;            // odd: the rows of one column lie in different banks
  constexpr int kRows = kGroup * kRow + kGroup;   // an operand tile of the last row reads up to 16 columns past it
  static_assert((NL == 2 ? cD2 : cD1) + 31 < kRow + kGroup && cDY + 15 < kRow + kGroup, "operand tiles stay within the wave's rows");
  static_assert(np + 1 <= kRows, "the wave's gradient fits its rows");
  __shared__ float sm[kWaves][kRows];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;
  float    *row = &sm[wave][c * kRow];

  // neuron of tile t's row i, of contraction step s at this lane's g; output of row i
  auto hrow = [&](int t) { return t == 0 ? c : (c % 4 == 0 ? 16 + c / 4 : -1); };
  auto hk   = [&](int s) { return s < 4 ? 4 * g + s : 16 + g; };
  const int oi = c % 4 == 0 ? c / 4 : (c % 4 == 1 && c / 4 < NO - 4 ? 4 + c / 4 : -1);
  float     w1[2][2], w2[NL == 2 ? 2 : 1][5], w2t[NL == 2 ? 2 : 1][5], wo[5], wot[2][2];
#pragma unroll
  for (int t = 0; t < 2; t++) {
    const int i = hrow(t);
#pragma unroll
    for (int s = 0; s < 2; s++) {
      const int k = 4 * s + g;  // input and output index alike (NI = NO)
      w1[t][s]    = i >= 0 && k < NI ? theta[i * NI + k] : 0.f;
      wot[t][s]   = i >= 0 && k < NO ? theta[oWo + k * NH + i] : 0.f;
    }
    if constexpr (NL == 2)
#pragma unroll
      for (int s = 0; s < 5; s++) {
        w2[t][s]  = i >= 0 ? theta[oW2 + i * NH + hk(s)] : 0.f;
        w2t[t][s] = i >= 0 ? theta[oW2 + hk(s) * NH + i] : 0.f;
      }
  }
#pragma unroll
  for (int s = 0; s < 5; s++) wo[s] = oi >= 0 ? theta[oWo + oi * NH + hk(s)] : 0.f;
  // biases in the products' accumulators: rows 4 g + r, and 4 g of the second tile
  auto bias_tiles = [&](int at, f32x4 &b0, f32x4 &b1) {
#pragma unroll
    for (int r = 0; r < 4; r++) b0[r] = theta[at + 4 * g + r];
    b1 = f32x4{theta[at + 16 + g], 0.f, 0.f, 0.f};
  };
  f32x4 bh[NL][2];
  bias_tiles(oB1, bh[0][0], bh[0][1]);
  if constexpr (NL == 2) bias_tiles(oB2, bh[NL - 1][0], bh[NL - 1][1]);
  const f32x4 bo = {theta[oBo + g], g < NO - 4 ? theta[oBo + 4 + g] : 0.f, 0.f, 0.f};
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};

  f32x4 G1[2] = {zero, zero}, G2[2][2] = {{zero, zero}, {zero, zero}}, Go[2] = {zero, zero};
  float loss = 0;
  for (long long s0 = (blockIdx.x * kWaves + wave) * kGroup; s0 < count; s0 += gridDim.x * kWaves * kGroup) {
    const long long s = s0 + c;
    const bool ok  = s < count;
    const int  smp = ok ? (idx ? idx[first + s] : (int)(first + s)) : 0;
    const float *xs = X + (long long)smp * NI, *ts = T + (long long)smp * NO;
    const float  x0 = ok ? xs[g] : 0.f, x1 = ok && g < 2 ? xs[4 + g] : 0.f;
    const float  t0 = ok ? ts[g] : 0.f, t1 = ok && g < 2 ? ts[4 + g] : 0.f;

    // forward: a[l] activations, m[l] the slopes alpha or 1
    float a[NL][5], m[NL][5];
    auto  hidden = [&](int l, const f32x4 &d0, const f32x4 &d1) {
#pragma unroll
      for (int r = 0; r < 5; r++) {
        const float h = r < 4 ? d0[r] : d1[0];
        m[l][r]       = h < 0 ? alpha : 1.f;
        a[l][r]       = m[l][r] * h;
      }
    };
    {
      f32x4 d[2];
#pragma unroll
      for (int t = 0; t < 2; t++) d[t] = mfma16(w1[t][1], x1, mfma16(w1[t][0], x0, bh[0][t]));
      hidden(0, d[0], d[1]);
    }
    if constexpr (NL == 2) {
      f32x4 d[2] = {bh[NL - 1][0], bh[NL - 1][1]};
#pragma unroll
      for (int k = 0; k < 5; k++)
#pragma unroll
        for (int t = 0; t < 2; t++) d[t] = mfma16(w2[t][k], a[0][k], d[t]);
      hidden(NL - 1, d[0], d[1]);
    }
    f32x4 y = bo;
#pragma unroll
    for (int k = 0; k < 5; k++) y = mfma16(wo[k], a[NL - 1][k], y);
    const float e0 = ok ? y[0] - t0 : 0.f, e1 = ok && g < NO - 4 ? y[1] - t1 : 0.f;
    loss += e0 * e0 + e1 * e1;
    const float dy0 = 2.f * e0 * inv_norm, dy1 = 2.f * e1 * inv_norm;

    // backward: e[l] errors of the hidden layers
    float e[NL][5];
    auto  error = [&](int l, const f32x4 &d0, const f32x4 &d1) {
#pragma unroll
      for (int r = 0; r < 5; r++) e[l][r] = (r < 4 ? d0[r] : d1[0]) * m[l][r];
    };
    {
      f32x4 d[2];
#pragma unroll
      for (int t = 0; t < 2; t++) d[t] = mfma16(wot[t][1], dy1, mfma16(wot[t][0], dy0, zero));
      error(NL - 1, d[0], d[1]);
    }
    if constexpr (NL == 2) {
      f32x4 d[2] = {zero, zero};
#pragma unroll
      for (int k = 0; k < 5; k++)
#pragma unroll
        for (int t = 0; t < 2; t++) d[t] = mfma16(w2t[t][k], e[NL - 1][k], d[t]);
      error(0, d[0], d[1]);
    }

    // the sample's LDS row; each wave writes and reads only its own rows
    row[cX + g] = x0;
    if (g < 2) row[cX + 4 + g] = x1;
    if (g == 2) row[cX + NI] = row[cA1 + NH] = 1.f;
    if (NL == 2 && g == 3) row[cA2 + NH] = 1.f;
#pragma unroll
    for (int r = 0; r < 5; r++) {
      row[cA1 + hk(r)] = a[0][r];
      row[cD1 + hk(r)] = e[0][r];
      if constexpr (NL == 2) {
        row[cA2 + hk(r)] = a[NL - 1][r];
        row[cD2 + hk(r)] = e[NL - 1][r];
      }
    }
    row[cDY + g] = dy0;
    if (g < NO - 4) row[cDY + 4 + g] = dy1;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // operand tiles: row or column index c, sample 4 k + g.  Columns past an array belong to unused rows and columns of
    // the results.
    constexpr int cAo = NL == 2 ? cA2 : cA1;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const float *q  = &sm[wave][(4 * k + g) * kRow];
      const float  xk = q[cX + c], dk = q[cDY + c];
      G1[0] = mfma16(q[cD1 + c], xk, G1[0]);
      G1[1] = mfma16(q[cD1 + 16 + c], xk, G1[1]);
      if constexpr (NL == 2) {
#pragma unroll
        for (int i = 0; i < 2; i++) {
          const float d2 = q[cD2 + 16 * i + c];
          G2[i][0]       = mfma16(d2, q[cA1 + c], G2[i][0]);
          G2[i][1]       = mfma16(d2, q[cA1 + 16 + c], G2[i][1]);
        }
      }
      Go[0] = mfma16(dk, q[cAo + c], Go[0]);
      Go[1] = mfma16(dk, q[cAo + 16 + c], Go[1]);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();  // the rows are read before the next step overwrites them
  }

  // the wave's gradient (parameter order), then the block's sum over its waves in order
  __syncthreads();
  float *gw = sm[wave];
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int i = 4 * g + r;
#pragma unroll
    for (int t = 0; t < 2; t++) {
      const int n = 16 * t + i;
      if (n < NH) {
        if (c < NI) gw[n * NI + c] = G1[t][r];
        else if (c == NI) gw[oB1 + n] = G1[t][r];
        if constexpr (NL == 2)
#pragma unroll
          for (int u = 0; u < 2; u++) {
            const int k = 16 * u + c;
            if (k < NH) gw[oW2 + n * NH + k] = G2[t][u][r];
            else if (k == NH) gw[oB2 + n] = G2[t][u][r];
          }
      }
      const int k = 16 * t + c;
      if (i < NO) {
        if (k < NH) gw[oWo + i * NH + k] = Go[t][r];
        else if (k == NH) gw[oBo + i] = Go[t][r];
      }
    }
  }
#pragma unroll
  for (int w = 32; w > 0; w >>= 1) loss += __shfl_down(loss, w);
  if (lane == 0) gw[np] = loss * inv_norm;
  __syncthreads();
  for (int p = threadIdx.x; p <= np; p += kTpb) {
    float acc = 0;
#pragma unroll
    for (int w = 0; w < kWaves; w++) acc += sm[w][p];
    partial[(long long)blockIdx.x * (np + 1) + p] = acc;
  }
}

template <int NI, int NH, int NH2, int NO>
__global__ void k_mlp2_predict(float alpha, const float *__restrict__ theta, const float *__restrict__ X, int n, float *__restrict__ Y) {
  constexpr int    np = NH * NI + NH + NH2 * NH + NH2 + NO * NH2 + NO;
  constexpr int    o1 = NH * NI, o2 = o1 + NH, o3 = o2 + NH2 * NH, o4 = o3 + NH2, o5 = o4 + NO * NH2;
  __shared__ float sP[np];
  for (int i = threadIdx.x; i < np; i += blockDim.x) sP[i] = theta[i];
  __syncthreads();
  const float *W1 = sP, *b1 = sP + o1, *W2 = sP + o2, *b2 = sP + o3, *W3 = sP + o4, *b3 = sP + o5;
  const int    s  = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  float x[NI], a1[NH], a2[NH2];
  for (int i = 0; i < NI; i++) x[i] = X[(long long)s * NI + i];
  for (int j = 0; j < NH; j++) {
    float acc = b1[j];
    for (int i = 0; i < NI; i++) acc += W1[j * NI + i] * x[i];
    a1[j] = acc < 0 ? alpha * acc : acc;
  }
  for (int k = 0; k < NH2; k++) {
    float acc = b2[k];
    for (int j = 0; j < NH; j++) acc += W2[k * NH + j] * a1[j];
    a2[k] = acc < 0 ? alpha * acc : acc;
  }
  for (int o = 0; o < NO; o++) {
    float acc = b3[o];
    for (int k = 0; k < NH2; k++) acc += W3[o * NH2 + k] * a2[k];
    Y[(long long)s * NO + o] = acc;
  }
}

// Sum of the block partials (row b: np gradient entries and the loss) in a fixed order: a thread sums every kSlices-th
// row of one column, then the slices are added in order.  Adam (bias-corrected moments) when apply is set, else the
// gradient only.  One block per 32 columns, whose rows are read as 128 contiguous bytes: bound by the latency of one
// load round and the launch.  Measured at 64 rows of 687: 17.4 -> 4.5 us against one block with a serial sum per column.
constexpr int kSlices = 8;

__global__ void __launch_bounds__(32 * kSlices) k_mlp_reduce_adam(int np, int nblocks, const float *__restrict__ partial, float *__restrict__ grad,
                                                                  float *__restrict__ loss, float *theta, float *m, float *v, MlpAdam adam, int apply) {
  __shared__ float s[kSlices][32];
  const int        col = threadIdx.x & 31, slice = threadIdx.x >> 5, p = blockIdx.x * 32 + col;
  float            acc = 0;
  if (p <= np)
#pragma unroll 4
    for (int b = slice; b < nblocks; b += kSlices) acc += partial[(long long)b * (np + 1) + p];
  s[slice][col] = acc;
  __syncthreads();
  if (slice > 0 || p > np) return;
  float g = 0;
#pragma unroll
  for (int i = 0; i < kSlices; i++) g += s[i][col];
  if (p == np) {
    *loss = g;
    return;
  }
  grad[p] = g;
  if (apply) {
    const float mp = adam.beta1 * m[p] + (1.f - adam.beta1) * g;
    const float vp = adam.beta2 * v[p] + (1.f - adam.beta2) * g * g;
    m[p]           = mp;
    v[p]           = vp;
    const float mh = mp / adam.bc1, vh = vp / adam.bc2;
    theta[p] -= adam.lr * mh / (sqrtf(vh) + adam.eps);
  }
}

template <int NI, int NH, int NO>
__global__ void k_mlp_predict(float alpha, const float *__restrict__ theta, const float *__restrict__ X, int n, float *__restrict__ Y) {
  constexpr int    ni = NI, nh = NH, no = NO, np = NH * NI + NH + NO * NH + NO;
  __shared__ float sP[np];
  const MlpDims    d{NI, NH, NO, alpha};
  for (int i = threadIdx.x; i < np; i += blockDim.x) sP[i] = theta[i];
  __syncthreads();
  const float *W1 = sP, *b1 = sP + nh * ni, *W2 = b1 + nh, *b2 = W2 + no * nh;
  const int    s  = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  float x[NI], a[NH];
  for (int i = 0; i < ni; i++) x[i] = X[(long long)s * ni + i];
  for (int j = 0; j < nh; j++) {
    float acc = b1[j];
    for (int i = 0; i < ni; i++) acc += W1[j * ni + i] * x[i];
    a[j] = acc < 0 ? d.alpha * acc : acc;
  }
  for (int k = 0; k < no; k++) {
    float acc = b2[k];
    for (int j = 0; j < nh; j++) acc += W2[k * nh + j] * a[j];
    Y[(long long)s * no + k] = acc;
  }
}

// Model-space samples from the nodal training fields: the closure inputs of the filtered state (ComputeSgsDDInputs,
// qfunctions/sgs_dd_utils.h:58-90) and the filtered SGS stress tau rotated into the input's eigenframe and scaled as
// ComputeSgsDDOutputs undoes it (qfunctions/sgs_dd_utils.h:92-127): S = E tau E^T / (delta^2 |grad u|^2), stored in
// the model's output order S00 S11 S22 S01 S02 S12.
__global__ void k_sgs_model_samples(long long n, const double *__restrict__ train, const double *__restrict__ filtered, const double *__restrict__ G,
                                    const double *__restrict__ A, CeedMiGas gas, float *__restrict__ X, double *__restrict__ S) {
  const auto g = ns::Gas<double>::from(gas);
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const double        *yf = filtered + i * 11;
    double               yi[5], gu[3][3], kmA[6], E[3][3], in[6], gmag;
#pragma unroll
    for (int c = 0; c < 5; c++) yi[c] = yf[c];
#pragma unroll
    for (int j = 0; j < 3; j++)
#pragma unroll
      for (int k = 0; k < 3; k++) gu[j][k] = G[i * 9 + j * 3 + k];
#pragma unroll
    for (int c = 0; c < 6; c++) kmA[c] = A[i * 7 + c];
    const double         delta = A[i * 7 + 6];
    const ns::St<double> s     = ns::state_from_q<ns::VAR_PRIM>(g, yi);
    sgs::sgs_inputs(gu, kmA, delta, g.mu / s.U[0], E, in, gmag);
    const double *t       = train + i * 12 + 6;  // XX YY ZZ YZ XZ XY
    const double  tau[3][3] = {{t[0], t[5], t[4]}, {t[5], t[1], t[3]}, {t[4], t[3], t[2]}};
    double        Et[3][3], R[3][3];
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int b = 0; b < 3; b++) Et[a][b] = E[a][0] * tau[0][b] + E[a][1] * tau[1][b] + E[a][2] * tau[2][b];
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int b = 0; b < 3; b++) R[a][b] = Et[a][0] * E[b][0] + Et[a][1] * E[b][1] + Et[a][2] * E[b][2];
    const double sc = 1.0 / (delta * delta * (gmag * gmag));
#pragma unroll
    for (int c = 0; c < 6; c++) X[i * 6 + c] = (float)in[c];
    double *o = S + i * 6;
    o[0]      = R[0][0] * sc;
    o[1]      = R[1][1] * sc;
    o[2]      = R[2][2] * sc;
    o[3]      = R[0][1] * sc;
    o[4]      = R[0][2] * sc;
    o[5]      = R[1][2] * sc;
  }
}

}  // namespace

// 6-20-6 (the reference's closure) and 6-20-20-6
bool mlp_dims_supported(const MlpDims &d) { return d.ni == 6 && d.nh == 20 && d.no == 6 && (d.nh2 == 0 || d.nh2 == 20); }

int mlp_grad_blocks(int count) {
  const int per = kWaves * kGroup;
  return std::min((count + per - 1) / per, kGradBlocks);
}

hipError_t launch_mlp_grad(const MlpDims &d, const float *theta, const float *X, const float *T, const int *idx, int first, int count, float inv_norm,
                           float *partial, hipStream_t s) {
  if (!mlp_dims_supported(d)) return hipErrorInvalidValue;
  const int nb = mlp_grad_blocks(count);
  if (nb <= 0) return hipSuccess;
  if (d.nh2 > 0) hipLaunchKernelGGL(k_mlp_grad<2>, dim3(nb), dim3(kTpb), 0, s, d.alpha, theta, X, T, idx, first, count, inv_norm, partial);
  else hipLaunchKernelGGL(k_mlp_grad<1>, dim3(nb), dim3(kTpb), 0, s, d.alpha, theta, X, T, idx, first, count, inv_norm, partial);
  return hipGetLastError();
}

hipError_t launch_mlp_reduce_adam(int np, int nblocks, const float *partial, float *grad, float *loss, float *theta, float *m, float *v,
                                  const MlpAdam &adam, bool apply, hipStream_t s) {
  hipLaunchKernelGGL(k_mlp_reduce_adam, dim3((np + 1 + 31) / 32), dim3(32 * kSlices), 0, s, np, nblocks, partial, grad, loss, theta, m, v, adam,
                     apply ? 1 : 0);
  return hipGetLastError();
}

hipError_t launch_mlp_predict(const MlpDims &d, const float *theta, const float *X, int n, float *Y, hipStream_t s) {
  if (!mlp_dims_supported(d)) return hipErrorInvalidValue;
  if (n <= 0) return hipSuccess;
  if (d.nh2 > 0) hipLaunchKernelGGL((k_mlp2_predict<6, 20, 20, 6>), dim3((n + kTpb - 1) / kTpb), dim3(kTpb), 0, s, d.alpha, theta, X, n, Y);
  else hipLaunchKernelGGL((k_mlp_predict<6, 20, 6>), dim3((n + kTpb - 1) / kTpb), dim3(kTpb), 0, s, d.alpha, theta, X, n, Y);
  return hipGetLastError();
}

hipError_t launch_sgs_model_samples(long long n, const double *train, const double *filtered, const double *G, const double *A, const CeedMiGas &gas,
                                    float *X, double *S, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const int grid = (int)((n + 255) / 256 < 8192 ? (n + 255) / 256 : 8192);
  hipLaunchKernelGGL(k_sgs_model_samples, dim3(grid), dim3(256), 0, s, n, train, filtered, G, A, gas, X, S);
  return hipGetLastError();
}
