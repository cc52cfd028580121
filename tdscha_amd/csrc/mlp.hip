// Small fully connected network in FP32 for the learned continued-fraction
// terminator: n_in -> width (x n_hidden, SiLU) -> n_out (linear), with
// forward, backward and Adam on the device.  Two losses:
//   kind 0  weighted mean-squared error against FP32 targets;
//   kind 1  spectral loss: the n_out = 10 outputs are the tail parameters of a
//           continued fraction (asymptotic a_inf, b_inf and four corrections
//           each to the next a and b), appended to the first K coefficients
//           of a chain; the loss is the mean squared deviation of the
//           resulting spectrum from a reference spectrum, and its gradient
//           comes from the adjoint of the continued-fraction recurrence (FP64).
// Every reduction is a fixed-order loop or tree (no atomics), so training is
// reproducible.  Parameters are one contiguous FP32 array
//   [W0 (d1 x d0), b0 (d1), W1 (d2 x d1), b1 (d2), ...], W row-major [out][in].
#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "common.hpp"
#include "../../include/tdscha_amd.h"

namespace tdscha {

constexpr int kCfOut = 10;   // a_inf, b_inf, da[4], db[4]
constexpr int kCfTail = 4;
constexpr int kCfBlocks = 2048;   // work-groups of the spectral loss that fill the chip

struct Mlp {
  int n_layers = 0;              // linear layers = n_hidden + 1
  std::vector<int> dims;         // d0 = n_in, ..., d_L = n_out
  std::vector<long> w_off, b_off;
  long n_params = 0;
  int max_batch = 0, max_dim = 0;
  float* params = nullptr;       // device
  float* grads = nullptr;
  float* m1 = nullptr;           // Adam moments
  float* m2 = nullptr;
  float* act = nullptr;          // [n_layers + 1][max_batch][max_dim] layer outputs (act[0] = input)
  float* pre = nullptr;          // [n_layers][max_batch][max_dim] pre-activations
  float* dz = nullptr;           // fused: [n_layers][max_batch][max_dim], the gradient at
                                 // each layer's output; else [2] of them in turn
  float* target = nullptr;       // [max_batch][n_out] (kind 0)
  float* wout = nullptr;         // [n_out] loss weights (kind 0)
  float* loss_part = nullptr;    // [max_batch], in the pinned memory
  int* idx = nullptr;            // [max_batch] rows of the data arrays in use
  // data arrays (device): either one batch (direct calls) or a training set
  float* data_x = nullptr;       // [n][n_in]
  float* data_t = nullptr;       // [n][n_out]       kind 0
  double* data_ch = nullptr;     // [n][2K + 2]      kind 1: a[K], b[K], b0, 1/max|S_ref|
  double* data_ref = nullptr;    // [n][n_w]         kind 1: S_ref / max|S_ref|
  long data_cap_x = 0, data_cap_t = 0, data_cap_ch = 0, data_cap_ref = 0;
  // spectral loss configuration
  int cf_K = 0, cf_nw = 0;
  double cf_eta = 0.0, cf_scale = 1.0;
  double* cf_w = nullptr;        // [n_w]
  double* cf_mean = nullptr;     // [10]
  double* cf_std = nullptr;      // [10]
  double* cf_part = nullptr;     // [samples x slices <= max_batch + kCfBlocks][11]
  long step = 0;                 // Adam steps taken
  bool fused = false;            // all layers of a pass in one kernel
  char* pinned = nullptr;        // host memory the kernels access: small inputs (kPinned
                                 // bytes), outputs (kPinned), losses (max_batch)
  char* staged = nullptr;        // [kPinned] device copy of small inputs
  hipStream_t stream = nullptr;
};

__device__ __forceinline__ float silu(float z) { return z / (1.0f + expf(-z)); }
__device__ __forceinline__ float dsilu(float z) {
  const float s = 1.0f / (1.0f + expf(-z));
  return s * (1.0f + z * (1.0f - s));
}

// Z[b][o] = sum_i X[b][i] W[o][i] + bias[o]; A = act ? SiLU(Z) : Z.  16 x 16
// output tile per block, K in chunks of 16 through LDS.
__global__ void mlp_linear_fwd(const float* __restrict__ X, const float* __restrict__ W,
                               const float* __restrict__ bias, float* __restrict__ Z,
                               float* __restrict__ A, int B, int in, int out, int ld, int act) {
  __shared__ float xs[16][17], ws[16][17];
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const int b = blockIdx.y * 16 + ty, o = blockIdx.x * 16 + tx;
  float s = 0.f;
  for (int k0 = 0; k0 < in; k0 += 16) {
    const int xk = k0 + tx;
    xs[ty][tx] = (b < B && xk < in) ? X[(long)b * ld + xk] : 0.f;
    const int wo = blockIdx.x * 16 + ty;
    ws[ty][tx] = (wo < out && xk < in) ? W[(long)wo * in + xk] : 0.f;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k) s += xs[ty][k] * ws[tx][k];
    __syncthreads();
  }
  if (b < B && o < out) {
    const float z = s + bias[o];
    Z[(long)b * ld + o] = z;
    A[(long)b * ld + o] = act ? silu(z) : z;
  }
}

// Small networks (at most kFuseLayers layers of at most kFuseDim): every layer of a
// pass in one kernel, a work-group per R batch rows, its activations in LDS.  The
// weights pass through LDS in panels of 128 of the summed index by 128 outputs, the
// next panel (of the next layer too) in registers meanwhile.  The sums run in the order
// of the kernels above.  Bound by the latency of a panel; the separate kernels were 3
// to 5 launches of 4.6 to 5.6 us per pass (64 rows of 80-128-128-128-10: forward 22 ->
// 19 us, input gradients 16 -> 12 us; one row: forward 21 -> 15 us).
constexpr int kFuseLayers = 8;
constexpr int kFuseDim = 256;
constexpr int kFusePanel = 128;
constexpr int kFuseThreads = 512;

struct MlpShape {
  int layers, ld;                      // ld: row stride of activations
  long stride;                         // of a layer's activations
  int dim[kFuseLayers + 1];
  long w[kFuseLayers], b[kFuseLayers];
  int tile[kFuseLayers + 1];           // first 16 x 16 weight tile of a layer
};

template <int R>
constexpr int fused_lds() {
  return (kFusePanel * (kFusePanel + 1) + 2 * R * kFuseDim) * (int)sizeof(float);
}

// Panels of `steps` layers in turn; sizes(s) = (nk, no) and weights pw(s) of step s:
// W(k, o) at pw[o * nk + k] (KC) or pw[k * no + o].  done(s, o, row, sum) takes the sum
// over k of output o, row = t / 128 + 4 r, from x = xs[s & 1]; columns of x from nk on
// are zero.  Thread: output t % 128 of a panel, rows t / 128 + 4 r.
template <int R, bool KC, typename Sizes, typename Weights, typename Done>
__device__ __forceinline__ void fused_layers(int steps, Sizes sizes, Weights weights, Done done,
                                             float (*xs)[R][kFuseDim],
                                             float (*ws)[kFusePanel + 1]) {
  constexpr int P = kFusePanel, E = P * P / kFuseThreads, RT = R / 4;
  const int t = threadIdx.x, lo = t & 127, hi = t >> 7;
  float v[E];
  auto fetch = [&](int s, int o0, int k0) {
    const int2 z = sizes(s);
    const float* pw = weights(s);
#pragma unroll
    for (int e = 0; e < E; ++e) {   // clamped, so that every load can be in flight
      const int k = min(k0 + (KC ? lo : hi + 4 * e), z.x - 1);
      const int o = min(o0 + (KC ? hi + 4 * e : lo), z.y - 1);
      v[e] = KC ? pw[o * z.x + k] : pw[k * z.y + o];
    }
  };
  float acc[RT];
  int s = 0, o0 = 0, k0 = 0;
  fetch(0, 0, 0);
  while (s < steps) {
    const int2 z = sizes(s);
    __syncthreads();
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int k = KC ? lo : hi + 4 * e, o = KC ? hi + 4 * e : lo;
      ws[k][o] = k0 + k < z.x && o0 + o < z.y ? v[e] : 0.f;
    }
    __syncthreads();
    int s1 = s, o1 = o0, k1 = k0 + P;
    if (k1 >= z.x) {
      k1 = 0;
      o1 += P;
    }
    if (o1 >= z.y) {
      o1 = 0;
      ++s1;
    }
    if (s1 < steps) fetch(s1, o1, k1);
    if (k0 == 0)
#pragma unroll
      for (int r = 0; r < RT; ++r) acc[r] = 0.f;
    const int ke = min(P, z.x - k0);
    for (int kb = 0; kb < ke; kb += 8)
#pragma unroll
      for (int k = kb; k < kb + 8; ++k) {
        const float w = ws[k][lo];
#pragma unroll
        for (int r = 0; r < RT; ++r) acc[r] += xs[s & 1][hi + 4 * r][k0 + k] * w;
      }
    if (k1 == 0)
#pragma unroll
      for (int r = 0; r < RT; ++r) done(s, o0 + lo, hi + 4 * r, acc[r]);
    s = s1;
    o0 = o1;
    k0 = k1;
  }
}

// forward of rows idx[..] (or the rows themselves) of x: the last layer's output to
// y_out [B][n_out], or (null) every layer's pre-activations and activations
template <int R>
__global__ __launch_bounds__(kFuseThreads) void mlp_fused_fwd(
    MlpShape m, const float* __restrict__ params, const float* __restrict__ x, int xld,
    const int* __restrict__ idx, int B, float* __restrict__ y_out, float* __restrict__ act,
    float* __restrict__ pre) {
  extern __shared__ float fsh[];
  auto ws = reinterpret_cast<float(*)[kFusePanel + 1]>(fsh);
  auto xs = reinterpret_cast<float(*)[R][kFuseDim]>(fsh + kFusePanel * (kFusePanel + 1));
  const int b0 = blockIdx.x * R;
  for (int e = threadIdx.x; e < R * kFuseDim; e += kFuseThreads) {
    const int r = e / kFuseDim, i = e % kFuseDim, b = b0 + r;
    const bool in = b < B && i < m.dim[0];
    const float v = in ? x[(long)(idx ? idx[b] : b) * xld + i] : 0.f;
    xs[0][r][i] = v;
    if (!y_out && in) act[(long)b * m.ld + i] = v;
  }
  fused_layers<R, true>(
      m.layers, [&](int l) { return make_int2(m.dim[l], m.dim[l + 1]); },
      [&](int l) { return params + m.w[l]; },
      [&](int l, int o, int row, float sum) {
        const bool last = l + 1 == m.layers, in = o < m.dim[l + 1];
        const float z = sum + (in ? params[m.b[l] + o] : 0.f), y = last ? z : silu(z);
        // (zero past the layer's width whatever the sum: 0 x Inf is not)
        xs[(l + 1) & 1][row][o] = in ? y : 0.f;
        const int b = b0 + row;
        if (b >= B || !in) return;
        if (!y_out) {
          const long e = (long)b * m.ld + o;
          pre[l * m.stride + e] = z;
          act[(l + 1) * m.stride + e] = y;
        } else if (last) {
          y_out[(long)b * m.dim[l + 1] + o] = y;
        }
      },
      xs, ws);
}

// gradients at the outputs of layers layers - 2 .. 0 from the one at the last
template <int R>
__global__ __launch_bounds__(kFuseThreads) void mlp_fused_bwd_x(MlpShape m,
                                                                const float* __restrict__ params,
                                                                const float* __restrict__ pre,
                                                                int B, float* __restrict__ dz) {
  extern __shared__ float fsh[];
  auto ws = reinterpret_cast<float(*)[kFusePanel + 1]>(fsh);
  auto xs = reinterpret_cast<float(*)[R][kFuseDim]>(fsh + kFusePanel * (kFusePanel + 1));
  const int b0 = blockIdx.x * R, L = m.layers;
  for (int e = threadIdx.x; e < R * kFuseDim; e += kFuseThreads) {
    const int r = e / kFuseDim, i = e % kFuseDim, b = b0 + r;
    xs[0][r][i] = b < B && i < m.dim[L] ? dz[(L - 1) * m.stride + (long)b * m.ld + i] : 0.f;
  }
  // step s: through layer l = L - 1 - s to the output of layer l - 1
  fused_layers<R, false>(
      L - 1, [&](int s) { return make_int2(m.dim[L - s], m.dim[L - 1 - s]); },
      [&](int s) { return params + m.w[L - 1 - s]; },
      [&](int s, int i, int row, float sum) {
        const int b = b0 + row, l = L - 1 - s;
        float g = 0.f;
        if (b < B && i < m.dim[l]) {
          const long e = (l - 1) * m.stride + (long)b * m.ld + i;
          g = sum * dsilu(pre[e]);
          dz[e] = g;
        }
        xs[(s + 1) & 1][row][i] = g;
      },
      xs, ws);
}

// kind 0: dY = 2 w (Y - T) / B, loss_part = sum_o w (Y - T)^2 / B
__global__ void mlp_mse_grad(const float* __restrict__ Y, const float* __restrict__ T,
                             const float* __restrict__ w, float* __restrict__ dY,
                             float* __restrict__ loss_part, int B, int out, int ld) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= B) return;
  float l = 0.f;
  for (int o = 0; o < out; ++o) {
    const float d = Y[(long)b * ld + o] - T[(long)b * out + o];
    dY[(long)b * ld + o] = 2.0f * w[o] * d / (float)B;
    l += w[o] * d * d;
  }
  loss_part[b] = l / (float)B;
}

struct cplx {
  double r, i;
};
__device__ __forceinline__ cplx cmul(cplx a, cplx b) {
  return {a.r * b.r - a.i * b.i, a.r * b.i + a.i * b.r};
}
__device__ __forceinline__ cplx cinv(cplx z) {
  const double d = 1.0 / (z.r * z.r + z.i * z.i);
  return {z.r * d, -z.i * d};
}
__device__ __forceinline__ cplx cscale(cplx a, double s) { return {a.r * s, a.i * s}; }

// kind 1: a slice of the frequency grid of one sample per block (grid.x samples,
// grid.y slices; cf_loss_sum adds the slices).
// Tail: terminator root from (A, B) = b0 (p0, p1) as in the reference's
// terminator (no smearing in its discriminant, smaller-modulus root, ties to
// the minus root), then the four predicted levels a_j = b0 (p0 + p_{2+j}),
// b_j = b0 (p1 + p_{6+j}), then the chain's K measured levels.  The
// derivative of g with respect to the ten parameters is carried through the
// tail levels; above them dG/dg_K = prod_i b_i^2 g_i^2.
__global__ void __launch_bounds__(256) cf_loss_kernel(
    const float* __restrict__ Y, int ld, const int* __restrict__ idx,
    const double* __restrict__ chains, const double* __restrict__ ref,
    const double* __restrict__ wgrid, int n_w, int K, double eta,
    const double* __restrict__ out_mean, const double* __restrict__ out_std,
    double* __restrict__ part) {
  __shared__ double red[kCfOut + 1][4];
  const int bi = blockIdx.x;
  const long row = idx ? idx[bi] : bi;
  const double* ch = chains + row * (2 * K + 2);
  const double* av = ch;
  const double* bv = ch + K;
  const double b0 = ch[2 * K];
  const double inv_s = ch[2 * K + 1];
  const double* rf = ref + row * n_w;
  double p[kCfOut];
#pragma unroll
  for (int o = 0; o < kCfOut; ++o) p[o] = out_mean[o] + out_std[o] * (double)Y[(long)bi * ld + o];
  double lsum = 0.0, gacc[kCfOut];
#pragma unroll
  for (int o = 0; o < kCfOut; ++o) gacc[o] = 0.0;
  const double A = b0 * p[0], Bt = b0 * p[1];
  for (int k = blockIdx.y * 256 + threadIdx.x; k < n_w; k += 256 * gridDim.y) {
    const double om = wgrid[k];
    const double w2 = om * om, sm = 2.0 * om * eta;
    // terminator root and its derivatives
    const double d = A + w2;
    const double disc = d * d - 4.0 * Bt * Bt;
    const double den = 2.0 * Bt * Bt;
    cplx g, delta;
    if (disc < 0.0) {
      const double sq = sqrt(-disc);
      g = {d / den, -sq / den};
      delta = {0.0, -sq};
    } else {
      const double sq = sqrt(disc);
      const double gp = (d + sq) / den, gmi = (d - sq) / den;
      if (fabs(gp) < fabs(gmi)) {
        g = {gp, 0.0};
        delta = {sq, 0.0};
      } else {
        g = {gmi, 0.0};
        delta = {-sq, 0.0};
      }
    }
    cplx dg[kCfOut];
#pragma unroll
    for (int o = 0; o < kCfOut; ++o) dg[o] = {0.0, 0.0};
    if (delta.r != 0.0 || delta.i != 0.0) {
      const cplx idl = cinv(delta);
      dg[0] = cscale(cmul(g, idl), b0);
      dg[1] = cscale(cmul(cmul(g, g), idl), -2.0 * Bt * b0);
    }
    // predicted tail levels, bottom up
#pragma unroll
    for (int j = kCfTail - 1; j >= 0; --j) {
      const double aj = b0 * (p[0] + p[2 + j]);
      const double bj = b0 * (p[1] + p[6 + j]);
      const double bj2 = bj * bj;
      const cplx gn = cinv({aj + w2 - bj2 * g.r, sm - bj2 * g.i});
      const cplx mg2 = cscale(cmul(gn, gn), -1.0);
      const cplx dbt = cscale(g, -2.0 * bj * b0);   // d(e - b^2 g)/dp through b: -2 b b0 g
#pragma unroll
      for (int o = 0; o < kCfOut; ++o) {
        cplx t = cscale(dg[o], -bj2);
        if (o == 0 || o == 2 + j) t.r += b0;
        if (o == 1 || o == 6 + j) {
          t.r += dbt.r;
          t.i += dbt.i;
        }
        dg[o] = cmul(mg2, t);
      }
      g = gn;
    }
    // the chain's own levels
    // (eight levels' coefficients loaded at once: one wait per eight)
    cplx D = {1.0, 0.0};
    for (int i0 = K - 1; i0 >= 0; i0 -= 8) {
      double la[8], lb[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int i = i0 - e > 0 ? i0 - e : 0;
        la[e] = av[i];
        lb[e] = bv[i];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if (i0 - e < 0) break;
        const double bi2 = lb[e] * lb[e];
        const cplx gn = cinv({la[e] + w2 - bi2 * g.r, sm - bi2 * g.i});
        D = cscale(cmul(D, cmul(gn, gn)), bi2);
        g = gn;
      }
    }
    // Wigner convention: spectrum = -Im(G)
    const double r = -g.i * inv_s - rf[k];
    lsum += r * r;
    const double c = 2.0 * r * inv_s;
#pragma unroll
    for (int o = 0; o < kCfOut; ++o) {
      const cplx t = cmul(D, dg[o]);
      gacc[o] -= c * t.i;
    }
  }
  // sums over the grid: a wave, then the four waves in order
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int q = 0; q <= kCfOut; ++q) {
    double v = q ? gacc[q - 1] : lsum;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if (lane == 0) red[q][wave] = v;
  }
  __syncthreads();
  if (threadIdx.x <= kCfOut) {
    const int q = threadIdx.x;
    part[((long)bi * gridDim.y + blockIdx.y) * (kCfOut + 1) + q] =
        (red[q][0] + red[q][1]) + (red[q][2] + red[q][3]);
  }
}

// slices of cf_loss_kernel in order: loss and gradient of sample blockIdx.x
__global__ void cf_loss_sum(const double* __restrict__ part, int slices, int n_w, int ld,
                            const double* __restrict__ out_std, double scale,
                            float* __restrict__ dY, float* __restrict__ loss_part) {
  const int bi = blockIdx.x, q = threadIdx.x;
  if (q > kCfOut) return;
  const double* p = part + (long)bi * slices * (kCfOut + 1) + q;
  double v = 0.0;
#pragma unroll 8
  for (int k = 0; k < slices; ++k) v += p[k * (kCfOut + 1)];
  if (q == 0)
    loss_part[bi] = (float)(scale * v / n_w);
  else
    dY[(long)bi * ld + q - 1] = (float)(scale * v / n_w * out_std[q - 1]);
}

// dW[o][i] = sum_b dZ[b][o] Ain[b][i]; db[o] = sum_b dZ[b][o] (fixed order in b)
__device__ __forceinline__ void bwd_w_tile(const float* __restrict__ dZ,
                                           const float* __restrict__ Ain, float* __restrict__ dW,
                                           float* __restrict__ db, int B, int in, int out, int ld,
                                           int bx, int by) {
  __shared__ float zs[16][17], as[16][17];
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const int o = by * 16 + ty, i = bx * 16 + tx;
  float s = 0.f, sb = 0.f;
  for (int b0 = 0; b0 < B; b0 += 16) {
    const int zb = b0 + tx;
    zs[ty][tx] = (zb < B && o < out) ? dZ[(long)zb * ld + o] : 0.f;   // zs[o][b]
    const int ab = b0 + ty;
    as[ty][tx] = (ab < B && i < in) ? Ain[(long)ab * ld + i] : 0.f;   // as[b][i]
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      s += zs[ty][k] * as[k][tx];
      sb += zs[ty][k];
    }
    __syncthreads();
  }
  if (o < out && i < in) dW[(long)o * in + i] = s;
  if (o < out && bx == 0 && tx == 0) db[o] = sb;
}

__global__ void mlp_linear_bwd_w(const float* __restrict__ dZ, const float* __restrict__ Ain,
                                 float* __restrict__ dW, float* __restrict__ db, int B, int in,
                                 int out, int ld) {
  bwd_w_tile(dZ, Ain, dW, db, B, in, out, ld, blockIdx.x, blockIdx.y);
}

// the weight gradients of every layer in one launch
__global__ void mlp_fused_bwd_w(MlpShape m, const float* __restrict__ dz,
                                const float* __restrict__ act, float* __restrict__ grads, int B) {
  int l = 0;
  while ((int)blockIdx.x >= m.tile[l + 1]) ++l;
  const int q = blockIdx.x - m.tile[l], nx = (m.dim[l] + 15) / 16;
  bwd_w_tile(dz + l * m.stride, act + l * m.stride, grads + m.w[l], grads + m.b[l], B, m.dim[l],
             m.dim[l + 1], m.ld, q % nx, q / nx);
}

// dZprev[b][i] = (sum_o dZ[b][o] W[o][i]) * SiLU'(Zprev[b][i])
__global__ void mlp_linear_bwd_x(const float* __restrict__ dZ, const float* __restrict__ W,
                                 const float* __restrict__ Zprev, float* __restrict__ dZprev,
                                 int B, int in, int out, int ld) {
  __shared__ float zs[16][17], ws[16][17];
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const int b = blockIdx.y * 16 + ty, i = blockIdx.x * 16 + tx;
  float s = 0.f;
  for (int o0 = 0; o0 < out; o0 += 16) {
    const int zo = o0 + tx;
    zs[ty][tx] = (b < B && zo < out) ? dZ[(long)b * ld + zo] : 0.f;   // zs[b][o]
    const int wo = o0 + ty;
    ws[ty][tx] = (wo < out && i < in) ? W[(long)wo * in + i] : 0.f;   // ws[o][i]
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k) s += zs[ty][k] * ws[k][tx];
    __syncthreads();
  }
  if (b < B && i < in) dZprev[(long)b * ld + i] = s * dsilu(Zprev[(long)b * ld + i]);
}

__global__ void mlp_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                         float* __restrict__ v, long n, float lr, float b1, float b2, float eps,
                         float bc1, float bc2) {
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const float gi = g[e];
  const float mi = b1 * m[e] + (1.f - b1) * gi;
  const float vi = b2 * v[e] + (1.f - b2) * gi * gi;
  m[e] = mi;
  v[e] = vi;
  p[e] -= lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
}

// minibatch rows into the first layer's input (and kind-0 targets)
__global__ void mlp_gather(const float* __restrict__ dx, const float* __restrict__ dt,
                           const int* __restrict__ idx, int B, int n_in, int n_out, int ld,
                           float* __restrict__ x, float* __restrict__ t) {
  const int b = blockIdx.x;
  if (b >= B) return;
  const long r = idx ? idx[b] : b;
  for (int i = threadIdx.x; i < n_in; i += blockDim.x) x[(long)b * ld + i] = dx[r * n_in + i];
  if (dt)
    for (int o = threadIdx.x; o < n_out; o += blockDim.x) t[(long)b * n_out + o] = dt[r * n_out + o];
}

// rows of stride ld to contiguous ones
__global__ void mlp_rows(const float* __restrict__ y, int B, int n, int ld,
                         float* __restrict__ out) {
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e < (long)B * n) out[e] = y[e / n * ld + e % n];
}

static float* act_l(Mlp* m, int l) { return m->act + (long)l * m->max_batch * m->max_dim; }
static float* pre_l(Mlp* m, int l) { return m->pre + (long)l * m->max_batch * m->max_dim; }

// the fused kernels use more than 64 KB of the CU's 160 KB of LDS
static bool fused_ready() {
  auto allow = [](const void* f, int bytes) {
    return hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) == hipSuccess;
  };
  const bool ok = allow((const void*)mlp_fused_fwd<4>, fused_lds<4>()) &&
                  allow((const void*)mlp_fused_fwd<8>, fused_lds<8>()) &&
                  allow((const void*)mlp_fused_bwd_x<4>, fused_lds<4>()) &&
                  allow((const void*)mlp_fused_bwd_x<8>, fused_lds<8>());
  if (!ok) (void)hipGetLastError();
  return ok;
}

static MlpShape shape(const Mlp* m) {
  MlpShape h;
  h.layers = m->n_layers;
  h.ld = m->max_dim;
  h.stride = (long)m->max_batch * m->max_dim;
  h.tile[0] = 0;
  for (int l = 0; l < m->n_layers; ++l) {
    h.dim[l] = m->dims[l];
    h.w[l] = m->w_off[l];
    h.b[l] = m->b_off[l];
    h.tile[l + 1] = h.tile[l] + ((m->dims[l] + 15) / 16) * ((m->dims[l + 1] + 15) / 16);
  }
  h.dim[m->n_layers] = m->dims[m->n_layers];
  return h;
}

// fused forward of rows of x (y: see mlp_fused_fwd); 4 rows to a work-group until every CU
// has four of them, then 8
static void forward_fused(Mlp* m, int B, const float* x, const int* idx, float* y) {
  const int xld = m->dims[0];
  const MlpShape h = shape(m);
  if (B <= 4096)
    hipLaunchKernelGGL(mlp_fused_fwd<4>, dim3((B + 3) / 4), dim3(kFuseThreads), fused_lds<4>(),
                       m->stream, h, m->params, x, xld, idx, B, y, m->act, m->pre);
  else
    hipLaunchKernelGGL(mlp_fused_fwd<8>, dim3((B + 7) / 8), dim3(kFuseThreads), fused_lds<8>(),
                       m->stream, h, m->params, x, xld, idx, B, y, m->act, m->pre);
}

static void backward_fused(Mlp* m, int B) {
  const MlpShape h = shape(m);
  if (m->n_layers > 1) {
    if (B <= 4096)
      hipLaunchKernelGGL(mlp_fused_bwd_x<4>, dim3((B + 3) / 4), dim3(kFuseThreads), fused_lds<4>(),
                         m->stream, h, m->params, m->pre, B, m->dz);
    else
      hipLaunchKernelGGL(mlp_fused_bwd_x<8>, dim3((B + 7) / 8), dim3(kFuseThreads), fused_lds<8>(),
                         m->stream, h, m->params, m->pre, B, m->dz);
  }
  hipLaunchKernelGGL(mlp_fused_bwd_w, dim3(h.tile[m->n_layers]), dim3(256), 0, m->stream, h, m->dz,
                     m->act, m->grads, B);
}

static void forward(Mlp* m, int B) {
  const int ld = m->max_dim;
  for (int l = 0; l < m->n_layers; ++l) {
    const int in = m->dims[l], out = m->dims[l + 1];
    dim3 g((out + 15) / 16, (B + 15) / 16);
    hipLaunchKernelGGL(mlp_linear_fwd, g, dim3(256), 0, m->stream, act_l(m, l),
                       m->params + m->w_off[l], m->params + m->b_off[l], pre_l(m, l),
                       act_l(m, l + 1), B, in, out, ld, l + 1 < m->n_layers ? 1 : 0);
  }
}

// device arrays of a pass: rows idx[0 .. B) (null: the first B rows) of each
struct MlpData {
  const float *x = nullptr, *t = nullptr;
  const double *ch = nullptr, *ref = nullptr;
  const int* idx = nullptr;
};

// loss partials and the gradient with respect to the network outputs
static void loss_head(Mlp* m, const MlpData& d, int kind, int B) {
  const int ld = m->max_dim, L = m->n_layers;
  float* dz = m->dz + (m->fused ? (long)(L - 1) * m->max_batch * ld : 0);
  if (kind == 0) {
    hipLaunchKernelGGL(mlp_mse_grad, dim3((B + 255) / 256), dim3(256), 0, m->stream,
                       act_l(m, L), m->target, m->wout, dz, m->loss_part, B, m->dims[L], ld);
  } else {
    // slices of 256 frequencies while they fill the chip (64 samples of 2000: 60 us
    // with one block each, 17 us in eight, and 4 us to add them)
    const int slices = std::min((m->cf_nw + 255) / 256, (kCfBlocks + B - 1) / B);
    hipLaunchKernelGGL(cf_loss_kernel, dim3(B, slices), dim3(256), 0, m->stream, act_l(m, L), ld,
                       d.idx, d.ch, d.ref, m->cf_w, m->cf_nw, m->cf_K, m->cf_eta,
                       m->cf_mean, m->cf_std, m->cf_part);
    hipLaunchKernelGGL(cf_loss_sum, dim3(B), dim3(64), 0, m->stream, m->cf_part, slices, m->cf_nw,
                       ld, m->cf_std, m->cf_scale / B, dz, m->loss_part);
  }
}

static void backward(Mlp* m, int B) {
  const int ld = m->max_dim, L = m->n_layers;
  float* dzb[2] = {m->dz, m->dz + (long)m->max_batch * m->max_dim};
  int cur = 0;
  for (int l = L - 1; l >= 0; --l) {
    const int in = m->dims[l], out = m->dims[l + 1];
    hipLaunchKernelGGL(mlp_linear_bwd_w, dim3((in + 15) / 16, (out + 15) / 16), dim3(256), 0,
                       m->stream, dzb[cur], act_l(m, l), m->grads + m->w_off[l],
                       m->grads + m->b_off[l], B, in, out, ld);
    if (l > 0) {
      hipLaunchKernelGGL(mlp_linear_bwd_x, dim3((in + 15) / 16, (B + 15) / 16), dim3(256), 0,
                         m->stream, dzb[cur], m->params + m->w_off[l], pre_l(m, l - 1),
                         dzb[1 - cur], B, in, out, ld);
      cur = 1 - cur;
    }
  }
}

static void adam(Mlp* m, float lr, float b1, float b2, float eps) {
  m->step += 1;
  const float bc1 = 1.f - powf(b1, (float)m->step), bc2 = 1.f - powf(b2, (float)m->step);
  hipLaunchKernelGGL(mlp_adam, dim3((unsigned)((m->n_params + 255) / 256)), dim3(256), 0,
                     m->stream, m->params, m->grads, m->m1, m->m2, m->n_params, lr, b1, b2, eps,
                     bc1, bc2);
}

template <typename T>
static int ensure(T** p, long* cap, long n) {
  if (*cap >= n && *p) return 0;
  if (*p) TDS_CHECK_HIP(hipFree(*p));
  *p = nullptr;
  *cap = 0;
  TDS_CHECK_HIP(hipMalloc((void**)p, sizeof(T) * (n > 0 ? n : 1)));
  *cap = n;
  return 0;
}

// Upload n rows of data for the given loss kind to the device arrays (the host arrays
// may be released on return).  What fits goes through the pinned memory in one copy.
static int upload_data(Mlp* m, int kind, long n, const float* x, const float* t,
                       const double* chains, const double* ref, MlpData* d) {
  const int n_in = m->dims[0], n_out = m->dims[m->n_layers];
  TDS_CHECK_HIP(hipStreamSynchronize(m->stream));
  size_t used = 0;
  auto place = [&](auto** dev, long* cap, const auto* host, auto** out, size_t count) -> int {
    const size_t bytes = sizeof(*host) * count;
    if (used + bytes <= kPinned) {
      std::memcpy(m->pinned + used, host, bytes);
      *out = reinterpret_cast<std::remove_reference_t<decltype(*out)>>(m->staged + used);
      used += (bytes + 255) / 256 * 256;
      return 0;
    }
    const int rc = ensure(dev, cap, (long)count);
    if (rc) return rc;
    TDS_CHECK_HIP(hipMemcpy(*dev, host, bytes, hipMemcpyHostToDevice));
    *out = *dev;
    return 0;
  };
  int rc = place(&m->data_x, &m->data_cap_x, x, &d->x, (size_t)n * n_in);
  if (rc) return rc;
  if (kind == 0) {
    rc = place(&m->data_t, &m->data_cap_t, t, &d->t, (size_t)n * n_out);
  } else {
    rc = place(&m->data_ch, &m->data_cap_ch, chains, &d->ch, (size_t)n * (2L * m->cf_K + 2));
    if (rc) return rc;
    rc = place(&m->data_ref, &m->data_cap_ref, ref, &d->ref, (size_t)n * m->cf_nw);
  }
  if (rc) return rc;
  if (used)
    TDS_CHECK_HIP(hipMemcpyAsync(m->staged, m->pinned, std::min(used, kPinned),
                                 hipMemcpyHostToDevice, m->stream));
  return 0;
}

// one minibatch: gather rows, forward, loss head, backward
static void batch_pass(Mlp* m, const MlpData& d, int kind, int B) {
  const int n_in = m->dims[0], n_out = m->dims[m->n_layers];
  if (kind == 0 || !m->fused)
    hipLaunchKernelGGL(mlp_gather, dim3(B), dim3(128), 0, m->stream, d.x,
                       kind == 0 ? d.t : nullptr, d.idx, B, m->fused ? 0 : n_in, n_out,
                       m->max_dim, act_l(m, 0), m->target);
  if (m->fused)
    forward_fused(m, B, d.x, d.idx, nullptr);
  else
    forward(m, B);
  loss_head(m, d, kind, B);
  if (m->fused)
    backward_fused(m, B);
  else
    backward(m, B);
}

static int check_kind(Mlp* m, int kind, const float* t, const double* chains, const double* ref) {
  TDS_REQUIRE(kind == 0 || kind == 1, 2, "mlp: loss kind must be 0 (MSE) or 1 (spectral)");
  if (kind == 0) {
    TDS_REQUIRE(t != nullptr, 2, "mlp: MSE loss needs targets");
  } else {
    TDS_REQUIRE(m->cf_K > 0, 2, "mlp: spectral loss not configured (tdscha_mlp_set_cf_loss)");
    TDS_REQUIRE(chains != nullptr && ref != nullptr, 2, "mlp: spectral loss needs chains and ref");
  }
  return 0;
}

// sum of the pass's losses (waits for the stream)
static int read_loss(Mlp* m, int B, double* loss) {
  TDS_CHECK_HIP(hipStreamSynchronize(m->stream));
  double s = 0.0;
  for (int b = 0; b < B; ++b) s += m->loss_part[b];
  *loss = s;
  return 0;
}

// up to max_batch rows, contiguous on the host, through the pinned memory where they
// fit; the kernels read and write it directly
static int forward_start(Mlp* m, int B, const float* x, float* y) {
  const size_t bx = sizeof(float) * B * m->dims[0], by = sizeof(float) * B * m->dims[m->n_layers];
  const float* dx = reinterpret_cast<const float*>(m->pinned);
  if (m->fused && bx <= kPinned) {
    std::memcpy(m->pinned, x, bx);
  } else {
    const int rc = ensure(&m->data_x, &m->data_cap_x, (long)B * m->dims[0]);
    if (rc) return rc;
    TDS_CHECK_HIP(hipMemcpyAsync(m->data_x, x, bx, hipMemcpyHostToDevice, m->stream));
    dx = m->data_x;
  }
  const bool out = by <= kPinned;
  float* dy = out ? reinterpret_cast<float*>(m->pinned + kPinned) : m->target;
  if (m->fused) {
    forward_fused(m, B, dx, nullptr, dy);
  } else {
    hipLaunchKernelGGL(mlp_gather, dim3(B), dim3(128), 0, m->stream, dx, (const float*)nullptr,
                       (const int*)nullptr, B, m->dims[0], 0, m->max_dim, act_l(m, 0),
                       (float*)nullptr);
    forward(m, B);
    const long n = (long)B * m->dims[m->n_layers];
    hipLaunchKernelGGL(mlp_rows, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, m->stream,
                       act_l(m, m->n_layers), B, m->dims[m->n_layers], m->max_dim, dy);
  }
  TDS_CHECK_HIP(hipGetLastError());
  if (!out) TDS_CHECK_HIP(hipMemcpyAsync(y, dy, by, hipMemcpyDeviceToHost, m->stream));
  return 0;
}

static int forward_end(Mlp* m, int B, float* y) {
  TDS_CHECK_HIP(hipStreamSynchronize(m->stream));
  const size_t by = sizeof(float) * B * m->dims[m->n_layers];
  if (by <= kPinned) std::memcpy(y, m->pinned + kPinned, by);
  return 0;
}

}  // namespace tdscha

using namespace tdscha;

extern "C" {

int tdscha_mlp_create(tdscha_mlp** out, int n_in, int width, int n_hidden, int n_out,
                      int max_batch, const float* init_params) {
  TDS_REQUIRE(out != nullptr, 2, "tdscha_mlp_create: NULL out");
  TDS_REQUIRE(n_in > 0 && width > 0 && n_hidden >= 0 && n_out > 0 && max_batch > 0, 2,
              "tdscha_mlp_create: sizes must be positive");
  TDS_REQUIRE(n_in <= 4096 && width <= 4096 && n_out <= 4096 && n_hidden <= 64 &&
                  max_batch <= 65536,
              2, "tdscha_mlp_create: sizes above the supported maxima");
  *out = nullptr;
  Mlp* m = new Mlp();
  m->n_layers = n_hidden + 1;
  m->dims.push_back(n_in);
  for (int h = 0; h < n_hidden; ++h) m->dims.push_back(width);
  m->dims.push_back(n_out);
  long off = 0;
  for (int l = 0; l < m->n_layers; ++l) {
    m->w_off.push_back(off);
    off += (long)m->dims[l + 1] * m->dims[l];
    m->b_off.push_back(off);
    off += m->dims[l + 1];
  }
  m->n_params = off;
  m->max_batch = max_batch;
  for (int d : m->dims) m->max_dim = d > m->max_dim ? d : m->max_dim;
  const long act_n = (long)(m->n_layers + 1) * max_batch * m->max_dim;
  const long pre_n = (long)m->n_layers * max_batch * m->max_dim;
  m->fused = m->n_layers <= kFuseLayers && m->max_dim <= kFuseDim && fused_ready();
  const long dz_n = (m->fused ? m->n_layers : 2L) * max_batch * m->max_dim;
  auto fail = [&]() {
    tdscha_mlp_destroy(reinterpret_cast<tdscha_mlp*>(m));
    return -1;
  };
  if (hipStreamCreate(&m->stream) != hipSuccess ||
      hipMalloc((void**)&m->params, sizeof(float) * off) != hipSuccess ||
      hipMalloc((void**)&m->grads, sizeof(float) * off) != hipSuccess ||
      hipMalloc((void**)&m->m1, sizeof(float) * off) != hipSuccess ||
      hipMalloc((void**)&m->m2, sizeof(float) * off) != hipSuccess ||
      hipMalloc((void**)&m->act, sizeof(float) * act_n) != hipSuccess ||
      hipMalloc((void**)&m->pre, sizeof(float) * pre_n) != hipSuccess ||
      hipMalloc((void**)&m->dz, sizeof(float) * dz_n) != hipSuccess ||
      hipMalloc((void**)&m->target, sizeof(float) * max_batch * n_out) != hipSuccess ||
      hipMalloc((void**)&m->wout, sizeof(float) * n_out) != hipSuccess ||
      hipHostMalloc((void**)&m->pinned, 2 * kPinned + sizeof(float) * max_batch) != hipSuccess ||
      hipMalloc((void**)&m->staged, kPinned) != hipSuccess ||
      hipMalloc((void**)&m->idx, sizeof(int) * max_batch) != hipSuccess) {
    set_error("tdscha_mlp_create: device allocation failed");
    return fail();
  }
  m->loss_part = reinterpret_cast<float*>(m->pinned + 2 * kPinned);
  // zero once so padded columns of the activations stay finite
  if (hipMemset(m->act, 0, sizeof(float) * act_n) != hipSuccess ||
      hipMemset(m->pre, 0, sizeof(float) * pre_n) != hipSuccess ||
      hipMemset(m->dz, 0, sizeof(float) * dz_n) != hipSuccess ||
      hipMemset(m->m1, 0, sizeof(float) * off) != hipSuccess ||
      hipMemset(m->m2, 0, sizeof(float) * off) != hipSuccess) {
    set_error("tdscha_mlp_create: hipMemset failed");
    return fail();
  }
  std::vector<float> ones(n_out, 1.0f);
  hipError_t e = hipMemcpy(m->wout, ones.data(), sizeof(float) * n_out, hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = init_params ? hipMemcpy(m->params, init_params, sizeof(float) * off, hipMemcpyHostToDevice)
                    : hipMemset(m->params, 0, sizeof(float) * off);
  if (e != hipSuccess) {
    set_error(std::string("tdscha_mlp_create: ") + hipGetErrorString(e));
    return fail();
  }
  *out = reinterpret_cast<tdscha_mlp*>(m);
  return 0;
}

void tdscha_mlp_destroy(tdscha_mlp* h) {
  if (!h) return;
  Mlp* m = reinterpret_cast<Mlp*>(h);
  if (m->stream) hipStreamSynchronize(m->stream);
  void* ptrs[] = {m->params,  m->grads,  m->m1,      m->m2,       m->act,  m->pre,
                  m->dz,      m->target, m->wout,    m->staged, m->idx, m->data_x,
                  m->data_t,  m->data_ch, m->data_ref, m->cf_w,    m->cf_mean, m->cf_std,
                  m->cf_part};
  for (void* p : ptrs)
    if (p) hipFree(p);
  if (m->pinned) hipHostFree(m->pinned);
  if (m->stream) hipStreamDestroy(m->stream);
  delete m;
}

int tdscha_mlp_n_params(const tdscha_mlp* h, long* n) {
  TDS_REQUIRE(h && n, 2, "tdscha_mlp_n_params: NULL argument");
  *n = reinterpret_cast<const Mlp*>(h)->n_params;
  return 0;
}

int tdscha_mlp_get_params(tdscha_mlp* h, float* out) {
  TDS_REQUIRE(h && out, 2, "tdscha_mlp_get_params: NULL argument");
  Mlp* m = reinterpret_cast<Mlp*>(h);
  TDS_CHECK_HIP(hipStreamSynchronize(m->stream));
  TDS_CHECK_HIP(hipMemcpy(out, m->params, sizeof(float) * m->n_params, hipMemcpyDeviceToHost));
  return 0;
}

int tdscha_mlp_set_params(tdscha_mlp* h, const float* in, int reset_optimizer) {
  TDS_REQUIRE(h && in, 2, "tdscha_mlp_set_params: NULL argument");
  Mlp* m = reinterpret_cast<Mlp*>(h);
  TDS_CHECK_HIP(hipStreamSynchronize(m->stream));
  TDS_CHECK_HIP(hipMemcpy(m->params, in, sizeof(float) * m->n_params, hipMemcpyHostToDevice));
  if (reset_optimizer) {
    TDS_CHECK_HIP(hipMemset(m->m1, 0, sizeof(float) * m->n_params));
    TDS_CHECK_HIP(hipMemset(m->m2, 0, sizeof(float) * m->n_params));
    m->step = 0;
  }
  return 0;
}

int tdscha_mlp_set_mse_weights(tdscha_mlp* h, const float* w) {
  TDS_REQUIRE(h && w, 2, "tdscha_mlp_set_mse_weights: NULL argument");
  Mlp* m = reinterpret_cast<Mlp*>(h);
  TDS_CHECK_HIP(hipStreamSynchronize(m->stream));
  TDS_CHECK_HIP(hipMemcpy(m->wout, w, sizeof(float) * m->dims[m->n_layers], hipMemcpyHostToDevice));
  return 0;
}

int tdscha_mlp_set_cf_loss(tdscha_mlp* h, int K, int n_w, const double* w, double smearing,
                           const double* out_mean, const double* out_std, double loss_scale) {
  TDS_REQUIRE(h && w && out_mean && out_std, 2, "tdscha_mlp_set_cf_loss: NULL argument");
  Mlp* m = reinterpret_cast<Mlp*>(h);
  TDS_REQUIRE(m->dims[m->n_layers] == kCfOut, 2,
              "tdscha_mlp_set_cf_loss: the spectral loss needs 10 network outputs");
  TDS_REQUIRE(K > 0 && K <= 4096 && n_w > 0 && n_w <= (1 << 20), 2,
              "tdscha_mlp_set_cf_loss: K or n_w out of range");
  TDS_CHECK_HIP(hipStreamSynchronize(m->stream));
  if (m->cf_w) TDS_CHECK_HIP(hipFree(m->cf_w));
  m->cf_w = nullptr;
  if (!m->cf_mean) TDS_CHECK_HIP(hipMalloc((void**)&m->cf_mean, sizeof(double) * kCfOut));
  if (!m->cf_std) TDS_CHECK_HIP(hipMalloc((void**)&m->cf_std, sizeof(double) * kCfOut));
  if (!m->cf_part)
    TDS_CHECK_HIP(hipMalloc((void**)&m->cf_part, sizeof(double) * (kCfOut + 1) *
                                                     ((size_t)m->max_batch + kCfBlocks)));
  TDS_CHECK_HIP(hipMalloc((void**)&m->cf_w, sizeof(double) * n_w));
  TDS_CHECK_HIP(hipMemcpy(m->cf_w, w, sizeof(double) * n_w, hipMemcpyHostToDevice));
  TDS_CHECK_HIP(hipMemcpy(m->cf_mean, out_mean, sizeof(double) * kCfOut, hipMemcpyHostToDevice));
  TDS_CHECK_HIP(hipMemcpy(m->cf_std, out_std, sizeof(double) * kCfOut, hipMemcpyHostToDevice));
  m->cf_K = K;
  m->cf_nw = n_w;
  m->cf_eta = smearing;
  m->cf_scale = loss_scale;
  return 0;
}

int tdscha_mlp_forward(tdscha_mlp* h, int batch, const float* x, float* y) {
  TDS_REQUIRE(h && x && y, 2, "tdscha_mlp_forward: NULL argument");
  TDS_REQUIRE(batch >= 0, 2, "tdscha_mlp_forward: negative batch");
  return tdscha_mlp_forward_many(1, &h, batch, x, y);
}

int tdscha_mlp_forward_many(int n_nets, tdscha_mlp* const* nets, int batch, const float* x,
                            float* y) {
  TDS_REQUIRE(n_nets >= 0 && (n_nets == 0 || nets) && x && y, 2,
              "tdscha_mlp_forward_many: NULL argument");
  TDS_REQUIRE(batch >= 0, 2, "tdscha_mlp_forward: negative batch");
  for (int k = 0; k < n_nets; ++k) {
    TDS_REQUIRE(nets[k], 2, "tdscha_mlp_forward_many: NULL network");
    const Mlp *m = reinterpret_cast<const Mlp*>(nets[k]), *f = reinterpret_cast<const Mlp*>(nets[0]);
    TDS_REQUIRE(m->dims[0] == f->dims[0] && m->dims[m->n_layers] == f->dims[f->n_layers], 2,
                "tdscha_mlp_forward_many: networks of different inputs or outputs");
    for (int j = 0; j < k; ++j)
      TDS_REQUIRE(nets[j] != nets[k], 2, "tdscha_mlp_forward_many: the same network twice");
  }
  // each network's rows max_batch at a time, the networks of a round side by side
  for (int done = 0, left = n_nets ? batch : 0; left > 0;) {
    int step = left;
    for (int k = 0; k < n_nets; ++k)
      step = std::min(step, reinterpret_cast<const Mlp*>(nets[k])->max_batch);
    int rc = 0;
    for (int pass = 0; pass < 2; ++pass)
      for (int k = 0; k < n_nets; ++k) {
        Mlp* m = reinterpret_cast<Mlp*>(nets[k]);
        const long n_out = m->dims[m->n_layers];
        float* yk = y + (k * (long)batch + done) * n_out;
        const int r = pass ? forward_end(m, step, yk)
                           : forward_start(m, step, x + (long)done * m->dims[0], yk);
        if (r) rc = r;
      }
    if (rc) return rc;
    done += step;
    left -= step;
  }
  return 0;
}

int tdscha_mlp_loss_grad(tdscha_mlp* h, int kind, int batch, const float* x, const float* target,
                         const double* chains, const double* ref, float* loss, float* grad) {
  TDS_REQUIRE(h && x && loss, 2, "tdscha_mlp_loss_grad: NULL argument");
  Mlp* m = reinterpret_cast<Mlp*>(h);
  TDS_REQUIRE(batch > 0 && batch <= m->max_batch, 2, "tdscha_mlp_loss_grad: batch out of range");
  int rc = check_kind(m, kind, target, chains, ref);
  if (rc) return rc;
  MlpData d;
  rc = upload_data(m, kind, batch, x, target, chains, ref, &d);
  if (rc) return rc;
  batch_pass(m, d, kind, batch);
  TDS_CHECK_HIP(hipGetLastError());
  if (grad)
    TDS_CHECK_HIP(hipMemcpyAsync(grad, m->grads, sizeof(float) * m->n_params,
                                 hipMemcpyDeviceToHost, m->stream));
  double sum = 0.0;
  rc = read_loss(m, batch, &sum);
  if (!rc) *loss = (float)sum;
  return rc;
}

int tdscha_mlp_adam_step(tdscha_mlp* h, int kind, int batch, const float* x, const float* target,
                         const double* chains, const double* ref, float lr, float beta1,
                         float beta2, float eps, float* loss) {
  TDS_REQUIRE(h && x, 2, "tdscha_mlp_adam_step: NULL argument");
  Mlp* m = reinterpret_cast<Mlp*>(h);
  TDS_REQUIRE(batch > 0 && batch <= m->max_batch, 2, "tdscha_mlp_adam_step: batch out of range");
  int rc = check_kind(m, kind, target, chains, ref);
  if (rc) return rc;
  MlpData d;
  rc = upload_data(m, kind, batch, x, target, chains, ref, &d);
  if (rc) return rc;
  batch_pass(m, d, kind, batch);
  adam(m, lr, beta1, beta2, eps);
  TDS_CHECK_HIP(hipGetLastError());
  double sum = 0.0;
  rc = read_loss(m, batch, &sum);
  if (!rc && loss) *loss = (float)sum;
  return rc;
}

int tdscha_mlp_train(tdscha_mlp* h, int kind, long n_samples, const float* x, const float* target,
                     const double* chains, const double* ref, int batch, int epochs, float lr,
                     float beta1, float beta2, float eps, unsigned long long seed,
                     float* epoch_loss) {
  TDS_REQUIRE(h && x, 2, "tdscha_mlp_train: NULL argument");
  Mlp* m = reinterpret_cast<Mlp*>(h);
  TDS_REQUIRE(batch > 0 && batch <= m->max_batch && n_samples >= batch && epochs > 0 &&
                  n_samples <= (1L << 30),
              2, "tdscha_mlp_train: need 0 < batch <= max_batch, batch <= n_samples, epochs > 0");
  int rc = check_kind(m, kind, target, chains, ref);
  if (rc) return rc;
  MlpData d;
  rc = upload_data(m, kind, n_samples, x, target, chains, ref, &d);
  if (rc) return rc;
  d.idx = m->idx;
  // per-epoch permutation on the host (splitmix64-driven Fisher-Yates); the
  // last n_samples % batch rows of each permutation sit the epoch out
  std::vector<int> perm(n_samples);
  unsigned long long st = seed;
  auto next = [&st]() {
    st += 0x9E3779B97F4A7C15ull;
    unsigned long long z = st;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
  };
  const long n_batches = n_samples / batch;
  for (int ep = 0; ep < epochs; ++ep) {
    for (long i = 0; i < n_samples; ++i) perm[i] = (int)i;
    for (long i = n_samples - 1; i > 0; --i) {
      const long j = (long)(next() % (unsigned long long)(i + 1));
      const int tmp = perm[i];
      perm[i] = perm[j];
      perm[j] = tmp;
    }
    double ep_loss = 0.0;
    for (long bi = 0; bi < n_batches; ++bi) {
      TDS_CHECK_HIP(hipMemcpyAsync(m->idx, perm.data() + bi * batch, sizeof(int) * batch,
                                   hipMemcpyHostToDevice, m->stream));
      batch_pass(m, d, kind, batch);
      adam(m, lr, beta1, beta2, eps);
      // one synchronisation per batch, which also keeps the pageable index
      // upload from racing the next permutation
      double sum = 0.0;
      rc = read_loss(m, batch, &sum);
      if (rc) return rc;
      ep_loss += sum;
    }
    TDS_CHECK_HIP(hipGetLastError());
    if (epoch_loss) epoch_loss[ep] = (float)(ep_loss / n_batches);
  }
  TDS_CHECK_HIP(hipStreamSynchronize(m->stream));
  return 0;
}

}  // extern "C"
