// q-space (Bloch basis) Lanczos on the device, FP64 complex.
//
// L application of Modules/QSpaceLanczos.py (apply_full_L, QL:870-893):
// harmonic part (QL:485-576) plus the perturbed averages of
// Modules/tdscha_qspace.jl:455-628 assembled into the a'/b' blocks
// (QL:718-758), for a batch of chains that each have
// their own perturbation q-point (q_pert) and hence their own pair list and
// psi layout (QL:297-343).  The Hermitian Lanczos with full
// reorthogonalisation (QL:967-1182) runs on the device for the whole batch,
// every chain stopping at its own cap or at |b| < tol.
//
// Layouts on the device:
//   X, Y     double2 [n_q][nb][N]   Bloch components, configurations fastest
//   psi      double2 [C][ld]        chain c's vector in the reference layout,
//                                   zero-padded to the common stride ld
// Kernels of one L application:
//   q_unpack   alpha1 blocks (QL:662-716) and R1 per chain and pair
//   q_weights  per configuration and chain: buffer_u = A x_partner summed
//              into total_sum and buf_f_weight, the D3/D4 weights and the
//              f_pert contribution (JQ:489-573)
//   q_d2v      per chain, pair and configuration chunk: the d2v block as a
//              sum of two rank-1 complex products per configuration
//              (JQ:575-610)
//   q_finish   fixed-order reduction of the partials, normalisation and
//              assembly of harmonic + anharmonic parts
// Point-group images (the per-(configuration, symmetry) rotation
// x_rot = S_j x of JQ:496-502) are expanded once per context by q_expand:
// the ensemble then holds n_sym N configurations, normalised by
// n_sym N_eff (JQ:621), and every kernel above runs unchanged.
// All sums are fixed-order trees or loops: results do not depend on timing.
#include <algorithm>
#include <array>
#include <atomic>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "common.hpp"
#include "../../include/tdscha_amd.h"

namespace tdscha {

constexpr int kQMaxChains = 256;
constexpr int kQMaxQ = 512;
constexpr size_t kQKeep = 1L << 30;  // batch memory kept between calls
constexpr int kD2vChains = 15;       // chains per slab q_d2v workgroup
constexpr int kSlabBytes = 65536;    // LDS of one slab q_d2v workgroup (two buffers)
constexpr int kD2vThreads = 256;     // threads (items) per slab q_d2v workgroup
constexpr int kMmaUnits = 3584;      // entries of one LDS buffer of q_d2v_mma
constexpr int kMmaGroups = 3;        // groups of four items per wave of q_d2v_mma

struct QCtx {
  int nq = 0, nb = 0, N = 0;
  int n_sym = 1;            // point-group images expanded so far (1: none)
  double T = 0.0, neff = 0.0;
  double2* X = nullptr;     // [nq][nb][N]
  double2* Y = nullptr;
  double* rho = nullptr;    // [N]
  double* wq = nullptr;     // [nq][nb]
  double* nbose = nullptr;  // [nq][nb]
  int* valid = nullptr;     // [nq][nb]
  double* fY = nullptr;     // [nq][nb]
  double* fP = nullptr;     // [nq][nb]
  double2* S = nullptr;     // slab images of (fY X, Y) for q_d2v_slab
  int slabT = 0;            // configurations per slab (0: no slab images)
  bool mma = false;         // the slabs are q_d2v_mma's
  int d2v_form = 1;         // 1: q_d2v_slab when slab images exist, 0: q_d2v
  int n_cu = 256;           // compute units of the context's device
  // tile choices (autotuner)
  int weights_tile = 128;   // configurations per workgroup of q_weights
  int d2v_chunk = 0;        // configurations per workgroup of q_d2v (0 = automatic)
  int reorth_jtile = 16;    // basis vectors per workgroup of the reorthogonalisation dots
  hipStream_t stream = nullptr;
  // device and pinned memory of a batch, kept for the next call (as large as the
  // largest batch so far, at most kQKeep bytes each; 64 chains on 4x4x4 and 20000
  // configurations take 0.1 GB); `busy` while a batch uses it, another batch at that
  // time allocates its own
  void* work = nullptr;
  void* pinned = nullptr;
  size_t work_size = 0, pinned_size = 0;
  std::atomic<bool> busy{false};
};

// Chain tables and work buffers of one batch.
struct QBatch {
  QCtx* owner = nullptr;    // whose kept memory this batch uses
  void* mem = nullptr;      // or its own
  double2* psi = nullptr;   // [C][ld] input and output of a single application
  double2* out = nullptr;
  double2* host = nullptr;  // pinned, [C][ld] (with psi)
  int C = 0, MP = 0, maxp = 0, ld = 0, nch = 1, ntile = 1;
  std::vector<int> h_len, h_np;
  int* iqp = nullptr;       // [C]
  int* npairs = nullptr;    // [C]
  int* pq1 = nullptr;       // [C][MP]
  int* pq2 = nullptr;
  int* offa = nullptr;
  int* offb = nullptr;
  int* apair = nullptr;     // [C][nq]
  int* aorient = nullptr;   // [C][nq]
  int* active = nullptr;    // [C]
  double2* alpha = nullptr; // [C][nq][nb*nb] oriented alpha1 block of each q
  double2* R1 = nullptr;    // [C][nb]
  double2* wc = nullptr;    // [C][N]
  double2* wd = nullptr;
  double2* fpart = nullptr; // [C][ntile][nb]
  double2* dpart = nullptr; // [C][MP][nch][nb*nb]
  // slab form of q_d2v: (chain, pair, q1, q2) items sorted by chain, cut into
  // workgroups of at most kD2vThreads items and kD2vChains chains
  int slabT = 0, chunk = 0, nib = 0, n_items = 0;
  int4* items = nullptr;    // [n_items]
  int* blk_start = nullptr; // [nib + 1]
};

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 cmulcj(double2 a, double2 b) {   // a * conj(b)
  return make_double2(a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y);
}
__device__ __forceinline__ double2 cj(double2 a) { return make_double2(a.x, -a.y); }
__device__ __forceinline__ double2 cadd(double2 a, double2 b) {
  return make_double2(a.x + b.x, a.y + b.y);
}
__device__ __forceinline__ double2 csc(double2 a, double s) { return make_double2(a.x * s, a.y * s); }
// acc + a b and acc + a conj(b) as four FMAs
__device__ __forceinline__ double2 cmac(double2 acc, double2 a, double2 b) {
  acc.x = __builtin_fma(a.x, b.x, acc.x);
  acc.x = __builtin_fma(-a.y, b.y, acc.x);
  acc.y = __builtin_fma(a.x, b.y, acc.y);
  acc.y = __builtin_fma(a.y, b.x, acc.y);
  return acc;
}
__device__ __forceinline__ double2 cmacj(double2 acc, double2 a, double2 b) {
  acc.x = __builtin_fma(a.x, b.x, acc.x);
  acc.x = __builtin_fma(a.y, b.y, acc.x);
  acc.y = __builtin_fma(a.y, b.x, acc.y);
  acc.y = __builtin_fma(-a.x, b.y, acc.y);
  return acc;
}

__device__ __forceinline__ int tri_index(int i, int j, int nb) {   // i <= j
  return i * nb - i * (i - 1) / 2 + (j - i);
}

// entry (i, j) of the a' or b' block at offset off: full row-major, or the
// Hermitian fill of the row-major upper triangle (QL:345-405)
__device__ __forceinline__ double2 block_entry(const double2* psi, int off, int full, int i, int j,
                                               int nb) {
  if (full) return psi[off + i * nb + j];
  if (i <= j) return psi[off + tri_index(i, j, nb)];
  return cj(psi[off + tri_index(j, i, nb)]);
}

// chi^-, chi^+ and w1 w2 / X of one band pair (QL:604-716), zero where a
// band is masked
struct PairFac {
  double chim, chip, w2x, vm;
};
__device__ __forceinline__ PairFac pair_factors(double w1, double w2, double n1, double n2,
                                                bool v1, bool v2) {
  PairFac f;
  const bool vm = v1 && v2;
  f.vm = vm ? 1.0 : 0.0;
  if (!vm) {
    f.chim = f.chip = f.w2x = 0.0;
    return f;
  }
  const double den = 2.0 * w1 * w2;
  f.chim = (w1 - w2) * (n1 - n2) / den;
  f.chip = (w1 + w2) * (1.0 + n1 + n2) / den;
  const double X = (1.0 + 2.0 * n1) * (1.0 + 2.0 * n2) / 8.0;
  f.w2x = w1 * w2 / X;
  return f;
}

// alpha1 block of the pair that q belongs to, oriented for q (JQ:519-526):
// alq[c][q][v1][v2] = alpha[v1][v2] when q is the pair's first q-point,
// conj(alpha[v2][v1]) when it is the second.  One workgroup per (q, chain).
template <int NB>
__global__ void q_unpack(const double2* __restrict__ psi, int ld, const int* __restrict__ active,
                         const int* __restrict__ pq1, const int* __restrict__ pq2,
                         const int* __restrict__ offa, const int* __restrict__ offb, int MP,
                         int nq, const int* __restrict__ apair, const int* __restrict__ aorient,
                         const double* __restrict__ wq, const double* __restrict__ nbose,
                         const int* __restrict__ valid, int ignore_v3,
                         double2* __restrict__ alq, double2* __restrict__ R1) {
  const int c = blockIdx.y, q = blockIdx.x, t = threadIdx.x;
  if (!active[c]) return;
  const double2* ps = psi + (long)c * ld;
  if (q == 0 && t < NB) R1[c * NB + t] = ignore_v3 ? make_double2(0.0, 0.0) : ps[t];
  if (t >= NB * NB) return;
  const int p = apair[c * nq + q], o = aorient[c * nq + q];
  const int i = o ? t % NB : t / NB, j = o ? t / NB : t % NB;
  const int q1 = pq1[c * MP + p], q2 = pq2[c * MP + p];
  const int full = q1 < q2;
  const double2 a = block_entry(ps, offa[c * MP + p], full, i, j, NB);
  const double2 b = block_entry(ps, offb[c * MP + p], full, i, j, NB);
  const PairFac f = pair_factors(wq[q1 * NB + i], wq[q2 * NB + j], nbose[q1 * NB + i],
                                 nbose[q2 * NB + j], valid[q1 * NB + i], valid[q2 * NB + j]);
  const double ca = f.w2x * sqrt(-0.5 * f.chim), cb = f.w2x * sqrt(0.5 * f.chip);
  const double2 al = make_double2(ca * a.x - cb * b.x, ca * a.y - cb * b.y);
  alq[((long)c * nq + q) * NB * NB + t] = o ? cj(al) : al;
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Workgroup b of a tiled launch runs on XCD b % 8.  This maps b to (tile,
// group) so that every group of one tile runs on the same XCD, tiles
// t = 8 s + x going to XCD x in order: the groups of a tile then read its
// data through one L2.  Returns false for the padding workgroups (tile >=
// ntile) of the last round.
__device__ __forceinline__ bool xcd_tile(int b, int ngroups, int ntile, int& tile, int& group) {
  const int s = b >> 3;
  group = s % ngroups;
  tile = (s / ngroups) * 8 + (b & 7);
  return tile < ntile;
}

// One thread per configuration, one chain per workgroup.  The oriented alpha block of a
// pair's second q-point is the conjugate transpose of the first one's: each pair is
// taken once, with 24 vectors in flight and its block (the same for every thread) read
// once, from LDS, for both products,
//   bu1 = A x2, bu2 = A^H x1,   tot += 2 Re x1^H bu1,
//   bfw += fP1 y1 . conj(bu1) + fP2 y2 . conj(bu2).
// Bound by the L2 reads and their latency.  64 chains on 4x4x4 / 8 chains on 2x2x2 with
// 48 images: 1095 / 59 us with a q-point at a time, two chains a workgroup and scalar
// loads of the blocks (more than the scalar registers hold); 871 / 52 us.
template <int NB>
__global__ void __launch_bounds__(256) q_weights(
    const double2* __restrict__ X, const double2* __restrict__ Y, const double* __restrict__ rho,
    int N, int nq, const double* __restrict__ fY, const double* __restrict__ fP,
    const int* __restrict__ active, const int* __restrict__ iqp, const int* __restrict__ npairs,
    const int* __restrict__ pq1, const int* __restrict__ pq2, int MP,
    const double2* __restrict__ alq, const double2* __restrict__ R1, int C, int ntile,
    int apply_v4, double2* __restrict__ wc, double2* __restrict__ wd,
    double2* __restrict__ fpart) {
  constexpr int PB = 16;   // pairs whose blocks are in LDS at a time
  __shared__ double2 As[PB][NB * NB];
  __shared__ double red[4][2 * NB];
  int tile, c;
  if (!xcd_tile(blockIdx.x, C, ntile, tile, c)) return;
  if (!active[c]) return;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int i = tile * blockDim.x + t;
  const bool in = i < N;
  const int il = min(i, N - 1);   // (what lanes past the end sum is not used)
  double2 tot = make_double2(0.0, 0.0), bfw = tot;
  const int np = npairs[c];
  for (int p = 0; p < np; ++p) {
    if (p % PB == 0) {
      __syncthreads();
      for (int e = t; e < min(PB, np - p) * NB * NB; e += blockDim.x)
        As[e / (NB * NB)][e % (NB * NB)] =
            alq[((long)c * nq + pq1[c * MP + p + e / (NB * NB)]) * NB * NB + e % (NB * NB)];
      __syncthreads();
    }
    const int q1 = pq1[c * MP + p], q2 = pq2[c * MP + p];
    const double2* A = As[p % PB];
    double2 x1[NB], y1[NB], x2[NB], y2[NB];
#pragma unroll
    for (int v = 0; v < NB; ++v) {
      x1[v] = X[((long)q1 * NB + v) * N + il];
      x2[v] = X[((long)q2 * NB + v) * N + il];
      y1[v] = Y[((long)q1 * NB + v) * N + il];
      y2[v] = Y[((long)q2 * NB + v) * N + il];
    }
    double2 b2[NB], t1 = make_double2(0.0, 0.0);
#pragma unroll
    for (int v = 0; v < NB; ++v) b2[v] = make_double2(0.0, 0.0);
#pragma unroll
    for (int v1 = 0; v1 < NB; ++v1) {
      double2 b1 = make_double2(0.0, 0.0);
#pragma unroll
      for (int v2 = 0; v2 < NB; ++v2) {
        const double2 e = A[v1 * NB + v2];
        b1 = cmac(b1, e, x2[v2]);
        b2[v2] = cmacj(b2[v2], x1[v1], e);   // conj(A[v1][v2]) x1[v1]
      }
      t1 = cmacj(t1, b1, x1[v1]);                                  // conj(x) bu
      bfw = cmacj(bfw, csc(y1[v1], fP[q1 * NB + v1]), b1);         // conj(bu) fP y
    }
    if (q1 == q2) {
      tot = cadd(tot, t1);
    } else {
      tot.x += 2.0 * t1.x;
#pragma unroll
      for (int v = 0; v < NB; ++v) bfw = cmacj(bfw, csc(y2[v], fP[q2 * NB + v]), b2[v]);
    }
  }
  const int qp = iqp[c];
  double2 fc[NB];
#pragma unroll
  for (int v = 0; v < NB; ++v) fc[v] = make_double2(0.0, 0.0);
  if (in) {
    const double r = rho[i];
    double2 wR = make_double2(0.0, 0.0), wRf = make_double2(0.0, 0.0);
    double2 xp[NB], yp[NB];
#pragma unroll
    for (int v = 0; v < NB; ++v) {
      xp[v] = X[((long)qp * NB + v) * N + i];
      yp[v] = Y[((long)qp * NB + v) * N + i];
      const double2 r1 = R1[c * NB + v];
      wR = cadd(wR, csc(cmulcj(xp[v], r1), fY[qp * NB + v]));
      wRf = cadd(wRf, cmulcj(yp[v], r1));
    }
    wR = csc(wR, r / 3.0);
    wRf = csc(wRf, r / 3.0);
    const double2 w1 = csc(tot, -0.5 * r / 3.0);
    const double2 w2 = csc(bfw, -r / 3.0);
#pragma unroll
    for (int v = 0; v < NB; ++v)
      fc[v] = cadd(cmul(w1, yp[v]), csc(cmul(w2, xp[v]), fY[qp * NB + v]));
    if (apply_v4) {
      wR = cadd(wR, csc(tot, -r / 8.0));
      wRf = cadd(wRf, csc(bfw, -r / 4.0));
    }
    wc[(long)c * N + i] = wR;
    wd[(long)c * N + i] = wRf;
  }
  // fixed-order reduction of the f_pert contributions: waves, then the
  // workgroup's waves in order
#pragma unroll
  for (int v = 0; v < NB; ++v) {
    const double sx = wave_sum(fc[v].x), sy = wave_sum(fc[v].y);
    if (lane == 0) {
      red[wv][2 * v] = sx;
      red[wv][2 * v + 1] = sy;
    }
  }
  __syncthreads();
  if (t < NB) {
    double sx = 0.0, sy = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) {
      sx += red[w][2 * t];
      sy += red[w][2 * t + 1];
    }
    fpart[((long)c * ntile + tile) * NB + t] = make_double2(sx, sy);
  }
}

// grid (largest pair count, chains, configuration chunks); the 36 complex
// accumulators take 144 VGPRs, the cap of two waves per SIMD leaves the rest
// for the loads of one configuration
template <int NB>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) q_d2v(
    const double2* __restrict__ X, const double2* __restrict__ Y, int N,
    const double* __restrict__ fY, const int* __restrict__ active,
    const int* __restrict__ npairs, const int* __restrict__ pq1, const int* __restrict__ pq2,
    int MP, const double2* __restrict__ wc, const double2* __restrict__ wd, int chunk, int nch,
    double2* __restrict__ dpart) {
  const int p = blockIdx.x, c = blockIdx.y, ch = blockIdx.z, t = threadIdx.x;
  if (!active[c] || p >= npairs[c]) return;
  __shared__ double red[4][2 * NB * NB];
  const int q1 = pq1[c * MP + p], q2 = pq2[c * MP + p];
  double f1[NB], f2[NB];
#pragma unroll
  for (int v = 0; v < NB; ++v) {
    f1[v] = fY[q1 * NB + v];
    f2[v] = fY[q2 * NB + v];
  }
  double2 acc[NB][NB];
#pragma unroll
  for (int a = 0; a < NB; ++a)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[a][b] = make_double2(0.0, 0.0);
  const int lo = ch * chunk;
  const int hi = min(N, lo + chunk);
  for (int i = lo + t; i < hi; i += blockDim.x) {
    const double2 wci = wc[(long)c * N + i], wdi = wd[(long)c * N + i];
    double2 r11[NB], r21[NB], Q1[NB], Q2[NB];
#pragma unroll
    for (int v = 0; v < NB; ++v) {
      r11[v] = csc(X[((long)q1 * NB + v) * N + i], f1[v]);
      r21[v] = Y[((long)q1 * NB + v) * N + i];
      const double2 r12 = csc(X[((long)q2 * NB + v) * N + i], f2[v]);
      const double2 r22 = Y[((long)q2 * NB + v) * N + i];
      // -Q1 = conj(wc) r22 + conj(wd) r12 ; -Q2 = conj(wc) r12
      Q1[v] = cmac(cmul(cj(wci), r22), cj(wdi), r12);
      Q2[v] = cmul(cj(wci), r12);
    }
    // accumulates -(r11 Q1^H + r21 Q2^H); the sign is restored below
#pragma unroll
    for (int a = 0; a < NB; ++a)
#pragma unroll
      for (int b = 0; b < NB; ++b)
        acc[a][b] = cmacj(cmacj(acc[a][b], r11[a], Q1[b]), r21[a], Q2[b]);
  }
  const int lane = t & 63, wv = t >> 6;
#pragma unroll
  for (int a = 0; a < NB; ++a)
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const double sx = -wave_sum(acc[a][b].x), sy = -wave_sum(acc[a][b].y);
      if (lane == 0) {
        red[wv][2 * (a * NB + b)] = sx;
        red[wv][2 * (a * NB + b) + 1] = sy;
      }
    }
  __syncthreads();
  if (t < NB * NB) {
    const int nw = blockDim.x >> 6;
    double sx = 0.0, sy = 0.0;
    for (int w = 0; w < nw; ++w) {
      sx += red[w][2 * t];
      sy += red[w][2 * t + 1];
    }
    dpart[(((long)c * MP + p) * nch + ch) * NB * NB + t] = make_double2(sx, sy);
  }
}

// Slab images: the configurations [s T, s T + T) of slab s as one
// contiguous block of U = 2 nq SR entries, SR = NB T + 1: entry
// (h nq + q) SR + v T + j holds fY[q][v] x_{q,v} (h = 0) or y_{q,v} (h = 1)
// of configuration s T + j, zero past N; the last entry of each row is a
// zero pad that puts the rows of neighbouring q-points on different LDS
// banks.  One thread per entry.
template <int NB>
__global__ void q_slab_build(const double2* __restrict__ X, const double2* __restrict__ Y,
                             const double* __restrict__ fY, int N, int nq, int lgT, long total,
                             double2* __restrict__ S) {
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= total) return;
  const int T = 1 << lgT, SR = NB * T + 1;
  const long U = 2L * nq * SR;
  const long sl = e / U;
  const int u = (int)(e - sl * U);
  const int hq = u / SR, w = u - hq * SR;
  const int h = hq >= nq, q = h ? hq - nq : hq;
  double2 val = make_double2(0.0, 0.0);
  if (w < NB * T) {
    const int v = w >> lgT, j = w & (T - 1);
    const long cfg = sl * T + j;
    if (cfg < N) {
      const long r = (long)q * NB + v;
      val = h ? Y[r * N + cfg] : csc(X[r * N + cfg], fY[r]);
    }
  }
  S[e] = val;
}

// d2v blocks from slab images in LDS.  Workgroup (item block ib,
// configuration chunk ch) copies the slab images of its chunk, and the
// weights wc, wd of its chains for the slab's configurations, into LDS with direct global -> LDS loads into two
// buffers in turn: the copy of slab k + 1 runs while the threads accumulate
// slab k.  The two buffers are distinct arrays and each half of the unrolled
// loop names its own, so that the compiler sees that the reads of one do not
// depend on the copies into the other.  Each thread accumulates the 6x6
// block of one (chain, pair) item, in configuration order; on small grids (long
// slabs, few items) ns threads take an item, every ns-th configuration each, and
// their blocks are added in LDS at the end (6 bands, 36 items at 8 chains on 2x2x2:
// 124 us with one thread each, 61 us).  ns follows from the grid alone, so that a
// chain's sums do not depend on its batch.  The item blocks
// of one chunk run on one XCD and share the chunk through its L2.  T is known at
// compile time so that the LDS offsets are immediates (6 bands, 64 chains on 4x4x4:
// 934 us with a run-time T, 859 us).  Three bands run here on every grid, six on those
// whose slabs are too short for q_d2v_mma (more than 69 q-points).
constexpr int kSlabUnits = kSlabBytes / 2 / (int)sizeof(double2);
constexpr int d2v_slices(int T) { return T > 2 ? T / 2 : 1; }

template <int NB, int T>
__global__ void __launch_bounds__(kD2vThreads) __attribute__((amdgpu_waves_per_eu(2))) q_d2v_slab(
    const double2* __restrict__ S, int N, int nq, const int* __restrict__ active,
    const int4* __restrict__ items, const int* __restrict__ blk_start, int nib, int MP,
    const double2* __restrict__ wc, const double2* __restrict__ wd, int chunk, int nch,
    double2* __restrict__ dpart) {
  __shared__ double2 bufA[kSlabUnits], bufB[kSlabUnits];
  int ch, ib;
  if (!xcd_tile(blockIdx.x, nib, nch, ch, ib)) return;
  constexpr int SR = NB * T + 1;
  const int U = 2 * nq * SR;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, nwave = blockDim.x >> 6;
  const int i0 = blk_start[ib], i1 = blk_start[ib + 1];
  const int c_lo = items[i0].x, ncb = items[i1 - 1].x - c_lo + 1;
  bool any = false;
  for (int k = 0; k < ncb; ++k) any |= active[c_lo + k] != 0;
  if (!any) return;
  const int ni = i1 - i0;
  constexpr int ns = d2v_slices(T);
  const int sl = t / ni, at = t - sl * ni;
  int4 it = make_int4(0, 0, 0, 0);
  bool mine = sl < ns;
  if (mine) {
    it = items[i0 + at];
    mine = active[it.x] != 0;
  }
  const int cw = (it.x - c_lo) * 2 * T;
  const int nW = ncb * 2 * T;
  const int lo = ch * chunk, hi = min(N, lo + chunk);
  auto issue = [&](int s0, double2* dst) {
    const long sl = s0 / T;
    const double2* src = S + sl * U;
    for (int k = wave; k * 64 < U; k += nwave)
      if (k * 64 + lane < U) dma16(src + k * 64 + lane, dst + k * 64);
    // weights: entry (chain k, c1 | c2, configuration j) at (2 k + h) T + j;
    // past N any finite value (the image is zero there)
    for (int k = wave; k * 64 < nW; k += nwave) {
      const int e = k * 64 + lane;
      if (e < nW) {
        const int j = e % T, h = (e / T) & 1, c = c_lo + e / (2 * T);
        dma16((h ? wd : wc) + (long)c * N + min(s0 + j, N - 1), dst + U + k * 64);
      }
    }
  };
  double2 acc[NB][NB];
#pragma unroll
  for (int a = 0; a < NB; ++a)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[a][b] = make_double2(0.0, 0.0);
  auto accumulate = [&](const double2* img) {
    if (!mine) return;
    for (int j = sl; j < T; j += ns) {
      const double2 wci = img[U + cw + j], wdi = img[U + cw + T + j];
      const double2* x1 = img + it.z * SR + j;
      const double2* y1 = img + (nq + it.z) * SR + j;
      const double2* x2 = img + it.w * SR + j;
      const double2* y2 = img + (nq + it.w) * SR + j;
      double2 Q1[NB], Q2[NB];
#pragma unroll
      for (int v = 0; v < NB; ++v) {
        // -Q1 = conj(wc) r22 + conj(wd) r12, -Q2 = conj(wc) r12 with
        // r12 = fY x2 (the image holds fY x) and r22 = y2
        const double2 r12 = x2[v * T], r22 = y2[v * T];
        Q1[v] = cmac(cmul(cj(wci), r22), cj(wdi), r12);
        Q2[v] = cmul(cj(wci), r12);
      }
#pragma unroll
      for (int a = 0; a < NB; ++a) {
        const double2 r11 = x1[a * T], r21 = y1[a * T];
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[a][b] = cmacj(cmacj(acc[a][b], r11, Q1[b]), r21, Q2[b]);
      }
    }
  };
  issue(lo, bufA);
  for (int s0 = lo; s0 < hi; s0 += 2 * T) {
    TDS_WAIT_VMCNT(0);
    lds_barrier();                     // slab s0 in bufA; bufB free
    if (s0 + T < hi) issue(s0 + T, bufB);
    accumulate(bufA);
    if (s0 + T >= hi) break;
    TDS_WAIT_VMCNT(0);
    lds_barrier();                     // slab s0 + T in bufB; bufA free
    if (s0 + 2 * T < hi) issue(s0 + 2 * T, bufA);
    accumulate(bufB);
  }
  if constexpr (ns == 1) {
    if (mine) {
      double2* o = dpart + (((long)it.x * MP + it.y) * nch + ch) * NB * NB;
#pragma unroll
      for (int a = 0; a < NB; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b) o[a * NB + b] = make_double2(-acc[a][b].x, -acc[a][b].y);
    }
    return;
  }
  // one row of the blocks at a time: [slice][item][b] (ns ni <= 256 threads)
#pragma unroll
  for (int a = 0; a < NB; ++a) {
    lds_barrier();
    if (sl < ns)
#pragma unroll
      for (int b = 0; b < NB; ++b) bufA[t * NB + b] = acc[a][b];
    lds_barrier();
    for (int e = t; e < ni * NB; e += kD2vThreads) {
      const int4 w = items[i0 + e / NB];
      if (!active[w.x]) continue;
      double2 v = make_double2(0.0, 0.0);
      for (int k = 0; k < ns; ++k) v = cadd(v, bufA[k * ni * NB + e]);
      dpart[((((long)w.x * MP + w.y) * nch + ch) * NB + a) * NB + e % NB] =
          make_double2(-v.x, -v.y);
    }
  }
}

// The blocks on the FP64 matrix instructions (6 bands): as real matrices the block of
// an item is r (12 x K) times Q (K x 12), K the configurations, for each of the two
// products; a 4 x 4 x 4 instruction takes four items at once (its four blocks) and
// four configurations, nine of them the 12 x 12 entries.  The same FP64 work as a
// thread per item, but 9 accumulators instead of 72 and each operand read once per
// four lanes' worth of configurations, so that a CU has 16 waves instead of 8, no lane
// without an item but in the last group, and slabs of at least four configurations.
// Sixteen waves: `slices` of the slab's steps of four configurations (fixed by T, so
// that a chain's sums do not depend on its batch) times 16 / slices columns, groups of
// items dealt to the columns in turn.  64 chains on 4x4x4: 859 us with a thread per
// item, 708 us; 8 chains on 2x2x2 with 48 images: 61, 41 us.
constexpr int mma_slices(int T) { return T / 4; }
constexpr int mma_cap(int T) { return 16 / mma_slices(T) * kMmaGroups * 4; }

template <int T>
__global__ __launch_bounds__(1024) void q_d2v_mma(
    const double2* __restrict__ S, int N, int nq, const int* __restrict__ active,
    const int4* __restrict__ items, const int* __restrict__ blk_start, int nib, int MP,
    const double2* __restrict__ wc, const double2* __restrict__ wd, int chunk, int nch,
    double2* __restrict__ dpart) {
  constexpr int NB = 6, SR = NB * T + 1, NSL = mma_slices(T), NCOL = 16 / NSL, G = kMmaGroups;
  __shared__ double2 bufA[kMmaUnits], bufB[kMmaUnits];
  // equal numbers of workgroups on the XCDs (one fits a CU: an XCD with one too many
  // would take twice the time), the item blocks of a chunk side by side
  const int total = nib * nch, per = (total + 7) >> 3, id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (id >= total) return;
  const int ch = id / nib, ib = id - ch * nib;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int slice = wave % NSL, col = wave / NSL;
  const int i = lane & 3, blk = (lane >> 2) & 3, k = lane >> 4, sgn = i & 1;
  const int i0 = blk_start[ib], i1 = blk_start[ib + 1], ni = i1 - i0, ng = (ni + 3) / 4;
  const int c_lo = items[i0].x, ncb = items[i1 - 1].x - c_lo + 1;
  bool any = false;
  for (int c = 0; c < ncb; ++c) any |= active[c_lo + c] != 0;
  if (!any) return;
  // entries of a slab, the weights behind them, both in whole copies of 64 entries
  const int U = 2 * nq * SR, U64 = (U + 63) / 64, nW = ncb * 2 * T, W64 = (nW + 63) / 64;
  const int oy = nq * SR * 2;   // from x to y, in doubles
  int ox1[G], ox2[G], ow[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int4 it = items[i0 + min(4 * (g * NCOL + col) + blk, ni - 1)];
    const int o = ((i >> 1) * T + 4 * slice + k) * 2 + sgn;
    ox1[g] = it.z * SR * 2 + o;
    ox2[g] = it.w * SR * 2 + o;
    ow[g] = U64 * 64 + (it.x - c_lo) * 2 * T + 4 * slice + k;
  }
  const int lo = ch * chunk, hi = min(N, lo + chunk);
  // (every lane takes part in each copy; those past the end repeat the last entry)
  auto issue = [&](int s0, double2* dst) {
    const double2* src = S + (long)(s0 / T) * U;
    for (int q = wave; q < U64; q += 16) dma16(src + min(q * 64 + lane, U - 1), dst + q * 64);
    for (int q = wave; q < W64; q += 16) {
      const int e = min(q * 64 + lane, nW - 1);
      const int j = e % T, h = (e / T) & 1, c = c_lo + e / (2 * T);
      dma16((h ? wd : wc) + (long)c * N + min(s0 + j, N - 1), dst + (U64 + q) * 64);
    }
  };
  double acc[G][3][3];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = 0; b < 3; ++b) acc[g][a][b] = 0.0;
  // the other half (imaginary for real) of the complex entry: lane ^ 1
  auto other = [](double v) {
    const int a = __builtin_amdgcn_mov_dpp(__double2loint(v), 0xB1, 0xf, 0xf, true);
    const int b = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0xB1, 0xf, 0xf, true);
    return __hiloint2double(b, a);
  };
  auto accumulate = [&](const double2* img) {
    const double* d = reinterpret_cast<const double*>(img);
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (g * NCOL + col >= ng) break;
      double x1[3], y1[3], Q1[3], Q2[3];
      const double2 c1 = img[ow[g]], c2 = img[ow[g] + T];
      const double c1y = sgn ? -c1.y : c1.y, c2y = sgn ? -c2.y : c2.y;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        // -Q1 = conj(wc) r22 + conj(wd) r12, -Q2 = conj(wc) r12
        const double x = d[ox2[g] + 4 * a * T], y = d[ox2[g] + oy + 4 * a * T];
        const double xo = other(x), yo = other(y);
        Q2[a] = __builtin_fma(c1y, xo, c1.x * x);
        Q1[a] = __builtin_fma(c2y, xo,
                              __builtin_fma(c2.x, x, __builtin_fma(c1y, yo, c1.x * y)));
        x1[a] = d[ox1[g] + 4 * a * T];
        y1[a] = d[ox1[g] + oy + 4 * a * T];
      }
#pragma unroll
      for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int b = 0; b < 3; ++b) acc[g][a][b] = mfma4(x1[a], Q1[b], acc[g][a][b]);
#pragma unroll
      for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int b = 0; b < 3; ++b) acc[g][a][b] = mfma4(y1[a], Q2[b], acc[g][a][b]);
    }
  };
  issue(lo, bufA);
  for (int s0 = lo; s0 < hi; s0 += 2 * T) {
    TDS_WAIT_VMCNT(0);
    lds_barrier();                     // slab s0 in bufA; bufB free
    if (s0 + T < hi) issue(s0 + T, bufB);
    accumulate(bufA);
    if (s0 + T >= hi) break;
    TDS_WAIT_VMCNT(0);
    lds_barrier();                     // slab s0 + T in bufB; bufA free
    if (s0 + 2 * T < hi) issue(s0 + 2 * T, bufA);
    accumulate(bufB);
  }
  if constexpr (NSL > 1) {   // the slices in order, three accumulators at a time
    double* red = reinterpret_cast<double*>(bufA);   // [wave][3][64]
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        lds_barrier();
#pragma unroll
        for (int b = 0; b < 3; ++b) red[(wave * 3 + b) * 64 + lane] = acc[g][a][b];
        lds_barrier();
        if (slice == 0)
#pragma unroll
          for (int q = 1; q < NSL; ++q)
#pragma unroll
            for (int b = 0; b < 3; ++b) acc[g][a][b] += red[((wave + q) * 3 + b) * 64 + lane];
      }
    if (slice) return;
  }
  // D: column lane % 4, item lane / 4 % 4, row lane / 16: complex entry (a, b) from the
  // four real ones (2 a + s, 2 b + s')
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int at = 4 * (g * NCOL + col) + blk;
    const int4 it = items[i0 + min(at, ni - 1)];
    const bool mine = at < ni && !(lane & 17) && active[it.x] != 0;
    double2* o = dpart + (((long)it.x * MP + it.y) * nch + ch) * NB * NB;
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = 0; b < 3; ++b) {
        const double v = acc[g][a][b];
        const double re = v + __shfl_xor(v, 17), im = __shfl_xor(v, 16) - __shfl_xor(v, 1);
        if (mine) o[(2 * a + (lane >> 5)) * NB + 2 * b + ((lane >> 1) & 1)] = make_double2(-re, -im);
      }
  }
}

// Sum over k of p[k W + t], k < n, for t < W of a 256-thread workgroup: the
// entries in 256 / W slices, four loads in flight each, the slices added in LDS in
// a fixed order.
template <int W>
__device__ __forceinline__ double2 slice_sum(const double2* __restrict__ p, int n) {
  constexpr int S = 256 / W, step = S * W;
  __shared__ double2 red[step];
  const int t = threadIdx.x;
  const long end = (long)n * W;
  double2 v = make_double2(0.0, 0.0);
  if (t < step) {
    long e = t;
    for (; e + 3 * step < end; e += 4 * step) {
      double2 x[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) x[j] = p[e + j * step];
#pragma unroll
      for (int j = 0; j < 4; ++j) v = cadd(v, x[j]);
    }
    for (; e < end; e += step) v = cadd(v, p[e]);
    red[t] = v;
  }
  __syncthreads();
  v = make_double2(0.0, 0.0);
  if (t < W)
#pragma unroll 4
    for (int k = 0; k < S; ++k) v = cadd(v, red[k * W + t]);
  return v;
}

// Static Liouvillian of the free-energy Hessian (QSpaceHessian,
// Modules/QSpaceHessian.py:605-692): psi = [R, one W sector].  The input of
// the perturbed averages is alpha = -2 Y_w1 Y_w2 W (QSH:675-679; Y_w = fY),
// oriented per q-point as in q_unpack.
template <int NB>
__global__ void q_unpack_static(const double2* __restrict__ psi, int ld,
                                const int* __restrict__ active, const int* __restrict__ pq1,
                                const int* __restrict__ pq2, const int* __restrict__ offa, int MP,
                                int nq, const int* __restrict__ apair,
                                const int* __restrict__ aorient, const double* __restrict__ fY,
                                int ignore_v3, double2* __restrict__ alq,
                                double2* __restrict__ R1) {
  const int c = blockIdx.y, q = blockIdx.x, t = threadIdx.x;
  if (!active[c]) return;
  const double2* ps = psi + (long)c * ld;
  if (q == 0 && t < NB) R1[c * NB + t] = ignore_v3 ? make_double2(0.0, 0.0) : ps[t];
  if (t >= NB * NB) return;
  const int p = apair[c * nq + q], o = aorient[c * nq + q];
  const int i = o ? t % NB : t / NB, j = o ? t / NB : t % NB;
  const int q1 = pq1[c * MP + p], q2 = pq2[c * MP + p];
  const double2 w = block_entry(ps, offa[c * MP + p], q1 < q2, i, j, NB);
  const double2 al = csc(w, -2.0 * fY[q1 * NB + i] * fY[q2 * NB + j]);
  alq[((long)c * nq + q) * NB * NB + t] = o ? cj(al) : al;
}

// Static two-phonon propagator (QSH:481-544): Lambda = ((n1 + n2 + 1) /
// (w1 + w2) - dn) / (4 w1 w2), dn = (n1 - n2) / (w1 - w2), or
// -beta e^{beta w} n^2 when |w1 - w2| < 1e-8; zero unless both modes count.
__device__ __forceinline__ double static_lambda(double w1, double w2, double n1, double n2,
                                                bool v1, bool v2, double beta) {
  if (!(v1 && v2)) return 0.0;
  double dn = 0.0;
  if (beta > 0.0) {
    if (fabs(w1 - w2) < 1e-8)
      dn = -beta * exp(w1 * beta) * n1 * n1;
    else
      dn = (n1 - n2) / (w1 - w2);
  }
  return ((n1 + n2 + 1.0) / (w1 + w2) - dn) / (4.0 * w1 * w2);
}

// R <- w^2 R - f_pert, W <- W / Lambda + d2v (QSH:605-692).  Block 0: R
// sector; block 1 + p: the W block of pair p.
template <int NB>
__global__ void __launch_bounds__(256) q_finish_static(const double2* __restrict__ psi, int ld, double2* __restrict__ out,
                                const int* __restrict__ active, const int* __restrict__ iqp,
                                const int* __restrict__ npairs, const int* __restrict__ pq1,
                                const int* __restrict__ pq2, const int* __restrict__ offa, int MP,
                                const double* __restrict__ wq, const double* __restrict__ nbose,
                                const int* __restrict__ valid, double beta,
                                const double2* __restrict__ fpart, int ntile,
                                const double2* __restrict__ dpart, int nch, double inv_norm,
                                int do_harm, int do_anh) {
  const int c = blockIdx.y, blk = blockIdx.x, t = threadIdx.x;
  if (!active[c]) return;
  const double2* ps = psi + (long)c * ld;
  double2* po = out + (long)c * ld;
  if (blk == 0) {
    const double2 f = slice_sum<NB>(fpart + (long)c * ntile * NB, do_anh ? ntile : 0);
    if (t >= NB) return;
    const int qp = iqp[c];
    double2 o = make_double2(0.0, 0.0);
    if (do_anh) o = csc(f, -inv_norm);
    if (do_harm) {
      const double w = wq[qp * NB + t];
      o = cadd(o, csc(ps[t], w * w));
    }
    po[t] = o;
    return;
  }
  const int p = blk - 1;
  if (p >= npairs[c]) return;
  double2 d = slice_sum<NB * NB>(dpart + ((long)c * MP + p) * nch * NB * NB, do_anh ? nch : 0);
  if (t >= NB * NB) return;
  const int i = t / NB, j = t % NB;
  const int q1 = pq1[c * MP + p], q2 = pq2[c * MP + p];
  const int full = q1 < q2;
  if (!full && i > j) return;
  const int e = offa[c * MP + p] + (full ? i * NB + j : tri_index(i, j, NB));
  double2 o = make_double2(0.0, 0.0);
  if (do_anh) o = csc(d, inv_norm);
  if (do_harm) {
    const double lam = static_lambda(wq[q1 * NB + i], wq[q2 * NB + j], nbose[q1 * NB + i],
                                     nbose[q2 * NB + j], valid[q1 * NB + i], valid[q2 * NB + j],
                                     beta);
    if (fabs(lam) > 1e-30) o = cadd(o, csc(ps[e], 1.0 / lam));
  }
  po[e] = o;
}

// block 0: R sector; block 1 + p: pair p.  A chain of dependent loads per entry when
// one thread adds the partials (125 us at 8 chains on 2x2x2 with 375 of them); 8 us
// in slices.
template <int NB>
__global__ void __launch_bounds__(256) q_finish(const double2* __restrict__ psi, int ld, double2* __restrict__ out,
                         const int* __restrict__ active, const int* __restrict__ iqp,
                         const int* __restrict__ npairs, const int* __restrict__ pq1,
                         const int* __restrict__ pq2, const int* __restrict__ offa,
                         const int* __restrict__ offb, int MP, const double* __restrict__ wq,
                         const double* __restrict__ nbose, const int* __restrict__ valid,
                         const double2* __restrict__ fpart, int ntile,
                         const double2* __restrict__ dpart, int nch, double inv_norm,
                         int do_harm, int do_anh) {
  const int c = blockIdx.y, blk = blockIdx.x, t = threadIdx.x;
  if (!active[c]) return;
  const double2* ps = psi + (long)c * ld;
  double2* po = out + (long)c * ld;
  if (blk == 0) {
    const double2 f = slice_sum<NB>(fpart + (long)c * ntile * NB, do_anh ? ntile : 0);
    if (t >= NB) return;
    const int qp = iqp[c];
    double2 o = make_double2(0.0, 0.0);
    if (do_anh) o = csc(f, inv_norm);
    if (do_harm && valid[qp * NB + t]) {
      const double w = wq[qp * NB + t];
      o = cadd(o, csc(ps[t], -w * w));
    }
    po[t] = o;
    return;
  }
  const int p = blk - 1;
  if (p >= npairs[c]) return;
  double2 d = slice_sum<NB * NB>(dpart + ((long)c * MP + p) * nch * NB * NB, do_anh ? nch : 0);
  if (t >= NB * NB) return;
  const int i = t / NB, j = t % NB;
  const int q1 = pq1[c * MP + p], q2 = pq2[c * MP + p];
  const int full = q1 < q2;
  if (!full && i > j) return;
  const int e = full ? i * NB + j : tri_index(i, j, NB);
  const int ea = offa[c * MP + p] + e, eb = offb[c * MP + p] + e;
  const double w1 = wq[q1 * NB + i], w2 = wq[q2 * NB + j];
  const PairFac f = pair_factors(w1, w2, nbose[q1 * NB + i], nbose[q2 * NB + j],
                                 valid[q1 * NB + i], valid[q2 * NB + j]);
  double2 oa = make_double2(0.0, 0.0), ob = make_double2(0.0, 0.0);
  if (do_anh) {
    d = csc(d, inv_norm);
    oa = csc(d, sqrt(-0.5 * f.chim));
    ob = csc(d, -sqrt(0.5 * f.chip));
  }
  if (do_harm) {
    oa = cadd(oa, csc(ps[ea], -(w1 - w2) * (w1 - w2) * f.vm));
    ob = cadd(ob, csc(ps[eb], -(w1 + w2) * (w1 + w2) * f.vm));
  }
  po[ea] = oa;
  po[eb] = ob;
}

// Images of every configuration under every symmetry: image j N + i of
// q-point perm[j][p] is D[j][p] x_i[p] (JQ:496-502).  Grid
// (ceil(N / 256), n_sym, n_q), configurations fastest on both sides.
template <int NB>
__global__ void q_expand(const double2* __restrict__ X, const double2* __restrict__ Y, int N,
                         int nq, const int* __restrict__ perm, const double2* __restrict__ D,
                         double2* __restrict__ XE, double2* __restrict__ YE) {
  const int p = blockIdx.z, j = blockIdx.y;
  __shared__ double2 d[NB * NB];
  for (int e = threadIdx.x; e < NB * NB; e += blockDim.x)
    d[e] = D[((long)j * nq + p) * NB * NB + e];
  __syncthreads();
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  const int q = perm[(long)j * nq + p];
  const long NE = (long)N * gridDim.y;
  double2 x[NB], y[NB];
#pragma unroll
  for (int m = 0; m < NB; ++m) {
    x[m] = X[((long)p * NB + m) * N + i];
    y[m] = Y[((long)p * NB + m) * N + i];
  }
#pragma unroll
  for (int v = 0; v < NB; ++v) {
    double2 sx = make_double2(0.0, 0.0), sy = make_double2(0.0, 0.0);
#pragma unroll
    for (int m = 0; m < NB; ++m) {
      sx = cadd(sx, cmul(d[v * NB + m], x[m]));
      sy = cadd(sy, cmul(d[v * NB + m], y[m]));
    }
    XE[((long)q * NB + v) * NE + (long)j * N + i] = sx;
    YE[((long)q * NB + v) * NE + (long)j * N + i] = sy;
  }
}

// ------------------------------------------------------------ batch setup
static void free_batch(QBatch& b) {
  if (b.owner) {
    QCtx* q = b.owner;
    (void)hipStreamSynchronize(q->stream);   // (a failed run may still use it)
    if (q->work_size > kQKeep) {
      (void)hipFree(q->work);
      q->work = nullptr;
      q->work_size = 0;
    }
    if (q->pinned_size > kQKeep) {
      (void)hipHostFree(q->pinned);
      q->pinned = nullptr;
      q->pinned_size = 0;
    }
    q->busy.store(false, std::memory_order_release);
  } else {
    if (b.mem) (void)hipFree(b.mem);
    if (b.host) (void)hipHostFree(b.host);
  }
  b = QBatch();
}

// device memory of `size` bytes and pinned memory of `host` bytes for a batch: the
// context's, if no other batch has it, else its own
static bool take_memory(QCtx* q, size_t size, size_t host, QBatch& b) {
  void *mem = nullptr, *pin = nullptr;
  if (!q->busy.exchange(true, std::memory_order_acquire)) {
    b.owner = q;
    if (q->work_size < size) {
      if (q->work) (void)hipFree(q->work);
      q->work_size = 0;
      q->work = nullptr;
      if (hipMalloc(&q->work, size) != hipSuccess) {
        q->work = nullptr;
        return false;
      }
      q->work_size = size;
    }
    if (q->pinned_size < host) {
      if (q->pinned) (void)hipHostFree(q->pinned);
      q->pinned_size = 0;
      q->pinned = nullptr;
      if (hipHostMalloc(&q->pinned, host) != hipSuccess) {
        q->pinned = nullptr;
        return false;
      }
      q->pinned_size = host;
    }
    mem = q->work;
    pin = q->pinned;
  } else {
    if (hipMalloc(&mem, size) != hipSuccess) return false;
    if (host && hipHostMalloc(&pin, host) != hipSuccess) {
      (void)hipFree(mem);
      return false;
    }
  }
  b.mem = mem;
  b.host = host ? static_cast<double2*>(pin) : nullptr;
  return true;
}

static int choose_chunk(const QCtx* q, int C, int MP_used) {
  if (q->d2v_chunk > 0) return q->d2v_chunk;
  // aim at ~2048 workgroups in total, at least 1024 configurations each
  long blocks = (long)C * std::max(1, MP_used);
  long nch = std::max(1L, 2048 / std::max(1L, blocks));
  int chunk = (int)((q->N + nch - 1) / nch);
  return std::max(chunk, std::min(q->N, 1024));
}

// Configurations per slab of the slab q_d2v: the largest power of two up to
// 16 whose slab image and the weights of kD2vChains chains fit one of its
// two LDS buffers (kSlabBytes / 2); 0 when one configuration does not fit.
static size_t slab_units(int nq, int nb, int T) {
  return 2 * (size_t)nq * (nb * T + 1) + 2 * (size_t)kD2vChains * T;
}

// (6 bands: grids whose slabs hold 4 configurations or more run q_d2v_mma)
template <int NB, typename Fn>
static void with_slab(int T, Fn fn) {
  if (T == 1) fn(std::integral_constant<int, 1>{});
  if (T == 2) fn(std::integral_constant<int, 2>{});
  if constexpr (NB != 6) {
    if (T == 4) fn(std::integral_constant<int, 4>{});
    if (T == 8) fn(std::integral_constant<int, 8>{});
    if (T == 16) fn(std::integral_constant<int, 16>{});
  }
}

static int log2_pow2(int T) {
  int lg = 0;
  while ((1 << lg) < T) ++lg;
  return lg;
}

static int slab_configs(int nq, int nb, bool* mma) {
  // q_d2v_mma: 16, 8 or 4 configurations, whole copies of 64 entries
  *mma = false;
  if (nb == 6)
    for (int T = 16; T >= 4; T >>= 1)
      if ((2 * nq * (6 * T + 1) + 63) / 64 * 64 + (2 * kD2vChains * T + 63) / 64 * 64 <= kMmaUnits) {
        *mma = true;
        return T;
      }
  int T = 16;
  while (T > 0 && slab_units(nq, nb, T) * sizeof(double2) > (size_t)kSlabBytes / 2) T >>= 1;
  return T;
}

// (Re)builds the slab images of the context's ensemble; without room for
// one configuration per slab the context keeps none and q_d2v runs instead.
static int build_slabs(QCtx* q) {
  if (q->S) (void)hipFree(q->S);
  q->S = nullptr;
  q->slabT = slab_configs(q->nq, q->nb, &q->mma);
  if (!q->slabT) return 0;
  const int lg = log2_pow2(q->slabT);
  const long nslab = (q->N + q->slabT - 1) / q->slabT;
  const long total = nslab * 2L * q->nq * (q->nb * q->slabT + 1);
  if (hipMalloc((void**)&q->S, sizeof(double2) * (size_t)total) != hipSuccess) {
    q->S = nullptr;
    set_error("q-space: allocation of the slab images failed");
    return -1;
  }
  const unsigned nblk = (unsigned)((total + 255) / 256);
  if (q->nb == 6)
    hipLaunchKernelGGL(q_slab_build<6>, dim3(nblk), dim3(256), 0, q->stream, q->X, q->Y, q->fY,
                       q->N, q->nq, lg, total, q->S);
  else
    hipLaunchKernelGGL(q_slab_build<3>, dim3(nblk), dim3(256), 0, q->stream, q->X, q->Y, q->fY,
                       q->N, q->nq, lg, total, q->S);
  if (hipGetLastError() != hipSuccess || hipStreamSynchronize(q->stream) != hipSuccess) {
    set_error("q-space: slab image kernel failed");
    return -1;
  }
  return 0;
}

// d2v chunk (configurations per workgroup) that gives `rounds` rounds of
// slab workgroups on the device (n_item_blocks workgroups per chunk, two
// resident workgroups per CU: two buffers of half the CU's LDS and 256
// threads at up to 256 VGPRs), at least 4 slabs.
static int slab_chunk(const QCtx* q, int n_item_blocks, int rounds) {
  const long slots = (q->mma ? 1L : 2L) * q->n_cu * rounds;
  const long nch = std::max(1L, slots / std::max(1, n_item_blocks));
  const long chunk = std::max<long>(4L * q->slabT, (q->N + nch - 1) / nch);
  return (int)((chunk + q->slabT - 1) / q->slabT * q->slabT);
}

// Host tables from the pair maps; ld_min forces a minimum stride.
static int build_batch(QCtx* q, int C, const int* iq_pert, const int* pair_map, QBatch& b,
                       int ld_min = 0, bool static_layout = false, bool with_psi = false) {
  const int nq = q->nq, nb = q->nb;
  b.C = C;
  b.MP = nq;
  std::vector<int> h_iqp(C), h_np(C), h_pq1((size_t)C * nq, 0), h_pq2((size_t)C * nq, 0),
      h_offa((size_t)C * nq, 0), h_offb((size_t)C * nq, 0),
      h_apair((size_t)C * nq), h_orient((size_t)C * nq), h_len(C);
  int maxp = 0;
  for (int c = 0; c < C; ++c) {
    TDS_REQUIRE(iq_pert[c] >= 0 && iq_pert[c] < nq, 2, "q-space: iq_pert out of range");
    const int* pm = pair_map + (long)c * nq;
    for (int i = 0; i < nq; ++i) {
      TDS_REQUIRE(pm[i] >= 0 && pm[i] < nq && pm[pm[i]] == i, 2,
                  "q-space: q_pair_map must be an involution on [0, n_q)");
    }
    h_iqp[c] = iq_pert[c];
    int np = 0;
    for (int i = 0; i < nq; ++i)
      if (i <= pm[i]) {
        h_pq1[(size_t)c * nq + np] = i;
        h_pq2[(size_t)c * nq + np] = pm[i];
        h_apair[(size_t)c * nq + i] = np;
        h_orient[(size_t)c * nq + i] = 0;
        if (pm[i] != i) {
          h_apair[(size_t)c * nq + pm[i]] = np;
          h_orient[(size_t)c * nq + pm[i]] = 1;
        }
        ++np;
      }
    int off = nb;
    for (int p = 0; p < np; ++p) {
      h_offa[(size_t)c * nq + p] = off;
      off += h_pq1[(size_t)c * nq + p] < h_pq2[(size_t)c * nq + p] ? nb * nb : nb * (nb + 1) / 2;
    }
    for (int p = 0; p < np; ++p) {     // the static layout has no b' sector
      h_offb[(size_t)c * nq + p] = static_layout ? h_offa[(size_t)c * nq + p] : off;
      if (!static_layout)
        off += h_pq1[(size_t)c * nq + p] < h_pq2[(size_t)c * nq + p] ? nb * nb : nb * (nb + 1) / 2;
    }
    h_np[c] = np;
    h_len[c] = off;
    maxp = std::max(maxp, np);
  }
  int ld = ld_min;
  for (int c = 0; c < C; ++c) ld = std::max(ld, h_len[c]);
  b.ld = ld;
  b.h_len = h_len;
  b.h_np = h_np;
  b.ntile = (q->N + q->weights_tile - 1) / q->weights_tile;
  b.maxp = maxp;
  // slab items and their workgroups
  std::vector<int4> h_items;
  std::vector<int> h_bs(1, 0);
  b.slabT = q->S && q->d2v_form ? q->slabT : 0;
  if (b.slabT) {
    // items sorted by chain, cut at `cap` items or kD2vChains chains
    auto partition = [&](int cap) {
      h_items.clear();
      h_bs.assign(1, 0);
      int first_c = -1;
      for (int c = 0; c < C; ++c)
        for (int p = 0; p < h_np[c]; ++p) {
          const int cur = (int)h_items.size() - h_bs.back();
          if (cur == cap || (cur > 0 && c - first_c >= kD2vChains))
            h_bs.push_back((int)h_items.size());
          if ((int)h_items.size() == h_bs.back()) first_c = c;
          h_items.push_back(make_int4(c, p, h_pq1[(size_t)c * nq + p], h_pq2[(size_t)c * nq + p]));
        }
      h_bs.push_back((int)h_items.size());
    };
    partition(q->mma ? mma_cap(b.slabT) : kD2vThreads / d2v_slices(b.slabT));
    const int nfull = (int)h_bs.size() - 1;      // then the same count of even workgroups
    partition(((int)h_items.size() + nfull - 1) / nfull);
    b.n_items = (int)h_items.size();
    b.nib = (int)h_bs.size() - 1;
  }
  int chunk;
  if (b.slabT) {
    // automatic: one round of workgroups on the device's CUs
    chunk = q->d2v_chunk > 0 ? q->d2v_chunk : slab_chunk(q, b.nib, 1);
    chunk = (chunk + b.slabT - 1) / b.slabT * b.slabT;
  } else {
    chunk = choose_chunk(q, C, maxp);
  }
  b.nch = (q->N + chunk - 1) / chunk;
  b.chunk = chunk;
  const size_t nbb = (size_t)nb * nb;
  // one allocation; the tables first, uploaded by one copy
  Carve carve;
  std::vector<std::pair<const void*, size_t>> tables;
  auto table = [&](auto** p, const auto& v) {
    carve.add(p, v.size());
    tables.push_back({v.data(), sizeof(v[0]) * v.size()});
  };
  const std::vector<int> ones(C, 1);
  table(&b.iqp, h_iqp);
  table(&b.npairs, h_np);
  table(&b.pq1, h_pq1);
  table(&b.pq2, h_pq2);
  table(&b.offa, h_offa);
  table(&b.offb, h_offb);
  table(&b.apair, h_apair);
  table(&b.aorient, h_orient);
  table(&b.active, ones);
  if (b.slabT) {
    table(&b.items, h_items);
    table(&b.blk_start, h_bs);
  }
  std::vector<char> packed(carve.total());
  carve.add(&b.alpha, (size_t)C * nq * nbb);
  carve.add(&b.R1, (size_t)C * nb);
  carve.add(&b.wc, (size_t)C * q->N);
  carve.add(&b.wd, (size_t)C * q->N);
  carve.add(&b.fpart, (size_t)C * b.ntile * nb);
  carve.add(&b.dpart, (size_t)C * nq * b.nch * nbb);
  if (with_psi) {
    carve.add(&b.psi, (size_t)C * b.ld);
    carve.add(&b.out, (size_t)C * b.ld);
  }
  if (!take_memory(q, carve.total(), with_psi ? sizeof(double2) * C * b.ld : 0, b)) {
    free_batch(b);
    set_error("q-space: device allocation failed");
    return -1;
  }
  carve.assign(b.mem);
  size_t at = 0;
  for (const auto& t : tables) {
    std::memcpy(packed.data() + at, t.first, t.second);
    at += (t.second + 255) / 256 * 256;
  }
  const bool ok =
      hipMemcpy(b.mem, packed.data(), packed.size(), hipMemcpyHostToDevice) == hipSuccess;
  if (!ok) {
    free_batch(b);
    set_error("q-space: table upload failed");
    return -1;
  }
  return 0;
}

template <int NB>
static void launch_L_nb(QCtx* q, QBatch& b, const double2* psi, double2* out, int ignore_harmonic,
                        int ignore_v3, int ignore_v4, hipStream_t s, bool static_op) {
  const int C = b.C, MP = b.MP, nq = q->nq;
  const int do_anh = !(ignore_v3 && ignore_v4);
  if (do_anh) {
    if (static_op)
      hipLaunchKernelGGL(q_unpack_static<NB>, dim3(nq, C), dim3(64), 0, s, psi, b.ld, b.active,
                         b.pq1, b.pq2, b.offa, MP, nq, b.apair, b.aorient, q->fY, ignore_v3,
                         b.alpha, b.R1);
    else
      hipLaunchKernelGGL(q_unpack<NB>, dim3(nq, C), dim3(64), 0, s, psi, b.ld, b.active, b.pq1,
                         b.pq2, b.offa, b.offb, MP, nq, b.apair, b.aorient, q->wq, q->nbose,
                         q->valid, ignore_v3, b.alpha, b.R1);
    hipLaunchKernelGGL(q_weights<NB>, dim3((b.ntile + 7) / 8 * 8 * C), dim3(q->weights_tile), 0, s,
                       q->X, q->Y, q->rho, q->N, nq, q->fY, q->fP, b.active, b.iqp, b.npairs,
                       b.pq1, b.pq2, MP, b.alpha, b.R1, C, b.ntile, ignore_v4 ? 0 : 1, b.wc, b.wd,
                       b.fpart);
    if (b.slabT) {
      const int nblk2 = q->mma ? (b.nch * b.nib + 7) / 8 * 8 : (b.nch + 7) / 8 * 8 * b.nib;
      auto run = [&](auto kernel, int threads) {
        hipLaunchKernelGGL(kernel, dim3(nblk2), dim3(threads), 0, s, q->S, q->N, nq, b.active,
                           b.items, b.blk_start, b.nib, MP, b.wc, b.wd, b.chunk, b.nch, b.dpart);
      };
      if (q->mma)
        run(b.slabT == 16 ? q_d2v_mma<16> : b.slabT == 8 ? q_d2v_mma<8> : q_d2v_mma<4>, 1024);
      else
        with_slab<NB>(b.slabT, [&](auto T) { run(q_d2v_slab<NB, decltype(T)::value>, kD2vThreads); });
    } else {
      hipLaunchKernelGGL(q_d2v<NB>, dim3(b.maxp, C, b.nch), dim3(256), 0, s, q->X, q->Y, q->N,
                         q->fY, b.active, b.npairs, b.pq1, b.pq2, MP, b.wc, b.wd, b.chunk, b.nch,
                         b.dpart);
    }
  }
  if (static_op)
    hipLaunchKernelGGL(q_finish_static<NB>, dim3(MP + 1, C), dim3(256), 0, s, psi, b.ld, out,
                       b.active, b.iqp, b.npairs, b.pq1, b.pq2, b.offa, MP, q->wq, q->nbose,
                       q->valid, q->T > 1e-12 ? RY_TO_K / q->T : 0.0, b.fpart, b.ntile, b.dpart,
                       b.nch, 1.0 / q->neff, ignore_harmonic ? 0 : 1, do_anh);
  else
    hipLaunchKernelGGL(q_finish<NB>, dim3(MP + 1, C), dim3(256), 0, s, psi, b.ld, out, b.active,
                       b.iqp, b.npairs, b.pq1, b.pq2, b.offa, b.offb, MP, q->wq, q->nbose,
                       q->valid, b.fpart, b.ntile, b.dpart, b.nch, 1.0 / q->neff,
                       ignore_harmonic ? 0 : 1, do_anh);
}

static void launch_L(QCtx* q, QBatch& b, const double2* psi, double2* out, int ih, int i3, int i4,
                     hipStream_t s, bool static_op = false) {
  if (q->nb == 6)
    launch_L_nb<6>(q, b, psi, out, ih, i3, i4, s, static_op);
  else
    launch_L_nb<3>(q, b, psi, out, ih, i3, i4, s, static_op);
}

// ------------------------------------------------------- Hermitian Lanczos
struct QLanczos {
  int kmax = 0;
  void* mem = nullptr;      // the arrays below
  double2* Q = nullptr;     // [C][kmax+1][ld]
  double2* qcur = nullptr;  // [C][ld]
  double2* Lq = nullptr;
  double2* r = nullptr;
  double* mask = nullptr;   // [C][ld]
  double* coef = nullptr;   // [C][kmax+1]
  double* a = nullptr;      // [C][kmax]
  double* bb = nullptr;
  double* cc = nullptr;
  double* scal = nullptr;   // [C][4]: a_k, b_k^2, |q'|^2
  int* k = nullptr;
  int* cont = nullptr;
  int* nextc = nullptr;
  int* cap = nullptr;
  int* ndone = nullptr;
};

static void free_ql(QLanczos& l) {
  if (l.mem) (void)hipFree(l.mem);
  l = QLanczos();
}

// Re <x_c, y_c>_M, one workgroup per chain (vectors of a few thousand entries)
__global__ void __launch_bounds__(256) ql_dot(const double2* __restrict__ x,
                                              const double2* __restrict__ y,
                                              const double* __restrict__ mask, int ld,
                                              const int* __restrict__ flag,
                                              double* __restrict__ scal, int slot) {
  const int c = blockIdx.x, t = threadIdx.x;
  if (!flag[c]) return;
  const double2* xc = x + (long)c * ld;
  const double2* yc = y + (long)c * ld;
  const double* mc = mask + (long)c * ld;
  double s = 0.0;
  for (int e = t; e < ld; e += blockDim.x) s += mc[e] * (xc[e].x * yc[e].x + xc[e].y * yc[e].y);
  __shared__ double red[4];
  s = wave_sum(s);
  if ((t & 63) == 0) red[t >> 6] = s;
  __syncthreads();
  if (t == 0) scal[c * 4 + slot] = red[0] + red[1] + red[2] + red[3];
}

__global__ void ql_init(const double2* __restrict__ psi0, int ld, int kmax,
                        const double* __restrict__ scal, double2* __restrict__ Q,
                        double2* __restrict__ qcur) {
  const int c = blockIdx.y;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= ld) return;
  const double nrm = sqrt(scal[c * 4 + 2]);
  const double2 v = csc(psi0[(long)c * ld + e], 1.0 / nrm);
  Q[(long)c * (kmax + 1) * ld + e] = v;
  qcur[(long)c * ld + e] = v;
}

// r = L q_k - a_k q_k - c_{k-1} q_{k-1}
__global__ void ql_residual(const double2* __restrict__ Lq, const double2* __restrict__ qcur,
                            const double2* __restrict__ Q, int ld, int kmax,
                            const int* __restrict__ active, const int* __restrict__ kk,
                            const double* __restrict__ scal, const double* __restrict__ cc,
                            double* __restrict__ a, double2* __restrict__ r) {
  const int c = blockIdx.y;
  if (!active[c]) return;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  const int k = kk[c];
  const double ak = scal[c * 4 + 0];
  if (e == 0) a[c * kmax + k] = ak;
  if (e >= ld) return;
  const long o = (long)c * ld + e;
  double2 v = make_double2(Lq[o].x - ak * qcur[o].x, Lq[o].y - ak * qcur[o].y);
  if (k > 0) {
    const double cp = cc[c * kmax + k - 1];
    const double2 qm = Q[((long)c * (kmax + 1) + k - 1) * ld + e];
    v.x -= cp * qm.x;
    v.y -= cp * qm.y;
  }
  r[o] = v;
}

// stop tests of QL:1083-1095 and the step cap
__global__ void ql_decide(int C, int kmax, double tol, int* __restrict__ active,
                          int* __restrict__ cont, const int* __restrict__ nextc,
                          const int* __restrict__ kk, const int* __restrict__ cap,
                          int* __restrict__ ndone, const double* __restrict__ scal,
                          double* __restrict__ bb, double* __restrict__ cc) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= C) return;
  cont[c] = 0;
  if (!active[c]) return;
  const int k = kk[c];
  const double b = sqrt(scal[c * 4 + 1]);
  ndone[c] = k + 1;
  const bool conv = !(fabs(b) >= tol) || nextc[c];
  if (conv) {
    active[c] = 0;
    return;
  }
  bb[c * kmax + k] = b;
  cc[c * kmax + k] = b;     // c_k = Re<r/b, r/b> b = b for the Hermitian chain
  if (k + 1 >= cap[c]) {
    active[c] = 0;
    return;
  }
  cont[c] = 1;
}

__global__ void ql_scale(int ld, const int* __restrict__ cont, const double* __restrict__ scal,
                         double2* __restrict__ r) {
  const int c = blockIdx.y;
  if (!cont[c]) return;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= ld) return;
  const double inv = 1.0 / sqrt(scal[c * 4 + 1]);
  r[(long)c * ld + e] = csc(r[(long)c * ld + e], inv);
}

// coef_j = Re <Q_j, r>_M for j <= k, JT basis vectors per workgroup
template <int JT>
__global__ void __launch_bounds__(256) ql_rdots(const double2* __restrict__ Q,
                                                const double2* __restrict__ r,
                                                const double* __restrict__ mask, int ld, int kmax,
                                                const int* __restrict__ cont,
                                                const int* __restrict__ kk,
                                                double* __restrict__ coef) {
  const int c = blockIdx.x, jt = blockIdx.y, t = threadIdx.x;
  if (!cont[c]) return;
  const int k = kk[c];
  const int j0 = jt * JT;
  if (j0 > k) return;
  const int nj = min(JT, k + 1 - j0);
  double s[JT];
#pragma unroll
  for (int j = 0; j < JT; ++j) s[j] = 0.0;
  const double2* rc = r + (long)c * ld;
  const double* mc = mask + (long)c * ld;
  const double2* Qc = Q + ((long)c * (kmax + 1) + j0) * ld;
  for (int e = t; e < ld; e += blockDim.x) {
    const double2 re = rc[e];
    const double m = mc[e];
#pragma unroll
    for (int j = 0; j < JT; ++j)
      if (j < nj) {
        const double2 qv = Qc[(long)j * ld + e];
        s[j] += m * (qv.x * re.x + qv.y * re.y);
      }
  }
  __shared__ double red[4][JT];
#pragma unroll
  for (int j = 0; j < JT; ++j) {
    const double v = wave_sum(s[j]);
    if ((t & 63) == 0) red[t >> 6][j] = v;
  }
  __syncthreads();
  if (t < nj) coef[c * (kmax + 1) + j0 + t] = red[0][t] + red[1][t] + red[2][t] + red[3][t];
}

__global__ void ql_rupdate(const double2* __restrict__ Q, const double* __restrict__ coef,
                           int ld, int kmax, const int* __restrict__ cont,
                           const int* __restrict__ kk, double2* __restrict__ r) {
  const int c = blockIdx.y;
  if (!cont[c]) return;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= ld) return;
  const int k = kk[c];
  const double2* Qc = Q + (long)c * (kmax + 1) * ld + e;
  const double* cf = coef + c * (kmax + 1);
  double2 v = r[(long)c * ld + e];
  for (int j = 0; j <= k; ++j) {
    const double2 qv = Qc[(long)j * ld];
    v.x -= cf[j] * qv.x;
    v.y -= cf[j] * qv.y;
  }
  r[(long)c * ld + e] = v;
}

__global__ void ql_store(int ld, int kmax, double tol, const int* __restrict__ cont,
                         const int* __restrict__ kk, const double* __restrict__ scal,
                         int* __restrict__ nextc, const double2* __restrict__ r,
                         double2* __restrict__ Q, double2* __restrict__ qcur) {
  const int c = blockIdx.y;
  if (!cont[c]) return;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  const int k = kk[c];
  const double nrm = sqrt(scal[c * 4 + 2]);
  const bool small = !(nrm >= tol);
  if (e == 0) nextc[c] = small ? 1 : 0;
  if (e >= ld) return;
  const double2 v = small ? r[(long)c * ld + e] : csc(r[(long)c * ld + e], 1.0 / nrm);
  Q[((long)c * (kmax + 1) + k + 1) * ld + e] = v;
  qcur[(long)c * ld + e] = v;
}

__global__ void ql_advance(int C, const int* __restrict__ cont, int* __restrict__ kk) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c < C && cont[c]) kk[c] += 1;
}

__global__ void q_fill_int(int* p, int n, int v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

template <int JT>
static void reorth_pass(QLanczos& l, QBatch& b, hipStream_t s) {
  const int ld = b.ld, C = b.C;
  hipLaunchKernelGGL(ql_rdots<JT>, dim3(C, (l.kmax + JT) / JT), dim3(256), 0, s, l.Q, l.r, l.mask,
                     ld, l.kmax, l.cont, l.k, l.coef);
  hipLaunchKernelGGL(ql_rupdate, dim3((ld + 255) / 256, C), dim3(256), 0, s, l.Q, l.coef, ld,
                     l.kmax, l.cont, l.k, l.r);
}

// The recurrence of one step for a short chain (ld <= 1024 kQShortE) in one
// work-group per chain: everything from a_k to the next vector, with r in registers,
// its masked copy and the coefficients in LDS and the basis from L2.  As separate
// kernels the step is eleven launches of about 4.7 us each: 250 us per step with the
// L application for 8 chains on 2x2x2, 200 us here.  The line against the separate
// kernels is the one of the mode-space recurrence (kQShortWork doubles of the basis).
constexpr int kQShortE = 3;
constexpr int kQShortBasis = 1024;
constexpr long kQShortWork = 300000;

__global__ __launch_bounds__(1024) void ql_short(
    const double2* __restrict__ Lq, const double* __restrict__ mask, int ld, int kmax, double tol,
    int* __restrict__ active, int* __restrict__ nextc, int* __restrict__ kk,
    const int* __restrict__ cap, int* __restrict__ ndone, double* __restrict__ a,
    double* __restrict__ bb, double* __restrict__ cc, double2* Qall, double2* qall) {
  const int c = blockIdx.x, t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int nt = blockDim.x, nw = nt >> 6;
  if (!active[c]) return;
  const int k = kk[c];
  __shared__ double2 rm[1024 * kQShortE];
  __shared__ double coef[kQShortBasis], red[16];
  double2* Q = Qall + (long)c * (kmax + 1) * ld;
  double2* qc = qall + (long)c * ld;
  auto block_sum = [&](double v) {
    v = wave_sum(v);
    if (lane == 0) red[wave] = v;
    __syncthreads();
    double s = 0.0;
    for (int w = 0; w < nw; ++w) s += red[w];
    __syncthreads();
    return s;
  };
  const double2 zero = make_double2(0.0, 0.0);
  double2 q[kQShortE], r[kQShortE];
  double m[kQShortE], v = 0.0;
#pragma unroll
  for (int e = 0; e < kQShortE; ++e) {
    const int i = t + nt * e;
    const bool in = i < ld;
    m[e] = in ? mask[(long)c * ld + i] : 0.0;
    q[e] = in ? qc[i] : zero;
    r[e] = in ? Lq[(long)c * ld + i] : zero;
    v += m[e] * (q[e].x * r[e].x + q[e].y * r[e].y);
  }
  const double ak = block_sum(v);
  const double cp = k > 0 ? cc[c * kmax + k - 1] : 0.0;
  v = 0.0;
#pragma unroll
  for (int e = 0; e < kQShortE; ++e) {
    const int i = t + nt * e;
    r[e] = make_double2(r[e].x - ak * q[e].x, r[e].y - ak * q[e].y);
    if (k > 0 && i < ld) {
      const double2 qm = Q[(long)(k - 1) * ld + i];
      r[e] = make_double2(r[e].x - cp * qm.x, r[e].y - cp * qm.y);
    }
    v += m[e] * (r[e].x * r[e].x + r[e].y * r[e].y);
  }
  // stop tests of QL:1083-1095 and the step cap (ql_decide)
  const double b = sqrt(block_sum(v));
  const bool conv = !(fabs(b) >= tol) || nextc[c], stop = conv || k + 1 >= cap[c];
  __syncthreads();   // every thread has read the chain's state
  if (t == 0) {
    a[c * kmax + k] = ak;
    ndone[c] = k + 1;
    if (!conv) bb[c * kmax + k] = cc[c * kmax + k] = b;
    if (stop) active[c] = 0;
  }
  if (stop) return;
  const double inv = 1.0 / b;
#pragma unroll
  for (int e = 0; e < kQShortE; ++e) r[e] = csc(r[e], inv);
  for (int pass = 0; pass < 2; ++pass) {
#pragma unroll
    for (int e = 0; e < kQShortE; ++e)
      if (t + nt * e < ld) rm[t + nt * e] = csc(r[e], m[e]);
    __syncthreads();
    for (int j = wave; j <= k; j += nw) {
      const double2* Qj = Q + (long)j * ld;
      double s = 0.0;
#pragma unroll 8
      for (int i = lane; i < ld; i += 64) {
        const double2 x = Qj[i], y = rm[i];
        s += x.x * y.x + x.y * y.y;
      }
      s = wave_sum(s);
      if (lane == 0) coef[j] = s;
    }
    __syncthreads();
#pragma unroll 4
    for (int j = 0; j <= k; ++j) {
      const double cj = coef[j];
#pragma unroll
      for (int e = 0; e < kQShortE; ++e)
        if (t + nt * e < ld) {
          const double2 x = Q[(long)j * ld + t + nt * e];
          r[e] = make_double2(r[e].x - cj * x.x, r[e].y - cj * x.y);
        }
    }
  }
  v = 0.0;
#pragma unroll
  for (int e = 0; e < kQShortE; ++e) v += m[e] * (r[e].x * r[e].x + r[e].y * r[e].y);
  const double nrm = sqrt(block_sum(v));
  const bool small = !(nrm >= tol);
  const double sc = small ? 1.0 : 1.0 / nrm;
#pragma unroll
  for (int e = 0; e < kQShortE; ++e) {
    const int i = t + nt * e;
    if (i < ld) {
      const double2 x = csc(r[e], sc);
      Q[(long)(k + 1) * ld + i] = x;
      qc[i] = x;
    }
  }
  if (t == 0) {
    nextc[c] = small ? 1 : 0;
    kk[c] = k + 1;
  }
}

static void ql_step(QCtx* q, QBatch& b, QLanczos& l, double tol, int ih, int i3, int i4,
                    hipStream_t s) {
  const int ld = b.ld, C = b.C;
  const dim3 gv((ld + 255) / 256, C);
  launch_L(q, b, l.qcur, l.Lq, ih, i3, i4, s);
  if (ld <= 1024 * kQShortE && l.kmax < kQShortBasis && 2L * ld * l.kmax <= kQShortWork) {
    hipLaunchKernelGGL(ql_short, dim3(C), dim3(ld <= 256 * kQShortE ? 256 : 1024), 0, s, l.Lq,
                       l.mask, ld, l.kmax, tol, b.active, l.nextc, l.k, l.cap, l.ndone, l.a, l.bb,
                       l.cc, l.Q, l.qcur);
    return;
  }
  hipLaunchKernelGGL(ql_dot, dim3(C), dim3(256), 0, s, l.qcur, l.Lq, l.mask, ld, b.active, l.scal,
                     0);
  hipLaunchKernelGGL(ql_residual, gv, dim3(256), 0, s, l.Lq, l.qcur, l.Q, ld, l.kmax, b.active,
                     l.k, l.scal, l.cc, l.a, l.r);
  hipLaunchKernelGGL(ql_dot, dim3(C), dim3(256), 0, s, l.r, l.r, l.mask, ld, b.active, l.scal, 1);
  hipLaunchKernelGGL(ql_decide, dim3((C + 63) / 64), dim3(64), 0, s, C, l.kmax, tol, b.active,
                     l.cont, l.nextc, l.k, l.cap, l.ndone, l.scal, l.bb, l.cc);
  hipLaunchKernelGGL(ql_scale, gv, dim3(256), 0, s, ld, l.cont, l.scal, l.r);
  for (int pass = 0; pass < 2; ++pass) {
    if (q->reorth_jtile == 8)
      reorth_pass<8>(l, b, s);
    else if (q->reorth_jtile == 32)
      reorth_pass<32>(l, b, s);
    else
      reorth_pass<16>(l, b, s);
  }
  hipLaunchKernelGGL(ql_dot, dim3(C), dim3(256), 0, s, l.r, l.r, l.mask, ld, l.cont, l.scal, 2);
  hipLaunchKernelGGL(ql_store, gv, dim3(256), 0, s, ld, l.kmax, tol, l.cont, l.k, l.scal, l.nextc,
                     l.r, l.Q, l.qcur);
  hipLaunchKernelGGL(ql_advance, dim3((C + 63) / 64), dim3(64), 0, s, C, l.cont, l.k);
}

// Hermitian metric of QL:441-480 for every chain's layout
static void host_mask(const QBatch& b, int nq, int nb, const int* pair_map, int c,
                      std::vector<double>& m) {
  const int ld = b.ld;
  std::fill(m.begin() + (long)c * ld, m.begin() + (long)(c + 1) * ld, 0.0);
  double* mc = m.data() + (long)c * ld;
  for (int v = 0; v < nb; ++v) mc[v] = 1.0;
  const int* pm = pair_map + (long)c * nq;
  int off = nb;
  std::vector<std::pair<int, int>> pairs;
  for (int i = 0; i < nq; ++i)
    if (i <= pm[i]) pairs.push_back({i, pm[i]});
  for (int sector = 0; sector < 2; ++sector)
    for (auto& pr : pairs) {
      if (pr.first < pr.second) {
        for (int e = 0; e < nb * nb; ++e) mc[off + e] = 2.0;
        off += nb * nb;
      } else {
        for (int i = 0; i < nb; ++i)
          for (int j = i; j < nb; ++j) mc[off++] = (i == j) ? 1.0 : 2.0;
      }
    }
}

// ------------------------------------------------- kernel polynomial method
// One work-group per chain: d = <x, y>_M (fixed-order sum), then moment m of
// chain c is d (mode 0) or 2 d - mom[c][ref] (mode 1: mu_{2n} with ref 0,
// mu_{2n+1} with ref 1; QSK:346-390).
__global__ void __launch_bounds__(256) kpm_moment(const double2* __restrict__ x,
                                                  const double2* __restrict__ y,
                                                  const double* __restrict__ mask, int ld,
                                                  double* __restrict__ mom, int n_mom, int m,
                                                  int mode, int ref) {
  const int c = blockIdx.x, t = threadIdx.x;
  const double2* xc = x + (long)c * ld;
  const double2* yc = y + (long)c * ld;
  const double* mc = mask + (long)c * ld;
  double s = 0.0;
  for (int e = t; e < ld; e += blockDim.x) s += mc[e] * (xc[e].x * yc[e].x + xc[e].y * yc[e].y);
  __shared__ double red[4];
  s = wave_sum(s);
  if ((t & 63) == 0) red[t >> 6] = s;
  __syncthreads();
  if (t == 0) {
    const double d = red[0] + red[1] + red[2] + red[3];
    mom[(long)c * n_mom + m] = mode ? 2.0 * d - mom[(long)c * n_mom + ref] : d;
  }
}

// Chebyshev step of chain c (blockIdx.y): t = (L v - b v) / a with (a, b) =
// rescale[c]; out = t (first step) or 2 t - vm (out may alias vm).
__global__ void kpm_combine(const double2* __restrict__ Lv, const double2* __restrict__ v,
                            const double2* vm, const double* __restrict__ rescale, int ld,
                            int first, double2* out) {
  const int c = blockIdx.y, e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= ld) return;
  const long i = (long)c * ld + e;
  const double a = rescale[2 * c], b = rescale[2 * c + 1];
  const double2 lv = Lv[i], vv = v[i];
  double2 r = make_double2((lv.x - b * vv.x) / a, (lv.y - b * vv.y) / a);
  if (!first) {
    const double2 p = vm[i];
    r = make_double2(2.0 * r.x - p.x, 2.0 * r.y - p.y);
  }
  out[i] = r;
}

}  // namespace tdscha

using namespace tdscha;

extern "C" {

int tdscha_qctx_create(tdscha_qctx** out, int n_q, int n_bands, int n_configs, const double* X_q,
                       const double* Y_q, const double* w_q, const int* valid_modes_q,
                       const double* rho, double T) {
  TDS_REQUIRE(out != nullptr, 2, "tdscha_qctx_create: NULL out");
  TDS_REQUIRE(n_q >= 1 && n_q <= kQMaxQ, 2, "tdscha_qctx_create: n_q must be in [1, 512]");
  TDS_REQUIRE(n_bands == 3 || n_bands == 6, 2,
              "tdscha_qctx_create: n_bands must be 3 or 6 (1 or 2 atoms per cell)");
  TDS_REQUIRE(n_configs >= 1, 2, "tdscha_qctx_create: n_configs must be positive");
  TDS_REQUIRE(X_q && Y_q && w_q && valid_modes_q && rho, 2, "tdscha_qctx_create: NULL array");
  *out = nullptr;
  const int nq = n_q, nb = n_bands, N = n_configs;
  QCtx* q = new QCtx();
  q->nq = nq;
  q->nb = nb;
  q->N = N;
  q->T = T;
  double neff = 0.0;
  for (int i = 0; i < N; ++i) neff += rho[i];
  TDS_REQUIRE(neff > 0, 2, "tdscha_qctx_create: sum(rho) must be positive");
  q->neff = neff;
  // host copies in device layouts
  const size_t ne = (size_t)nq * nb * N;
  std::vector<double2> hx(ne), hy(ne);
  for (int iq = 0; iq < nq; ++iq)
    for (int i = 0; i < N; ++i)
      for (int v = 0; v < nb; ++v) {
        const size_t src = (((size_t)iq * N + i) * nb + v) * 2;
        const size_t dst = ((size_t)iq * nb + v) * N + i;
        hx[dst] = make_double2(X_q[src], X_q[src + 1]);
        hy[dst] = make_double2(Y_q[src], Y_q[src + 1]);
      }
  std::vector<double> hw(nq * nb), hn(nq * nb), hfy(nq * nb), hfp(nq * nb);
  std::vector<int> hv(nq * nb);
  for (int iq = 0; iq < nq; ++iq)
    for (int v = 0; v < nb; ++v) {
      const double w = w_q[v * nq + iq];
      const int ok = valid_modes_q[v * nq + iq] ? 1 : 0;
      double n = 0.0;
      if (ok && T > 1e-12) n = 1.0 / (std::exp(w * RY_TO_K / T) - 1.0);   // QL:581-602
      hw[iq * nb + v] = w;
      hn[iq * nb + v] = n;
      hv[iq * nb + v] = ok;
      // JQ:680-699
      double nw = 0.0;
      if (ok && T > 0) nw = 1.0 / (std::exp(w * RY_TO_K / T) - 1.0);
      hfy[iq * nb + v] = ok ? 2.0 * w / (1.0 + 2.0 * nw) : 0.0;
      hfp[iq * nb + v] = ok ? (1.0 + 2.0 * nw) / (2.0 * w) : 0.0;
    }
  auto fail = [&](const char* what) {
    tdscha_qctx_destroy(reinterpret_cast<tdscha_qctx*>(q));
    set_error(std::string("tdscha_qctx_create: ") + what);
    return -1;
  };
  if (hipStreamCreate(&q->stream) != hipSuccess) return fail("hipStreamCreate failed");
  {
    int dev = 0, ncu = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
        ncu > 0)
      q->n_cu = ncu;
  }
  bool ok = hipMalloc((void**)&q->X, sizeof(double2) * ne) == hipSuccess &&
            hipMalloc((void**)&q->Y, sizeof(double2) * ne) == hipSuccess &&
            hipMalloc((void**)&q->rho, sizeof(double) * N) == hipSuccess &&
            hipMalloc((void**)&q->wq, sizeof(double) * nq * nb) == hipSuccess &&
            hipMalloc((void**)&q->nbose, sizeof(double) * nq * nb) == hipSuccess &&
            hipMalloc((void**)&q->valid, sizeof(int) * nq * nb) == hipSuccess &&
            hipMalloc((void**)&q->fY, sizeof(double) * nq * nb) == hipSuccess &&
            hipMalloc((void**)&q->fP, sizeof(double) * nq * nb) == hipSuccess;
  if (!ok) return fail("device allocation failed");
  ok = hipMemcpy(q->X, hx.data(), sizeof(double2) * ne, hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(q->Y, hy.data(), sizeof(double2) * ne, hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(q->rho, rho, sizeof(double) * N, hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(q->wq, hw.data(), sizeof(double) * nq * nb, hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(q->nbose, hn.data(), sizeof(double) * nq * nb, hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(q->valid, hv.data(), sizeof(int) * nq * nb, hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(q->fY, hfy.data(), sizeof(double) * nq * nb, hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(q->fP, hfp.data(), sizeof(double) * nq * nb, hipMemcpyHostToDevice) == hipSuccess;
  if (!ok) return fail("upload failed");
  if (build_slabs(q)) return fail("slab images failed");
  *out = reinterpret_cast<tdscha_qctx*>(q);
  return 0;
}

void tdscha_qctx_destroy(tdscha_qctx* ctx) {
  if (!ctx) return;
  QCtx* q = reinterpret_cast<QCtx*>(ctx);
  if (q->stream) (void)hipStreamSynchronize(q->stream);
  void* p[] = {q->X, q->Y, q->rho, q->wq, q->nbose, q->valid, q->fY, q->fP, q->S, q->work};
  for (void* x : p)
    if (x) (void)hipFree(x);
  if (q->pinned) (void)hipHostFree(q->pinned);
  if (q->stream) (void)hipStreamDestroy(q->stream);
  delete q;
}

int tdscha_qctx_symmetrize(tdscha_qctx* ctx, int n_sym, const int* q_perm, const double* D) {
  TDS_REQUIRE(ctx && q_perm && D, 2, "tdscha_qctx_symmetrize: NULL argument");
  QCtx* q = reinterpret_cast<QCtx*>(ctx);
  const int nq = q->nq, nb = q->nb, N = q->N;
  TDS_REQUIRE(n_sym >= 1 && n_sym <= 65535, 2, "tdscha_qctx_symmetrize: n_sym must be in [1, 65535]");
  TDS_REQUIRE(q->n_sym == 1, 2, "tdscha_qctx_symmetrize: the ensemble is already expanded");
  TDS_REQUIRE((long)N * n_sym <= 0x7fffffffL, 2,
              "tdscha_qctx_symmetrize: n_sym * n_configs exceeds 2^31 - 1");
  for (int j = 0; j < n_sym; ++j) {
    std::vector<char> seen(nq, 0);
    for (int p = 0; p < nq; ++p) {
      const int t = q_perm[(long)j * nq + p];
      TDS_REQUIRE(t >= 0 && t < nq && !seen[t], 2,
                  "tdscha_qctx_symmetrize: q_perm row is not a permutation of the q-points");
      seen[t] = 1;
    }
  }
  const int N2 = N * n_sym;
  const size_t ne2 = (size_t)nq * nb * N2;
  std::vector<double> hrho(N), hrho2((size_t)N2);
  if (hipMemcpy(hrho.data(), q->rho, sizeof(double) * N, hipMemcpyDeviceToHost) != hipSuccess) {
    set_error("tdscha_qctx_symmetrize: rho download failed");
    return -1;
  }
  for (int j = 0; j < n_sym; ++j)
    for (int i = 0; i < N; ++i) hrho2[(size_t)j * N + i] = hrho[i];
  double2 *XE = nullptr, *YE = nullptr, *dD = nullptr;
  double* rho2 = nullptr;
  int* dperm = nullptr;
  auto release = [&]() {
    void* p[] = {XE, YE, dD, rho2, dperm};
    for (void* x : p)
      if (x) (void)hipFree(x);
  };
  bool ok = hipMalloc((void**)&XE, sizeof(double2) * ne2) == hipSuccess &&
            hipMalloc((void**)&YE, sizeof(double2) * ne2) == hipSuccess &&
            hipMalloc((void**)&rho2, sizeof(double) * N2) == hipSuccess &&
            hipMalloc((void**)&dperm, sizeof(int) * (size_t)n_sym * nq) == hipSuccess &&
            hipMalloc((void**)&dD, sizeof(double2) * (size_t)n_sym * nq * nb * nb) == hipSuccess;
  if (!ok) {
    release();
    set_error("tdscha_qctx_symmetrize: device allocation failed");
    return -1;
  }
  ok = hipMemcpy(rho2, hrho2.data(), sizeof(double) * N2, hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(dperm, q_perm, sizeof(int) * (size_t)n_sym * nq, hipMemcpyHostToDevice) ==
           hipSuccess &&
       hipMemcpy(dD, D, sizeof(double2) * (size_t)n_sym * nq * nb * nb, hipMemcpyHostToDevice) ==
           hipSuccess;
  if (!ok) {
    release();
    set_error("tdscha_qctx_symmetrize: upload failed");
    return -1;
  }
  const dim3 g((unsigned)((N + 255) / 256), (unsigned)n_sym, (unsigned)nq);
  if (nb == 6)
    hipLaunchKernelGGL(q_expand<6>, g, dim3(256), 0, q->stream, q->X, q->Y, N, nq, dperm, dD, XE, YE);
  else
    hipLaunchKernelGGL(q_expand<3>, g, dim3(256), 0, q->stream, q->X, q->Y, N, nq, dperm, dD, XE, YE);
  if (hipGetLastError() != hipSuccess || hipStreamSynchronize(q->stream) != hipSuccess) {
    release();
    set_error("tdscha_qctx_symmetrize: expansion kernel failed");
    return -1;
  }
  (void)hipFree(q->X);
  (void)hipFree(q->Y);
  (void)hipFree(q->rho);
  (void)hipFree(dperm);
  (void)hipFree(dD);
  q->X = XE;
  q->Y = YE;
  q->rho = rho2;
  q->N = N2;
  q->neff *= n_sym;
  q->n_sym = n_sym;
  return build_slabs(q);
}

static int apply_L_host(tdscha_qctx* ctx, int n_chains, const int* iq_pert,
                        const int* q_pair_map, const double* psi, double* out,
                        int ignore_harmonic, int ignore_v3, int ignore_v4, bool static_op);

int tdscha_qspace_apply_L(tdscha_qctx* ctx, int n_chains, const int* iq_pert,
                          const int* q_pair_map, const double* psi, double* out,
                          int ignore_harmonic, int ignore_v3, int ignore_v4) {
  return apply_L_host(ctx, n_chains, iq_pert, q_pair_map, psi, out, ignore_harmonic, ignore_v3,
                      ignore_v4, false);
}

int tdscha_qspace_apply_L_static(tdscha_qctx* ctx, int n_chains, const int* iq_pert,
                                 const int* q_pair_map, const double* psi, double* out,
                                 int ignore_harmonic, int ignore_v3, int ignore_v4) {
  return apply_L_host(ctx, n_chains, iq_pert, q_pair_map, psi, out, ignore_harmonic, ignore_v3,
                      ignore_v4, true);
}

int tdscha_qspace_static_psi_size(int n_q, int n_bands, const int* q_pair_map, int* psi_size) {
  int full = 0;
  const int rc = tdscha_qspace_psi_size(n_q, n_bands, q_pair_map, &full);
  if (rc) return rc;
  *psi_size = n_bands + (full - n_bands) / 2;
  return 0;
}

int tdscha_qspace_psi_size(int n_q, int n_bands, const int* q_pair_map, int* psi_size) {
  TDS_REQUIRE(q_pair_map && psi_size && n_q > 0 && n_bands > 0, 2,
              "tdscha_qspace_psi_size: bad argument");
  int off = n_bands;
  for (int i = 0; i < n_q; ++i) {
    TDS_REQUIRE(q_pair_map[i] >= 0 && q_pair_map[i] < n_q && q_pair_map[q_pair_map[i]] == i, 2,
                "tdscha_qspace_psi_size: q_pair_map must be an involution");
    if (i < q_pair_map[i]) off += 2 * n_bands * n_bands;
    else if (i == q_pair_map[i]) off += n_bands * (n_bands + 1);
  }
  *psi_size = off;
  return 0;
}

int tdscha_qspace_set_tiles(tdscha_qctx* ctx, int weights_tile, int d2v_chunk, int reorth_jtile) {
  TDS_REQUIRE(ctx != nullptr, 2, "tdscha_qspace_set_tiles: NULL context");
  TDS_REQUIRE(weights_tile == 64 || weights_tile == 128 || weights_tile == 256, 2,
              "weights_tile must be 64, 128 or 256");
  TDS_REQUIRE(d2v_chunk >= 0, 2, "d2v_chunk must be >= 0 (0 = automatic)");
  TDS_REQUIRE(reorth_jtile == 8 || reorth_jtile == 16 || reorth_jtile == 32, 2,
              "reorth_jtile must be 8, 16 or 32");
  QCtx* q = reinterpret_cast<QCtx*>(ctx);
  q->weights_tile = weights_tile;
  q->d2v_chunk = d2v_chunk;
  q->reorth_jtile = reorth_jtile;
  return 0;
}

int tdscha_qspace_get_d2v_form(const tdscha_qctx* ctx, int* form) {
  TDS_REQUIRE(ctx && form, 2, "tdscha_qspace_get_d2v_form: NULL argument");
  const QCtx* q = reinterpret_cast<const QCtx*>(ctx);
  *form = q->S && q->d2v_form ? 1 : 0;
  return 0;
}

int tdscha_qspace_set_d2v_form(tdscha_qctx* ctx, int form) {
  TDS_REQUIRE(ctx != nullptr, 2, "tdscha_qspace_set_d2v_form: NULL context");
  TDS_REQUIRE(form == 0 || form == 1, 2, "d2v form must be 0 or 1");
  reinterpret_cast<QCtx*>(ctx)->d2v_form = form;
  return 0;
}

int tdscha_qspace_get_tiles(const tdscha_qctx* ctx, int* tiles_out) {
  TDS_REQUIRE(ctx && tiles_out, 2, "tdscha_qspace_get_tiles: NULL argument");
  const QCtx* q = reinterpret_cast<const QCtx*>(ctx);
  tiles_out[0] = q->weights_tile;
  tiles_out[1] = q->d2v_chunk;
  tiles_out[2] = q->reorth_jtile;
  return 0;
}

static int apply_L_host(tdscha_qctx* ctx, int n_chains, const int* iq_pert,
                        const int* q_pair_map, const double* psi, double* out,
                        int ignore_harmonic, int ignore_v3, int ignore_v4, bool static_op) {
  TDS_REQUIRE(ctx && iq_pert && q_pair_map && psi && out, 2, "tdscha_qspace_apply_L: NULL argument");
  TDS_REQUIRE(n_chains >= 1 && n_chains <= kQMaxChains, 2, "n_chains must be in [1, 256]");
  QCtx* q = reinterpret_cast<QCtx*>(ctx);
  QBatch b;
  int rc = build_batch(q, n_chains, iq_pert, q_pair_map, b, 0, static_op, true);
  if (rc) return rc;
  const int C = n_chains, ld = b.ld;
  const size_t bytes = sizeof(double2) * C * ld;
  long pos = 0;
  for (int c = 0; c < C; ++c) {
    const int len = b.h_len[c];
    std::memcpy(b.host + (size_t)c * ld, psi + 2 * pos, sizeof(double2) * len);
    std::fill(b.host + (size_t)c * ld + len, b.host + (size_t)(c + 1) * ld,
              make_double2(0.0, 0.0));
    pos += len;
  }
  hipStream_t s = q->stream;
  bool ok = hipMemcpyAsync(b.psi, b.host, bytes, hipMemcpyHostToDevice, s) == hipSuccess;
  if (ok) {
    launch_L(q, b, b.psi, b.out, ignore_harmonic, ignore_v3, ignore_v4, s, static_op);
    ok = hipGetLastError() == hipSuccess &&
         hipMemcpyAsync(b.host, b.out, bytes, hipMemcpyDeviceToHost, s) == hipSuccess &&
         hipStreamSynchronize(s) == hipSuccess;
  }
  pos = 0;
  for (int c = 0; ok && c < C; ++c) {
    std::memcpy(out + 2 * pos, b.host + (size_t)c * ld, sizeof(double2) * b.h_len[c]);
    pos += b.h_len[c];
  }
  free_batch(b);
  if (!ok) {
    set_error("tdscha_qspace_apply_L: device execution failed");
    return -1;
  }
  return 0;
}

int tdscha_qspace_lanczos_run(tdscha_qctx* ctx, int n_chains, const int* iq_pert,
                              const int* q_pair_map, const double* psi0, int n_steps,
                              const int* caps, double tol, int ignore_harmonic, int ignore_v3,
                              int ignore_v4, int use_graph, double* a_out, double* b_out,
                              double* c_out, int* n_done, double* elapsed_ms) {
  TDS_REQUIRE(ctx && iq_pert && q_pair_map && psi0 && a_out && b_out && n_done, 2,
              "tdscha_qspace_lanczos_run: NULL argument");
  TDS_REQUIRE(n_chains >= 1 && n_chains <= kQMaxChains, 2, "n_chains must be in [1, 256]");
  TDS_REQUIRE(n_steps >= 1 && n_steps <= 100000, 2, "n_steps must be in [1, 100000]");
  QCtx* q = reinterpret_cast<QCtx*>(ctx);
  QBatch b;
  int rc = build_batch(q, n_chains, iq_pert, q_pair_map, b);
  if (rc) return rc;
  const int C = n_chains, ld = b.ld, kmax = n_steps;
  QLanczos l;
  l.kmax = kmax;
  const size_t qn = (size_t)C * (kmax + 1) * ld;
  Carve carve;   // l.Lq to l.cc start from zero, with one fill
  carve.add(&l.Q, qn);
  carve.add(&l.Lq, (size_t)C * ld);
  carve.add(&l.a, (size_t)C * kmax);
  carve.add(&l.bb, (size_t)C * kmax);
  carve.add(&l.cc, (size_t)C * kmax);
  const size_t zeroed = carve.total();
  carve.add(&l.qcur, (size_t)C * ld);
  carve.add(&l.r, (size_t)C * ld);
  carve.add(&l.mask, (size_t)C * ld);
  carve.add(&l.coef, (size_t)C * (kmax + 1));
  carve.add(&l.scal, (size_t)C * 4);
  carve.add(&l.k, C);
  carve.add(&l.cont, C);
  carve.add(&l.nextc, C);
  carve.add(&l.cap, C);
  carve.add(&l.ndone, C);
  bool ok = hipMalloc(&l.mem, carve.total()) == hipSuccess;
  if (ok) carve.assign(l.mem);
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  auto fail = [&](const char* what) {
    if (exec) (void)hipGraphExecDestroy(exec);
    if (graph) (void)hipGraphDestroy(graph);
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    free_ql(l);
    free_batch(b);
    set_error(std::string("tdscha_qspace_lanczos_run: ") + what);
    return -1;
  };
  if (!ok) return fail("device allocation failed");
  hipStream_t s = q->stream;
  // zero-padded starting vectors, masks, caps
  std::vector<double2> hp((size_t)C * ld, make_double2(0.0, 0.0));
  std::vector<double> hm((size_t)C * ld, 0.0);
  std::vector<int> hcap(C, n_steps);
  long pos = 0;
  for (int c = 0; c < C; ++c) {
    for (int e = 0; e < b.h_len[c]; ++e)
      hp[(size_t)c * ld + e] = make_double2(psi0[2 * (pos + e)], psi0[2 * (pos + e) + 1]);
    pos += b.h_len[c];
    host_mask(b, q->nq, q->nb, q_pair_map, c, hm);
    if (caps) hcap[c] = std::max(1, std::min(caps[c], n_steps));
  }
  ok = hipMemcpy(l.r, hp.data(), sizeof(double2) * C * ld, hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(l.mask, hm.data(), sizeof(double) * C * ld, hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(l.cap, hcap.data(), sizeof(int) * C, hipMemcpyHostToDevice) == hipSuccess &&
       hipMemset(l.mem, 0, zeroed) == hipSuccess;
  if (!ok) return fail("upload failed");
  hipLaunchKernelGGL(q_fill_int, dim3((C + 63) / 64), dim3(64), 0, s, l.k, C, 0);
  hipLaunchKernelGGL(q_fill_int, dim3((C + 63) / 64), dim3(64), 0, s, l.cont, C, 1);
  hipLaunchKernelGGL(q_fill_int, dim3((C + 63) / 64), dim3(64), 0, s, l.nextc, C, 0);
  hipLaunchKernelGGL(q_fill_int, dim3((C + 63) / 64), dim3(64), 0, s, l.ndone, C, 0);
  hipLaunchKernelGGL(ql_dot, dim3(C), dim3(256), 0, s, l.r, l.r, l.mask, ld, l.cont, l.scal, 2);
  hipLaunchKernelGGL(ql_init, dim3((ld + 255) / 256, C), dim3(256), 0, s, l.r, ld, kmax, l.scal,
                     l.Q, l.qcur);
  if (hipGetLastError() != hipSuccess || hipStreamSynchronize(s) != hipSuccess)
    return fail("initialisation failed");
  if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess)
    return fail("event creation failed");
  if (use_graph) {
    // the whole run as one graph: one launch replays every step
    if (hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal) != hipSuccess)
      return fail("stream capture failed to start");
    for (int step = 0; step < n_steps; ++step)
      ql_step(q, b, l, tol, ignore_harmonic, ignore_v3, ignore_v4, s);
    if (hipStreamEndCapture(s, &graph) != hipSuccess) return fail("stream capture failed");
    if (hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0) != hipSuccess)
      return fail("graph instantiation failed");
  }
  (void)hipEventRecord(e0, s);
  if (use_graph) {
    if (hipGraphLaunch(exec, s) != hipSuccess) return fail("graph launch failed");
  } else {
    for (int step = 0; step < n_steps; ++step)
      ql_step(q, b, l, tol, ignore_harmonic, ignore_v3, ignore_v4, s);
  }
  (void)hipEventRecord(e1, s);
  if (hipStreamSynchronize(s) != hipSuccess || hipGetLastError() != hipSuccess)
    return fail("step execution failed");
  float ms = 0.f;
  (void)hipEventElapsedTime(&ms, e0, e1);
  if (elapsed_ms) *elapsed_ms = ms;
  ok = hipMemcpy(a_out, l.a, sizeof(double) * C * kmax, hipMemcpyDeviceToHost) == hipSuccess &&
       hipMemcpy(b_out, l.bb, sizeof(double) * C * kmax, hipMemcpyDeviceToHost) == hipSuccess &&
       (!c_out || hipMemcpy(c_out, l.cc, sizeof(double) * C * kmax, hipMemcpyDeviceToHost) == hipSuccess) &&
       hipMemcpy(n_done, l.ndone, sizeof(int) * C, hipMemcpyDeviceToHost) == hipSuccess;
  if (!ok) return fail("download failed");
  if (exec) (void)hipGraphExecDestroy(exec);
  if (graph) (void)hipGraphDestroy(graph);
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  free_ql(l);
  free_batch(b);
  return 0;
}

// Time one L application of the batch for every (weights tile, d2v chunk)
// candidate and every reorthogonalisation tile; keep the fastest.
int tdscha_qspace_kpm_run(tdscha_qctx* ctx, int n_chains, const int* iq_pert,
                          const int* q_pair_map, const double* rescale, int n_moments,
                          int n_have, double* moments, double* vm, double* v,
                          int ignore_harmonic, int ignore_v3, int ignore_v4, int use_graph,
                          double* elapsed_ms) {
  TDS_REQUIRE(ctx && iq_pert && q_pair_map && rescale && moments && vm && v, 2,
              "tdscha_qspace_kpm_run: NULL argument");
  TDS_REQUIRE(n_chains >= 1 && n_chains <= kQMaxChains, 2, "n_chains must be in [1, 256]");
  TDS_REQUIRE(n_moments >= 1 && n_moments <= 200000, 2, "n_moments must be in [1, 200000]");
  TDS_REQUIRE(n_have >= 0 && n_have < n_moments, 2, "n_have must be in [0, n_moments)");
  for (int c = 0; c < n_chains; ++c)
    TDS_REQUIRE(rescale[2 * c] > 0, 2, "tdscha_qspace_kpm_run: rescale a must be positive");
  QCtx* q = reinterpret_cast<QCtx*>(ctx);
  QBatch b;
  int rc = build_batch(q, n_chains, iq_pert, q_pair_map, b);
  if (rc) return rc;
  const int C = n_chains, ld = b.ld, N = n_moments;
  const size_t nv = (size_t)C * ld;
  double2 *B0 = nullptr, *B1 = nullptr, *B2 = nullptr, *LV = nullptr;
  double *dmask = nullptr, *dmom = nullptr, *dres = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  auto release = [&]() {
    if (exec) (void)hipGraphExecDestroy(exec);
    if (graph) (void)hipGraphDestroy(graph);
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    void* p[] = {B0, B1, B2, LV, dmask, dmom, dres};
    for (void* x : p)
      if (x) (void)hipFree(x);
    free_batch(b);
  };
  auto fail = [&](const char* what) {
    release();
    set_error(std::string("tdscha_qspace_kpm_run: ") + what);
    return -1;
  };
  bool ok = hipMalloc((void**)&B0, sizeof(double2) * nv) == hipSuccess &&
            hipMalloc((void**)&B1, sizeof(double2) * nv) == hipSuccess &&
            hipMalloc((void**)&B2, sizeof(double2) * nv) == hipSuccess &&
            hipMalloc((void**)&LV, sizeof(double2) * nv) == hipSuccess &&
            hipMalloc((void**)&dmask, sizeof(double) * nv) == hipSuccess &&
            hipMalloc((void**)&dmom, sizeof(double) * C * N) == hipSuccess &&
            hipMalloc((void**)&dres, sizeof(double) * 2 * C) == hipSuccess;
  if (!ok) return fail("device allocation failed");
  // vectors in the padded [C][ld] layout; masks; moments so far
  std::vector<double2> hvm(nv, make_double2(0.0, 0.0)), hv(nv, make_double2(0.0, 0.0));
  std::vector<double> hmask(nv, 0.0), hmom((size_t)C * N, 0.0);
  long pos = 0;
  for (int c = 0; c < C; ++c) {
    for (int e = 0; e < b.h_len[c]; ++e) {
      hvm[(size_t)c * ld + e] = make_double2(vm[2 * (pos + e)], vm[2 * (pos + e) + 1]);
      hv[(size_t)c * ld + e] = make_double2(v[2 * (pos + e)], v[2 * (pos + e) + 1]);
    }
    pos += b.h_len[c];
    host_mask(b, q->nq, q->nb, q_pair_map, c, hmask);
    for (int m = 0; m < n_have; ++m) hmom[(size_t)c * N + m] = moments[(size_t)c * N + m];
    hmom[(size_t)c * N] = n_have ? hmom[(size_t)c * N] : 1.0;
  }
  ok = hipMemcpy(B0, hvm.data(), sizeof(double2) * nv, hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(B1, hv.data(), sizeof(double2) * nv, hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(dmask, hmask.data(), sizeof(double) * nv, hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(dmom, hmom.data(), sizeof(double) * C * N, hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(dres, rescale, sizeof(double) * 2 * C, hipMemcpyHostToDevice) == hipSuccess &&
       hipMemset(B2, 0, sizeof(double2) * nv) == hipSuccess &&
       hipMemset(LV, 0, sizeof(double2) * nv) == hipSuccess;
  if (!ok) return fail("upload failed");
  hipStream_t s = q->stream;
  const dim3 gv((ld + 255) / 256, C);
  // The recurrence of QSK:301-440: vm, v hold T_{n-1}, T_n; a step computes
  // mu_{2n} = 2 <v, v> - mu_0, then vp = 2 L~ v - vm (into the third
  // buffer) and mu_{2n+1} = 2 <vp, v> - mu_1.  All launches are enqueued
  // here; with use_graph they are captured first and replayed as one graph.
  double2* pv[3] = {B0, B1, B2};   // pv[0] = vm, pv[1] = v, pv[2] = spare
  int n = 0;
  auto L = [&](const double2* in) {
    launch_L(q, b, in, LV, ignore_harmonic, ignore_v3, ignore_v4, s);
  };
  auto rotate = [&]() {             // vm, v = v, vp
    double2* old_vm = pv[0];
    pv[0] = pv[1];
    pv[1] = pv[2];
    pv[2] = old_vm;
  };
  auto enqueue = [&]() {
    if (n_have == 0) {
      // fresh start: vm = v = v0 (given in both); T_1 = L~ v0, mu_1 = <v0, T_1>
      if (N > 1) {
        L(pv[1]);
        hipLaunchKernelGGL(kpm_combine, gv, dim3(256), 0, s, LV, pv[1], pv[0], dres, ld, 1, pv[2]);
        hipLaunchKernelGGL(kpm_moment, dim3(C), dim3(256), 0, s, pv[1], pv[2], dmask, ld, dmom,
                           N, 1, 0, 0);
        rotate();
        n = 1;
      }
    } else if (n_have == 1) {
      L(pv[1]);
      hipLaunchKernelGGL(kpm_combine, gv, dim3(256), 0, s, LV, pv[1], pv[0], dres, ld, 1, pv[2]);
      hipLaunchKernelGGL(kpm_moment, dim3(C), dim3(256), 0, s, pv[0], pv[2], dmask, ld, dmom, N,
                         1, 0, 0);
      rotate();
      n = 1;
    } else if (n_have % 2 == 0) {
      n = n_have / 2;
    } else {
      const int h = n_have / 2;      // the interrupted odd moment
      L(pv[1]);
      hipLaunchKernelGGL(kpm_combine, gv, dim3(256), 0, s, LV, pv[1], pv[0], dres, ld, 0, pv[2]);
      hipLaunchKernelGGL(kpm_moment, dim3(C), dim3(256), 0, s, pv[2], pv[1], dmask, ld, dmom, N,
                         2 * h + 1, 1, 1);
      rotate();
      n = h + 1;
    }
    if (N > 1 || n_have > 0) {
      while (2 * n < N) {
        hipLaunchKernelGGL(kpm_moment, dim3(C), dim3(256), 0, s, pv[1], pv[1], dmask, ld, dmom,
                           N, 2 * n, 1, 0);
        if (2 * n + 1 >= N) break;
        L(pv[1]);
        hipLaunchKernelGGL(kpm_combine, gv, dim3(256), 0, s, LV, pv[1], pv[0], dres, ld, 0, pv[2]);
        hipLaunchKernelGGL(kpm_moment, dim3(C), dim3(256), 0, s, pv[2], pv[1], dmask, ld, dmom,
                           N, 2 * n + 1, 1, 1);
        rotate();
        ++n;
      }
    }
  };
  if (hipStreamSynchronize(s) != hipSuccess) return fail("upload synchronisation failed");
  if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess)
    return fail("event creation failed");
  if (use_graph) {
    if (hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal) != hipSuccess)
      return fail("stream capture failed to start");
    enqueue();
    if (hipStreamEndCapture(s, &graph) != hipSuccess) return fail("stream capture failed");
    if (hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0) != hipSuccess)
      return fail("graph instantiation failed");
    (void)hipEventRecord(e0, s);
    if (hipGraphLaunch(exec, s) != hipSuccess) return fail("graph launch failed");
  } else {
    (void)hipEventRecord(e0, s);
    enqueue();
  }
  (void)hipEventRecord(e1, s);
  if (hipStreamSynchronize(s) != hipSuccess || hipGetLastError() != hipSuccess)
    return fail("step execution failed");
  float ms = 0.f;
  (void)hipEventElapsedTime(&ms, e0, e1);
  if (elapsed_ms) *elapsed_ms = ms;
  // download the moments and the final recurrence vectors (vm, v)
  ok = hipMemcpy(hmom.data(), dmom, sizeof(double) * C * N, hipMemcpyDeviceToHost) == hipSuccess &&
       hipMemcpy(hvm.data(), pv[0], sizeof(double2) * nv, hipMemcpyDeviceToHost) == hipSuccess &&
       hipMemcpy(hv.data(), pv[1], sizeof(double2) * nv, hipMemcpyDeviceToHost) == hipSuccess;
  if (!ok) return fail("download failed");
  std::copy(hmom.begin(), hmom.end(), moments);
  pos = 0;
  for (int c = 0; c < C; ++c) {
    for (int e = 0; e < b.h_len[c]; ++e) {
      vm[2 * (pos + e)] = hvm[(size_t)c * ld + e].x;
      vm[2 * (pos + e) + 1] = hvm[(size_t)c * ld + e].y;
      v[2 * (pos + e)] = hv[(size_t)c * ld + e].x;
      v[2 * (pos + e) + 1] = hv[(size_t)c * ld + e].y;
    }
    pos += b.h_len[c];
  }
  release();
  return 0;
}

int tdscha_qspace_autotune(tdscha_qctx* ctx, int n_chains, const int* iq_pert,
                           const int* q_pair_map, int reps, int* tiles_out, double* best_ms) {
  TDS_REQUIRE(ctx && iq_pert && q_pair_map, 2, "tdscha_qspace_autotune: NULL argument");
  TDS_REQUIRE(n_chains >= 1 && n_chains <= kQMaxChains, 2, "n_chains must be in [1, 256]");
  QCtx* q = reinterpret_cast<QCtx*>(ctx);
  reps = std::max(1, reps);
  // candidates (d2v form, weights tile, d2v chunk): the slab form with the
  // chunks that give 1 to 4 rounds of its workgroups for this batch, and the
  // per-block form with fixed chunks
  const int saved[4] = {q->weights_tile, q->d2v_chunk, q->reorth_jtile, q->d2v_form};
  std::vector<std::array<int, 3>> cand;
  for (int wt : {64, 128, 256})
    for (int chk : {1024, 2048, 4096, 8192})
      if (chk <= q->N || chk == 1024) cand.push_back({0, wt, std::min(chk, q->N)});
  if (q->S) {
    q->d2v_form = 1;
    QBatch b0;
    if (build_batch(q, n_chains, iq_pert, q_pair_map, b0)) {
      q->d2v_form = saved[3];
      return -1;
    }
    const int nib = b0.nib;
    free_batch(b0);
    std::vector<int> ch;
    for (int r = 1; r <= 4; ++r) {
      const int c = slab_chunk(q, nib, r);
      if (std::find(ch.begin(), ch.end(), c) == ch.end()) ch.push_back(c);
    }
    for (int wt : {64, 128, 256})
      for (int c : ch) cand.push_back({1, wt, c});
  }
  hipStream_t s = q->stream;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
    q->d2v_form = saved[3];
    set_error("tdscha_qspace_autotune: event creation failed");
    return -1;
  }
  double best = 1e300;
  int bw = saved[0], bc = saved[1], bf = saved[3];
  double2 *dpsi = nullptr, *dout = nullptr;
  int rc = 0;
  for (const auto& cd : cand) {
    q->d2v_form = cd[0];
    q->weights_tile = cd[1];
    q->d2v_chunk = cd[2];
    QBatch b;
    rc = build_batch(q, n_chains, iq_pert, q_pair_map, b);
    if (rc) break;
    const size_t nbytes = sizeof(double2) * (size_t)n_chains * b.ld;
    if (!dpsi) {
      if (hipMalloc((void**)&dpsi, nbytes * 2) != hipSuccess ||
          hipMemset(dpsi, 0, nbytes * 2) != hipSuccess) {
        free_batch(b);
        set_error("tdscha_qspace_autotune: allocation failed");
        rc = -1;
        break;
      }
      dout = dpsi + (size_t)n_chains * b.ld;
    }
    launch_L(q, b, dpsi, dout, 0, 0, 0, s);   // warm-up
    (void)hipEventRecord(e0, s);
    for (int r = 0; r < reps; ++r) launch_L(q, b, dpsi, dout, 0, 0, 0, s);
    (void)hipEventRecord(e1, s);
    if (hipStreamSynchronize(s) != hipSuccess || hipGetLastError() != hipSuccess) {
      free_batch(b);
      set_error("tdscha_qspace_autotune: timing run failed");
      rc = -1;
      break;
    }
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, e0, e1);
    if (ms / reps < best) {
      best = ms / reps;
      bw = cd[1];
      bc = cd[2];
      bf = cd[0];
    }
    free_batch(b);
  }
  if (dpsi) (void)hipFree(dpsi);
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (rc) {
    q->weights_tile = saved[0];
    q->d2v_chunk = saved[1];
    q->reorth_jtile = saved[2];
    q->d2v_form = saved[3];
    return rc;
  }
  q->weights_tile = bw;
  q->d2v_chunk = bc;
  q->d2v_form = bf;
  if (tiles_out) {
    tiles_out[0] = q->weights_tile;
    tiles_out[1] = q->d2v_chunk;
    tiles_out[2] = q->reorth_jtile;
  }
  if (best_ms) *best_ms = best;
  return 0;
}

}  // extern "C"
