// Symmetrised perturbed averages from the orbit of the perturbation.
//
// With the S_j block diagonal over degenerate modes (on which fY and fpsi are
// constant), the average over all images is
//   T_sym(v) = (1 / n_syms) sum_j S_j T(S_j^T v),
// T the average over the configurations alone and v = (R1, Y1) with S^T v =
// (S^T R1, S^T Y1 S), S (f, d2v) = (S f, S d2v S^T) (rotate.hip).  T is
// linear, so when the n_syms rotated perturbations span only r dimensions,
//   S_j^T v = sum_k C_jk S_jk^T v   (k = 1 .. r),
//   T_sym(v) = (1 / n_syms) sum_j S_j sum_k C_jk T(S_jk^T v):
// r averages over the N configurations instead of one over N n_syms images.
// The perturbations of linear response have small orbits: r = 3 for an IR
// (vector) perturbation of a cubic crystal, at most 6 for a Raman (tensor) one,
// against 48 images.
//
// The rank is found for each chain and call from the perturbation itself: the
// row-dots of the averages (s1 = u.Y1.u, s2 = u.Y1.(fpsi f), s3 = (fY u).R1,
// s4 = f.R1) are evaluated on all images of kProbe random configurations of the
// thermal amplitudes: 2 kProbe functionals of R1 and as many of Y1.  A relation C that
// holds for both to kOrbTol of each one's size holds for the perturbation (random
// functionals: a remainder that all of them miss has probability zero, and one that
// the 10 beyond the rank understate tenfold 1e-11).  Otherwise the general form is
// used.  kOrbTol lies at the rounding of the symmetry tables: the images of an IR
// vector are 1e-14, those of a Raman tensor 2e-14 from their span on 381 modes (the
// tables are orthogonal to 1e-14).  The sum of |C| over an image, which the rounding of
// the averages enters with, is 2 and 5 there, and at most kOrbGain.
//
// A Lanczos run whose operator commutes with the symmetries (they form a group of
// orthogonal matrices and the translation average commutes with them, both checked
// numerically) keeps the relation C of its start vector, which is the one of all three
// parts of the packed vector: R and both pair sectors, A and B.  (Y1 = ca A - cb B alone
// would not do: ca is zero for pairs of equal frequencies, and for every pair at T = 0,
// and A and B can cancel.)  Rounding leaves that sector and the three-term recurrence
// amplifies it (about 5-fold per step), so the residual is projected back every
// kOrbClean steps with the same two kernels (0.2 ms for three chains of 381 modes).
// Spectra of the three IR chains, equal by symmetry, after 200
// FP64 steps at 128 atoms: apart by 3e-6 with a projection every third step, 1.2e-7
// every second and every step (4e-8 in the general form).
//
// The given tables are a representation to their own rounding, 1e-14, and the form uses
// that they are one: with exact arithmetic too, its averages of an IR vector are f 2e-15
// and d2v 7e-15 from the sum over the tables verbatim at 54 atoms (the general form's
// rounding: 6e-16), a whole application of L 1.7e-16 (1.5e-16).
//
// Measured, three IR vectors, one application of L in FP64 (host arrays in and out):
// 128 atoms x 20000 configurations x 48: 9 averages over 20,096 rows instead of
// three over 960,000 images, 29.1 -> 2.63 ms (weights 1.04, outer 1.04, rotations
// 0.13 ms); 54 atoms x 5000 x 48: 1.70 -> 0.42 ms.
#include <algorithm>
#include <cmath>
#include <random>
#include <vector>

#include "common.hpp"

namespace tdscha {

__global__ void expand_images(const double*, const double*, const double*, const int*, const int*,
                              const int*, const int*, const long*, const int*, const double*, int,
                              int, int, long, double*, double*, double*);
__global__ void rot_copy_configs(const double* X, const double* Y, const double* rho, int n, int np,
                                 long N, long Mp, double* U, double* F, double* rho_img);
int ensure_split(Ctx* c, int prec);
void free_split(Ctx* c);
int launch_pa_split(Ctx* c, int nc, int apply_d4, int prec, hipStream_t s, hipEvent_t* ev);
int rot_panels(const int* bs, const int* d, int n, int np, int* start, int* nreal);

constexpr int kOP = 32;          // modes of a panel (whole blocks)
constexpr int kOLd = kOP + 1;
constexpr int kLook = 8;         // symmetries and functionals of orbit_candidates

// ------------------------------------------------------------------- the probe
// row-dots of 16 probe rows over 16 columns of V = U Y1, a quarter of the K index
// per wave (the dots are linear in V); grid (rows / 16, ceil(n / 16), chains):
// many short work-groups, since the host waits for the result (31 us for three
// chains of 381 modes, 60 us with 64 rows to a work-group)
__global__ __launch_bounds__(256) void orb_probe(const double* __restrict__ U,
                                                 const double* __restrict__ F,
                                                 const double* __restrict__ Y1all,
                                                 const double* __restrict__ R1all,
                                                 const double* __restrict__ fy,
                                                 const double* __restrict__ fpsi, int np, int nk,
                                                 int rows, double* __restrict__ part) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lr = lane & 15, lg = lane >> 4, lq = lane & 3, lb = (lane >> 2) & 3;
  const int r0 = blockIdx.x * 16, c0 = blockIdx.y * 16, chain = blockIdx.z;
  const double* pu = U + (long)(r0 + lr) * np + lg;
  const double* py = Y1all + (long)chain * np * np + (long)lg * np + c0 + lr;
  const double* R1 = R1all + (long)chain * np;
  __shared__ double red[4][16][4];
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  for (int k0 = 16 * wave; k0 < nk; k0 += 64) {
    double a[4], b[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      a[k] = pu[k0 + 4 * k];
      b[k] = py[(long)(k0 + 4 * k) * np];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) mma16(a[k], b[k], acc);
  }
  const int row = r0 + 4 * lb + lg;
  double p[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int col = c0 + 4 * ((lb - r) & 3) + lq;
    const double u = U[(long)row * np + col], f = F[(long)row * np + col], r1 = R1[col];
    p[0] += acc[r] * u;
    p[1] += acc[r] * (f * fpsi[col]);
    if (wave == 0) {
      p[2] += u * (fy[col] * r1);
      p[3] += f * r1;
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    p[q] += __shfl_xor(p[q], 1);
    p[q] += __shfl_xor(p[q], 2);
  }
  red[wave][4 * lb + lg][lq] = lq < 2 ? (lq ? p[1] : p[0]) : (lq == 2 ? p[2] : p[3]);
  __syncthreads();
  if (wave == 0) {
    const int rr = lane >> 2;
    part[(((long)chain * gridDim.y + blockIdx.y) * rows + r0 + rr) * 4 + lq] =
        (red[0][rr][lq] + red[1][rr][lq]) + (red[2][rr][lq] + red[3][rr][lq]);
  }
}

__global__ void orb_probe_sum(const double* __restrict__ part, int ncol, int rows4,
                              double* __restrict__ out) {
  const int chain = blockIdx.y, e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= rows4) return;
  double s = 0.0;
#pragma unroll 8
  for (int c = 0; c < ncol; ++c) s += part[((long)chain * ncol + c) * rows4 + e];
  out[(long)chain * rows4 + e] = s;
}

// --------------------------------------------------------------- rotations
// Tiles of the panels (whole degenerate blocks, at most 32 modes): S_j is block
// diagonal, so a tile of S_j^T A S_j (or S_j A S_j^T) is a product of the tile of A
// with the two panels' diagonal parts of S_j, from tables padded with zeros to
// 32 x 32.  Four waves, one 16 x 16 quadrant each.
struct OrbPanels {
  const int* start;   // [npanel + 1]
  int npanel;
  int nsym;
  const double* S;    // [npanel, nsym, 32, 32]
  const double* ST;   // the same, transposed
};

// pair p = (source matrix, symmetry j): Yo[p] = S_j^T Y[src] S_j, Ro[p] =
// S_j^T R[src] (modes below n; the padding of Yo, Ro stays zero).  skip: see
// orb_out.
__global__ __launch_bounds__(256) void orb_in(OrbPanels pn, const int2* __restrict__ pairs,
                                              const double* __restrict__ Yb,
                                              const double* __restrict__ Rb, int np,
                                              const int* __restrict__ kk, int every,
                                              double* __restrict__ Yo, double* __restrict__ Ro) {
  if (every && (kk[0] % every) != every - 1) return;
  const int pi = blockIdx.x / pn.npanel, pj = blockIdx.x % pn.npanel, p = blockIdx.y;
  const int src = pairs[p].x, j = pairs[p].y;
  const int r0 = pn.start[pi], h = pn.start[pi + 1] - r0;
  const int q0 = pn.start[pj], w = pn.start[pj + 1] - q0;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wr = 16 * (wave >> 1), wc = 16 * (wave & 1);
  const int lr = lane & 15, lg = lane >> 4, lq = lane & 3, lb = (lane >> 2) & 3;
  __shared__ double T[kOP][kOLd];
  const double* Si = pn.S + ((long)pi * pn.nsym + j) * kOP * kOP;
  const double* Sj = pn.S + ((long)pj * pn.nsym + j) * kOP * kOP;
  const double* Y = Yb + (long)src * np * np;
  double a[8], b[8], s[8];
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) {
    const int k = 4 * ks + lg;
    a[ks] = Si[k * kOP + wr + lr];
    const bool in = k < h && wc + lr < w;
    b[ks] = in ? Y[(long)(r0 + k) * np + q0 + wc + lr] : 0.0;
    s[ks] = Sj[k * kOP + wc + lr];
  }
  double t[4] = {0.0, 0.0, 0.0, 0.0}, o[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) mma16(a[ks], b[ks], t);
#pragma unroll
  for (int r = 0; r < 4; ++r) T[wr + 4 * lb + lg][wc + 4 * ((lb - r) & 3) + lq] = t[r];
  __syncthreads();
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) mma16(T[wr + lr][4 * ks + lg], s[ks], o);
  const int row = wr + 4 * lb + lg;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int col = wc + 4 * ((lb - r) & 3) + lq;
    if (row < h && col < w) Yo[(long)p * np * np + (long)(r0 + row) * np + q0 + col] = o[r];
  }
  if (pj == 0 && (int)threadIdx.x < h) {
    const double* R = Rb + (long)src * np + r0;
    double v = 0.0;
    for (int m = 0; m < h; ++m) v += Si[m * kOP + threadIdx.x] * R[m];
    Ro[(long)p * np + r0 + threadIdx.x] = v;
  }
}

// Matrix (first pair, rank, relation, m): sum_j S_j (sum_k C_jk D_k) S_j^T and
// sum_j S_j sum_k C_jk f_k.  AVG: D_k = fY Z_k + (fY Z_k)^T of the raw outer
// sums, results to f_out, d_out (both halves) of chain m.  Else D_k the symmetric inputs,
// results to the packed vectors x [chain][n + 2 P] (m = 2 chain + sector; R
// with sector 0), in which case the kernel runs only on every `every`-th step.
// RM: largest rank of the plan (3, or kOrbRank).  grid (panel pairs pi <= pj, then
// panels for f; matrices); per symmetry a wave combines D in registers (its 16 rows),
// and the product with S_pj^T passes through LDS.  Bound by the latency of that chain:
// two groups of four waves take every other symmetry, every load is unconditional,
// rank 3 leaves two work-groups to a CU, and f has work-groups of its own (with
// conditional loads and f behind its diagonal tile: 97 us for three matrices of 159
// modes and 185 of 381; 59 and 101 now).
template <bool AVG, int RM>
__global__ __launch_bounds__(512, RM > 3 ? 2 : 4) void orb_out(
    OrbPanels pn, const int4* __restrict__ mats, const double* __restrict__ C,
    const double* __restrict__ Zb, const double* __restrict__ fb, const double* __restrict__ fy,
    int n, int np, double normf, double normd, const int* __restrict__ kk, int every,
    const int* __restrict__ active, double* __restrict__ f_out, double* __restrict__ d_out) {
  if (every && (kk[0] % every) != every - 1) return;
  const int4 mt = mats[blockIdx.y];
  const int m = mt.w;
  if (!AVG && !active[m >> 1]) return;
  const int ntile = pn.npanel * (pn.npanel + 1) / 2;
  const bool isf = (int)blockIdx.x >= ntile;
  int pj = 0, pi = blockIdx.x;
  if (isf)
    pi = pj = blockIdx.x - ntile;
  else
    while (pi > pj) pi -= ++pj;   // pair (pi, pj), pi <= pj
  const int r0 = pn.start[pi], h = pn.start[pi + 1] - r0;
  const int q0 = pn.start[pj], w = pn.start[pj + 1] - q0;
  const int lane = threadIdx.x & 63, wave = (threadIdx.x >> 6) & 3;
  const int half = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8);
  const int wr = 16 * (wave >> 1), wc = 16 * (wave & 1);
  const int lr = lane & 15, lg = lane >> 4, lq = lane & 3, lb = (lane >> 2) & 3;
  __shared__ double T[2][2][kOP][kOLd];
  const long nn = (long)np * np;
  const int rank = mt.y;
  const double* Cm = C + (long)mt.z * pn.nsym * kOrbRank;
  if (isf) {
    // f of a panel, sixteen symmetries at a time: h_j = sum_k C_jk f_k in LDS, then
    // S_j h_j, thread = (mode, symmetry)
    if (!AVG && (m & 1)) return;
    double(*hs)[kOP] = reinterpret_cast<double(*)[kOP]>(&T[0][0][0][0]);   // [16][32]
    double(*part)[kOP] = reinterpret_cast<double(*)[kOP]>(&T[1][0][0][0]); // [16][32]
    const int t = threadIdx.x & 31, sl = threadIdx.x >> 5;
    const double* St = pn.ST + (long)pi * pn.nsym * kOP * kOP + t;
    double fk[RM], v = 0.0;
#pragma unroll
    for (int k = 0; k < RM; ++k) {
      const double f = fb[(long)(mt.x + min(k, rank - 1)) * np + r0 + min(t, h - 1)];
      fk[k] = k < rank && t < h ? f : 0.0;
    }
    for (int j0 = 0; j0 < pn.nsym; j0 += 16) {
      const int j = min(j0 + sl, pn.nsym - 1);
      double st[kOP], x = 0.0;
#pragma unroll
      for (int b = 0; b < kOP; ++b) st[b] = St[((long)j * kOP + b) * kOP];
#pragma unroll
      for (int k = 0; k < RM; ++k) x += Cm[j * kOrbRank + k] * fk[k];   // (zero from rank on)
      __syncthreads();
      hs[sl][t] = j0 + sl < pn.nsym ? x : 0.0;
      __syncthreads();
#pragma unroll
      for (int b = 0; b < kOP; ++b) v += st[b] * hs[sl][b];
    }
    part[sl][t] = v;
    __syncthreads();
    if ((int)threadIdx.x < h) {
      double f = 0.0;
#pragma unroll
      for (int q = 0; q < 16; ++q) f += part[q][t];
      if (AVG)
        f_out[(long)m * n + r0 + t] = normf * f;
      else
        d_out[(m >> 1) * (n + (long)n * (n + 1)) + r0 + t] = normf * f;
    }
    return;
  }
  // (loads clamped to the tile, not conditional: all of them in flight)
  double d[RM][8];
#pragma unroll
  for (int k = 0; k < RM; ++k) {
    const double* z = Zb + (long)(mt.x + min(k, rank - 1)) * nn;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      const int a = wr + lr, b = 4 * ks + lg;
      const int ga = r0 + min(a, h - 1), gb = q0 + min(b, w - 1);
      double v = z[(long)ga * np + gb];
      if (AVG) v = fy[ga] * v + fy[gb] * z[(long)gb * np + ga];
      d[k][ks] = k < rank && a < h && b < w ? v : 0.0;
    }
  }
  const double* Ti = pn.ST + (long)pi * pn.nsym * kOP * kOP + wr + lr;
  const double* Tj = pn.ST + (long)pj * pn.nsym * kOP * kOP + wc + lr;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  // the halves take every other symmetry (weight zero past the last)
  for (int jj = 0; jj < pn.nsym; jj += 2) {
    const int jc = min(jj + half, pn.nsym - 1);
    const long o = (long)jc * kOP * kOP + lg * kOP;
    double sj[8], si[8], mm[8];
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      sj[ks] = Tj[o + 4 * ks * kOP];
      si[ks] = Ti[o + 4 * ks * kOP];
      mm[ks] = 0.0;
    }
#pragma unroll
    for (int k = 0; k < RM; ++k) {   // (zero from rank on)
      const double c = jj + half < pn.nsym ? Cm[jc * kOrbRank + k] : 0.0;
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) mm[ks] += c * d[k][ks];
    }
    double t[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) mma16(mm[ks], sj[ks], t);
    double(*Tb)[kOLd] = T[half][(jj >> 1) & 1];
#pragma unroll
    for (int r = 0; r < 4; ++r) Tb[wr + 4 * lb + lg][wc + 4 * ((lb - r) & 3) + lq] = t[r];
    __syncthreads();   // (the other buffer was last read before this barrier)
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) mma16(si[ks], Tb[4 * ks + lg][wc + lr], acc);
  }
  __syncthreads();
  double(*sum)[kOP * kOP / 4] = reinterpret_cast<double(*)[kOP * kOP / 4]>(&T[0][0][0][0]);
  if (half)
#pragma unroll
    for (int r = 0; r < 4; ++r) sum[r][threadIdx.x & 255] = acc[r];
  __syncthreads();
  if (!half)
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[r] += sum[r][threadIdx.x];
  const int row = wr + 4 * lb + lg;
  const long P = (long)n * (n + 1) / 2, len = n + 2 * P;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int col = wc + 4 * ((lb - r) & 3) + lq;
    if (half || row >= h || col >= w) continue;
    const int gr = r0 + row, gc = q0 + col;
    const double v = normd * acc[r];
    if (AVG) {
      if (gr > gc) continue;   // exactly symmetric
      double* o = d_out + (long)m * n * n;
      o[(long)gr * n + gc] = v;
      o[(long)gc * n + gr] = v;
    } else if (gr <= gc) {
      const long p = (long)gr * n - (long)gr * (gr - 1) / 2 + (gc - gr);
      d_out[(m >> 1) * len + n + (m & 1) * P + p] = v;
    }
  }
}

// packed vectors -> symmetric padded matrices [2 chain + sector] and R (zero for
// sector 1)
__global__ void orb_unpack(const double* __restrict__ x, int n, int np,
                           const int* __restrict__ kk, int every, double* __restrict__ Yb,
                           double* __restrict__ Rb) {
  if (every && (kk[0] % every) != every - 1) return;
  const int m = blockIdx.y;
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (long)np * np) return;
  const int a = (int)(e / np), b = (int)(e % np);
  const long P = (long)n * (n + 1) / 2, len = n + 2 * P;
  const double* v = x + (m >> 1) * len;
  double y = 0.0;
  if (a < n && b < n) {
    const int r = a < b ? a : b, c = a < b ? b : a;
    y = v[n + (m & 1) * P + (long)r * n - (long)r * (r - 1) / 2 + (c - r)];
  }
  Yb[(long)m * np * np + e] = y;
  if (e < np) Rb[(long)m * np + e] = (e < n && (m & 1) == 0) ? v[e] : 0.0;
}

// --------------------------------------------------------------------- tables
// panel parts of S_j, and transposed: grid (panels, symmetries), 1024 threads
__global__ void orb_tables(const int* __restrict__ start, const int* __restrict__ mode_block,
                           const int* __restrict__ mode_pos, const int* __restrict__ block_dim,
                           const long* __restrict__ block_soff, const double* __restrict__ syms,
                           int nsym, double* __restrict__ S, double* __restrict__ ST) {
  const int q = blockIdx.x, j = blockIdx.y, x = threadIdx.x >> 5, y = threadIdx.x & 31;
  const int r = start[q] + x, c = start[q] + y, e = start[q + 1];
  double v = 0.0;
  if (r < e && c < e && mode_block[r] == mode_block[c]) {
    const int b = mode_block[r], d = block_dim[b];
    v = syms[block_soff[b] + ((long)j * d + mode_pos[r]) * d + mode_pos[c]];
  }
  const long base = ((long)q * nsym + j) * kOP * kOP;
  S[base + x * kOP + y] = v;
  ST[base + y * kOP + x] = v;
}

// Whether the tables allow the orbit form: blocks of consecutive modes (at most
// 32) on which fY and fpsi are constant to 1e-13.
static bool blocks_fit(const Ctx* c, int n_blocks, const int* block_dim, const int* block_modes,
                       const std::vector<double>& fy) {
  int off = 0;
  for (int b = 0; b < n_blocks; ++b) {
    const int d = block_dim[b];
    if (d > kOP) return false;
    double lo = 1e300, hi = 0.0;
    for (int k = 0; k < d; ++k) {
      if (block_modes[off + k] != block_modes[off] + k) return false;
      lo = std::min(lo, fy[block_modes[off + k]]);
      hi = std::max(hi, fy[block_modes[off + k]]);
    }
    if (!(hi - lo <= 1e-13 * hi)) return false;
    off += d;
  }
  return true;
}

// S_j z (or S_j^T z)
static void apply_s(const Ctx* c, const std::vector<double>& syms, int j, bool transpose,
                    const double* z, double* out) {
  const Orbit& o = c->orb;
  long so = 0;
  int off = 0;
  for (int d : c->block_dim) {
    const double* S = syms.data() + so + (long)j * d * d;
    const int m0 = c->block_modes[off];
    for (int a = 0; a < d; ++a) {
      double v = 0.0;
      for (int b = 0; b < d; ++b) v += (transpose ? S[b * d + a] : S[a * d + b]) * z[m0 + b];
      out[m0 + a] = v;
    }
    so += (long)o.nsym * d * d;
    off += d;
  }
}

static double dot(const double* x, const double* y, int n) {
  double s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  int m = 0;
  for (; m + 8 <= n; m += 8)
    for (int k = 0; k < 8; ++k) s[k] += x[m + k] * y[m + k];
  for (; m < n; ++m) s[0] += x[m] * y[m];
  return ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
}

// Whether the S_j are a group of orthogonal matrices (then S_j^T, which takes the
// perturbation to its image, is one of them, and T_sym commutes with all).  Closed under
// multiplication: p.S_i S_j z equals p.S_k z for one k for two independent random pairs
// (p, z), to 1e-9 of their size.  Elements become generators until the products with
// them reach the whole list; every one of these products has to be in the list (then
// the list is the group they generate).
static bool closed(Ctx* c) {
  Orbit& o = c->orb;
  const int ns = o.nsym, n = c->n;
  std::mt19937_64 g(12345);
  std::normal_distribution<double> nd;
  std::vector<double> A[2], z[2], ref(2 * (size_t)ns), sz(n);
  for (int t = 0; t < 2; ++t) {
    std::vector<double> p(n);
    z[t].resize(n);
    for (double& v : p) v = nd(g);
    for (double& v : z[t]) v = nd(g);
    A[t].resize((size_t)ns * n);
    for (int j = 0; j < ns; ++j) {
      double* a = A[t].data() + (size_t)j * n;
      apply_s(c, o.syms, j, true, p.data(), a);
      ref[2 * (size_t)j + t] = dot(a, z[t].data(), n);
    }
  }
  const double tol = 1e-9 * n;
  std::vector<int> order(ns);
  for (int j = 0; j < ns; ++j) order[j] = j;
  std::sort(order.begin(), order.end(),
            [&](int a, int b) { return ref[2 * (size_t)a] < ref[2 * (size_t)b]; });
  std::vector<double> gz[2];   // S_q z of each generator q
  auto product = [&](int i, int q) {
    double v[2];
    for (int t = 0; t < 2; ++t)
      v[t] = dot(A[t].data() + (size_t)i * n, gz[t].data() + (size_t)q * n, n);
    auto it = std::lower_bound(order.begin(), order.end(), v[0] - tol,
                               [&](int a, double x) { return ref[2 * (size_t)a] < x; });
    for (; it != order.end() && ref[2 * (size_t)*it] <= v[0] + tol; ++it)
      if (std::fabs(ref[2 * (size_t)*it + 1] - v[1]) <= tol) return *it;
    return -1;
  };
  std::vector<char> in(ns, 0);
  std::vector<int> sub;
  o.gens.clear();
  for (int j = 0; j < ns; ++j) {
    if (in[j]) continue;
    for (int t = 0; t < 2; ++t) {
      apply_s(c, o.syms, j, false, z[t].data(), sz.data());
      gz[t].insert(gz[t].end(), sz.begin(), sz.end());
    }
    o.gens.push_back(j);
    in[j] = 1;
    sub.push_back(j);
    for (size_t a = 0; a < sub.size(); ++a)
      for (size_t q = 0; q < o.gens.size(); ++q) {
        const int k = product(sub[a], (int)q);
        if (k < 0) return false;
        if (!in[k]) {
          in[k] = 1;
          sub.push_back(k);
        }
      }
  }
  // the generators orthogonal: S_q^T S_q z is z
  std::vector<double> back(n);
  double scale = 0.0;
  for (double v : z[0]) scale = std::max(scale, std::fabs(v));
  for (size_t q = 0; q < o.gens.size(); ++q) {
    apply_s(c, o.syms, o.gens[q], true, gz[0].data() + q * n, back.data());
    for (int m = 0; m < n; ++m)
      if (!(std::fabs(back[m] - z[0][m]) <= 1e-9 * scale)) return false;
  }
  return true;
}

// Whether the translation average commutes with the group's generators, on random
// vectors: the mean projector (proj z against its rotation), and the second
// moment over the permutations that the average of d2v applies.
static bool orbit_translations(Ctx* c, int n_cart, const double* pols, int n_cells, const int* inv_perms,
                        const double* proj) {
  const Orbit& o = c->orb;
  const int n = c->n;
  std::mt19937_64 g(777);
  std::normal_distribution<double> nd;
  std::vector<double> z(n), p(n), sz(n), sp(n), u(n), v(n), t(n);
  std::vector<double> cz(n_cart), cp(n_cart), csz(n_cart), csp(n_cart);
  for (double& x : z) x = nd(g);
  for (double& x : p) x = nd(g);
  auto matvec = [&](const double* M, int rows, const std::vector<double>& x,
                    std::vector<double>& y) {
    for (int a = 0; a < rows; ++a) y[a] = dot(M + (size_t)a * n, x.data(), n);
  };
  // sum over t of (p . T_t z)^2, T_t = pols^T P_t pols: (P_t x)[a] = x[inv_perm_t[a]]
  auto second = [&](const std::vector<double>& pc, const std::vector<double>& zc) {
    double s = 0.0;
    for (int q = 0; q < n_cells; ++q) {
      double d = 0.0;
      for (int a = 0; a < n_cart; ++a) d += pc[a] * zc[inv_perms[(size_t)q * n_cart + a]];
      s += d * d;
    }
    return s;
  };
  matvec(proj, n, z, t);
  matvec(pols, n_cart, z, cz);
  matvec(pols, n_cart, p, cp);
  double scale = 0.0;
  for (int m = 0; m < n; ++m) scale = std::max(scale, std::fabs(z[m]));
  for (int j : o.gens) {
    apply_s(c, o.syms, j, false, z.data(), sz.data());
    apply_s(c, o.syms, j, false, t.data(), v.data());
    apply_s(c, o.syms, j, true, p.data(), sp.data());
    matvec(proj, n, sz, u);
    for (int m = 0; m < n; ++m)
      if (!(std::fabs(u[m] - v[m]) <= 1e-9 * scale)) return false;
    matvec(pols, n_cart, sz, csz);
    matvec(pols, n_cart, sp, csp);
    const double s1 = second(cp, csz), s2 = second(csp, cz);
    if (!(std::fabs(s1 - s2) <= 1e-9 * (std::fabs(s1) + std::fabs(s2)))) return false;
  }
  return true;
}

// Whether the operator commutes with the symmetries: they form a group, which commutes
// with the translation average.  Checked once per context, by its first Lanczos run
// that may use it (1.3 ms on the host at 381 modes).
int orbit_sector(Ctx* c, bool* ok) {
  Orbit& o = c->orb;
  if (o.group < 0) o.group = closed(c);
  if (o.group && c->n_cells > 0 && o.trans < 0) {
    const size_t n = c->n, nc = c->n_cart;
    std::vector<double> pols(nc * n), pt(n * n), proj(n * n);
    std::vector<int> perms((size_t)c->n_cells * nc);
    TDS_CHECK_HIP(hipMemcpy(pols.data(), c->pols, sizeof(double) * pols.size(),
                            hipMemcpyDeviceToHost));
    TDS_CHECK_HIP(hipMemcpy(pt.data(), c->tproj, sizeof(double) * pt.size(),
                            hipMemcpyDeviceToHost));
    TDS_CHECK_HIP(hipMemcpy(perms.data(), c->inv_perms, sizeof(int) * perms.size(),
                            hipMemcpyDeviceToHost));
    for (size_t a = 0; a < n; ++a)   // (kept transposed on the device)
      for (size_t b = 0; b < n; ++b) proj[a * n + b] = pt[b * n + a];
    o.trans = orbit_translations(c, c->n_cart, pols.data(), c->n_cells, perms.data(), proj.data());
  }
  *ok = o.group && (c->n_cells == 0 || o.trans);
  return 0;
}

// Time of the GEMM pairs of one chain over `rows` images: 55 TF/s in FP64 (columns in
// sixteens); the split kernels compute whole 128-column tiles, 270 TF/s (two chains of
// 381 modes, counted once, not three times) to 500 TF/s (three of 159).
static double estimate_us(const Ctx* c, double rows, int prec) {
  const double w = round_up(c->n, prec == PREC_FP64 ? 16 : kTile);
  return 4.0 * rows * w * w / (prec == PREC_FP64 ? 5.5e7 : 4e8);
}

// Whether the form may save enough for one chain in this precision.  Per chain, so that
// a chain's form, and with it its rounding, does not depend on its batch.
bool orbit_sized(const Ctx* c, int prec) {
  const Orbit& o = c->orb;
  return o.usable && c->row_lo == 0 && c->row_hi == c->M &&
         estimate_us(c, (double)c->N * (o.nsym - 1), prec) > kOrbWorthUs;
}

// The configurations, panel tables and probe rows; called at context creation
// with the configurations still on the device.  Leaves c->orb.usable false where
// the form does not apply or cannot pay in any precision (orbit_sized), or with more
// than 512 symmetries (the tables and the closure check grow with their number and its
// square).
int orbit_setup(Ctx* c, int n_syms, int n_blocks, const int* block_dim, const int* block_modes,
                const std::vector<double>& syms, const double* X_dev, const double* Y_dev,
                const double* rho_dev, const int* d_mb, const int* d_mp, const int* d_bd,
                const int* d_bmo, const long* d_bso, const int* d_bm, const double* d_syms) {
  Orbit& o = c->orb;
  o.nsym = n_syms;
  if (n_syms < 4 || n_syms > 512) return 0;
  const double saved = (double)c->N * (n_syms - 1);
  if (std::max(estimate_us(c, saved, PREC_FP64), estimate_us(c, saved, PREC_FP16X2)) <= kOrbWorthUs)
    return 0;
  const int n = c->n, np = c->np;
  std::vector<double> fy(np);
  TDS_CHECK_HIP(hipMemcpy(fy.data(), c->fy, sizeof(double) * np, hipMemcpyDeviceToHost));
  if (!blocks_fit(c, n_blocks, block_dim, block_modes, fy)) return 0;
  // panels
  std::vector<int> bs(n), dd(n), start(n + 2);
  {
    int off = 0;
    for (int b = 0; b < n_blocks; ++b)
      for (int k = 0, o0 = off; k < block_dim[b]; ++k, ++off) {
        bs[block_modes[off]] = block_modes[o0];
        dd[block_modes[off]] = block_dim[b];
      }
  }
  int nreal = 0;
  rot_panels(bs.data(), dd.data(), n, np, start.data(), &nreal);
  o.npanel = nreal;
  start[nreal] = n;
  const size_t ntab = (size_t)nreal * n_syms * kOP * kOP;
  o.syms = syms;
  const int look = std::min(n_syms, kLook);
  o.look.resize((size_t)look * kLook * n);
  // probe configurations: thermal amplitudes for x; forces of the same weight
  // in s2 = u.Y1.(fpsi f) as x has in s1
  std::mt19937_64 g(2024);
  std::normal_distribution<double> nd;
  std::vector<double> px((size_t)kProbe * n), py(px.size()), ones(kProbe, 1.0);
  for (int i = 0; i < kProbe; ++i)
    for (int m = 0; m < n; ++m) {
      px[(size_t)i * n + m] = nd(g) / std::sqrt(fy[m]);
      py[(size_t)i * n + m] = nd(g) * std::sqrt(fy[m]);
    }
  // (symmetries drawn from the whole list: the first ones often leave an axis alone)
  std::vector<int> pick(n_syms);
  for (int j = 0; j < n_syms; ++j) pick[j] = j;
  for (int j = 0; j < look; ++j) std::swap(pick[j], pick[j + g() % (n_syms - j)]);
  std::vector<double> pv(n);
  for (int i = 0; i < kLook; ++i) {
    for (double& v : pv) v = nd(g);
    for (int j = 0; j < look; ++j)
      apply_s(c, o.syms, pick[j], false, pv.data(), o.look.data() + ((size_t)j * kLook + i) * n);
  }
  o.rows = round_up(kProbe * n_syms, 16);
  // one allocation: tables, probe rows, and the inputs of the kernels that fill them
  size_t at = 0;
  auto place = [&](size_t count) {
    const size_t here = at;
    at += (count + 31) / 32 * 32;
    return here;
  };
  o.Mp = c->rotate ? c->Mp : round_up_l(c->N, 128);
  const size_t np_rows = (size_t)o.rows * np, own = c->rotate ? 0 : (size_t)o.Mp;
  const size_t aS = place(ntab), aST = place(ntab), apu = place(np_rows), apf = place(np_rows),
               apo = place(o.rows), adx = place(px.size()), ady = place(py.size()),
               ad1 = place(ones.size()), ast = place(nreal + 1), aU = place(own * np),
               aF = place(own * np), arho = place(own);
  auto up = [](void* dst, const void* src, size_t bytes) {
    return hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice) == hipSuccess;
  };
  o.arena_bytes = sizeof(double) * at;
  if (hipMalloc((void**)&o.arena, o.arena_bytes) != hipSuccess) {
    (void)hipGetLastError();   // no room: the general form serves every call
    o.arena = nullptr;
    return 0;
  }
  o.S = o.arena + aS; o.ST = o.arena + aST;
  o.pu = o.arena + apu; o.pf = o.arena + apf; o.pones = o.arena + apo;
  o.start = reinterpret_cast<int*>(o.arena + ast);
  double *dx = o.arena + adx, *dy = o.arena + ady, *d1 = o.arena + ad1;
  bool ok = up(dx, px.data(), sizeof(double) * px.size()) &&
       up(dy, py.data(), sizeof(double) * py.size()) &&
       up(d1, ones.data(), sizeof(double) * ones.size()) &&
       up(o.start, start.data(), sizeof(int) * (nreal + 1));
  if (ok) {
    hipLaunchKernelGGL(orb_tables, dim3(nreal, n_syms), dim3(1024), 0, c->stream, o.start, d_mb,
                       d_mp, d_bd, d_bso, d_syms, n_syms, o.S, o.ST);
    hipLaunchKernelGGL(expand_images, dim3((unsigned)o.rows, (np + 127) / 128), dim3(128), 0,
                       c->stream, dx, dy, d1, d_mb, d_mp, d_bd, d_bmo, d_bso, d_bm, d_syms, n, np,
                       n_syms, (long)kProbe * n_syms, o.pu, o.pf, o.pones);
    if (c->rotate) {   // its rows are the configurations
      o.U = c->U;
      o.F = c->F;
      o.rho = c->rho_img;
    } else {
      o.U = o.arena + aU;
      o.F = o.arena + aF;
      o.rho = o.arena + arho;
      const long count = o.Mp * np;
      hipLaunchKernelGGL(rot_copy_configs, dim3((unsigned)((count + 255) / 256)), dim3(256), 0,
                         c->stream, X_dev, Y_dev, rho_dev, n, np, (long)c->N, o.Mp, o.U, o.F,
                         o.rho);
    }
  }
  ok = ok && hipGetLastError() == hipSuccess && hipStreamSynchronize(c->stream) == hipSuccess;
  if (!ok) {
    set_error("tdscha_ctx_create: tables of the orbit form failed");
    return -1;
  }
  o.usable = true;
  return 0;
}

static void drop_sub(Orbit& o) {
  if (!o.sub) return;
  free_split(o.sub);
  delete o.sub;   // (its rows, inputs and outputs belong to this struct)
  o.sub = nullptr;
}

void orbit_free(Ctx* c) {
  Orbit& o = c->orb;
  drop_sub(o);
  if (o.arena) (void)hipFree(o.arena);
  if (o.work) (void)hipFree(o.work);
  if (o.pout) (void)hipHostFree(o.pout);
  for (OrbPlan& pl : o.plan) orbit_plan_free(pl);
}

void orbit_plan_free(OrbPlan& p) {
  if (p.dev) (void)hipFree(p.dev);
  if (p.general) (void)hipFree(p.general);
  p.dev = nullptr;
  p.general = nullptr;
  p.cap = 0;
  p.ok = false;
}

// K split of the outer product over the configurations: the same whatever the
// number of pairs, so that a chain's sums do not depend on its batch
static int orb_ksplit(const Ctx* c) {
  const int t = f64_tiles(c->n).ntile;
  int ks = std::min(24, round_up((2048 + 3 * t * t - 1) / (3 * t * t), 8));
  while (ks > 8 && (long)ks * 128 > c->orb.Mp) ks -= 8;
  return ks;
}

// workspaces of the orbit form (the partial sums are the context's, idle in these
// calls); false = no room: the general form serves this call
static bool ensure(Ctx* c, hipStream_t s) {
  Orbit& o = c->orb;
  if (o.work) return true;
  const size_t np = c->np, nn = np * np;
  const int ncol = (c->n + 15) / 16;
  const size_t count[] = {2 * (size_t)kMaxChains * ncol * o.rows * 4,
                          kOrbPairs * np, kOrbPairs * nn,
                          2 * kMaxChains * np, 2 * kMaxChains * nn,
                          kOrbPairs * (size_t)o.Mp * 4,
                          kOrbPairs * nn, kOrbPairs * np};
  double** dst[] = {&o.ppart, &o.R1, &o.Y1, &o.Rb, &o.Yb, &o.coef, &o.z, &o.f};
  size_t at = 0;
  for (size_t k : count) at += (k + 31) / 32 * 32;
  const size_t nout = 2 * (size_t)kMaxChains * o.rows * 4;
  if (!o.pout && hipHostMalloc((void**)&o.pout, sizeof(double) * nout) != hipSuccess)
    o.pout = nullptr;
  if (!o.pout || hipMalloc((void**)&o.work, sizeof(double) * at) != hipSuccess) {
    (void)hipGetLastError();
    o.work = nullptr;
    return false;
  }
  at = 0;
  for (size_t k = 0; k < sizeof(count) / sizeof(count[0]); ++k) {
    *dst[k] = o.work + at;
    at += (count[k] + 31) / 32 * 32;
  }
  // the padding of the rotated inputs is never written
  if (hipMemsetAsync(o.R1, 0, sizeof(double) * kOrbPairs * np, s) != hipSuccess ||
      hipMemsetAsync(o.Y1, 0, sizeof(double) * kOrbPairs * nn, s) != hipSuccess ||
      hipStreamSynchronize(s) != hipSuccess) {
    (void)hipGetLastError();
    (void)hipFree(o.work);
    o.work = nullptr;
    return false;
  }
  return true;
}

// Device memory of the context for anything but the orbit form, which gives way: first
// its workspaces and split images (made again by the next call that has room for them),
// then, where that is enough, its tables and configurations (the general form from then
// on).  A plan's own arrays stay.
hipError_t dev_alloc(Ctx* c, void** p, size_t bytes) {
  Orbit& o = c->orb;
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipSuccess && (o.work || o.sub)) {
    (void)hipGetLastError();
    (void)hipStreamSynchronize(c->stream);
    drop_sub(o);
    if (o.work) (void)hipFree(o.work);
    o.work = nullptr;
    e = hipMalloc(p, bytes);
  }
  size_t left = 0, all = 0;
  if (e != hipSuccess && o.arena && hipMemGetInfo(&left, &all) == hipSuccess &&
      left + o.arena_bytes >= bytes) {
    (void)hipGetLastError();
    (void)hipStreamSynchronize(c->stream);
    (void)hipFree(o.arena);
    o.arena = nullptr;
    o.usable = false;
    e = hipMalloc(p, bytes);
  }
  if (e != hipSuccess) {
    (void)hipGetLastError();
    *p = nullptr;
  }
  return e;
}

// ----------------------------------------------------------------- the relation
// Rank and relation of one chain: row j of W holds the functionals of `dots` of the
// image j, each kind scaled to unit size, so that the relation holds for every part of
// the perturbation to kOrbTol of that part's own size (f comes from Y1 alone, and
// without apply_d4 d2v from R1 alone).  A kind that is zero throughout obeys any
// relation.  Pivoted Gram-Schmidt; rank 0 = no use.
struct Dots {
  const double* s;   // row-dots [kProbe][ns][4] of one matrix and vector
  int q;             // which of the four
};

static int relation(const std::vector<Dots>& dots, int ns, std::vector<int>& piv,
                    std::vector<double>& C) {
  const int nd = (int)dots.size(), K = nd * kProbe;
  std::vector<double> W((size_t)ns * K);
  bool some = false;
  for (int d = 0; d < nd; ++d) {
    // scaled by the largest entry (whose square may be out of range), then by the rms
    double top = 0.0, sum = 0.0, sq = 0.0;
    const double* p = dots[d].s + dots[d].q;
    for (int e = 0; e < ns * kProbe; ++e) {
      top = std::max(top, std::fabs(p[4 * e]));
      sum += p[4 * e];
    }
    if (!std::isfinite(sum) || (top > 0.0 && top < 1e-290)) return 0;   // (too few digits)
    if (top == 0.0) continue;
    some = true;
    for (int i = 0; i < kProbe; ++i)
      for (int j = 0; j < ns; ++j) {
        double& w = W[(size_t)j * K + d * kProbe + i];
        w = p[4 * (i * ns + j)] / top;
        sq += w * w;
      }
    const double inv = 1.0 / std::sqrt(sq / ns);
    for (int j = 0; j < ns; ++j)
      for (int i = 0; i < kProbe; ++i) W[(size_t)j * K + d * kProbe + i] *= inv;
  }
  if (!some) return 0;
  std::vector<double> V = W, Q;
  piv.clear();
  double top = 0.0;
  std::vector<double> nrm(ns);
  for (;;) {
    int best = 0;
    for (int j = 0; j < ns; ++j) {
      nrm[j] = std::sqrt(dot(V.data() + (size_t)j * K, V.data() + (size_t)j * K, K));
      if (nrm[j] > nrm[best]) best = j;
    }
    if (piv.empty()) top = nrm[best];
    if (nrm[best] <= kOrbTol * top) break;
    // (a direction this weak is known to too few digits)
    if (nrm[best] < 1e-3 * top || (int)piv.size() == kOrbRank) return 0;
    piv.push_back(best);
    const size_t r = piv.size() - 1;
    Q.resize((r + 1) * K);
    double* qr = Q.data() + r * K;
    for (int e = 0; e < K; ++e) qr[e] = V[(size_t)best * K + e] / nrm[best];
    for (int j = 0; j < ns; ++j)   // twice: the second pass takes what rounding left
      for (int pass = 0; pass < 2; ++pass) {
        double* v = V.data() + (size_t)j * K;
        const double t = dot(v, qr, K);
        for (int e = 0; e < K; ++e) v[e] -= t * qr[e];
      }
  }
  // W_j = sum_k C_jk W_piv[k]: with W Q^T = A, C A_piv = A (A_piv lower triangular)
  const int r = (int)piv.size();
  std::vector<double> A((size_t)ns * r);
  for (int j = 0; j < ns; ++j)
    for (int k = 0; k < r; ++k) {
      A[(size_t)j * r + k] = dot(W.data() + (size_t)j * K, Q.data() + (size_t)k * K, K);
    }
  C.assign((size_t)ns * kOrbRank, 0.0);
  for (int j = 0; j < ns; ++j)
    for (int k = r - 1; k >= 0; --k) {
      double t = A[(size_t)j * r + k];
      for (int l = k + 1; l < r; ++l) t -= C[(size_t)j * kOrbRank + l] * A[(size_t)piv[l] * r + k];
      C[(size_t)j * kOrbRank + k] = t / A[(size_t)piv[k] * r + k];
    }
  // the rounding of the averages enters with the factors C
  for (int j = 0; j < ns; ++j) {
    double sum = 0.0;
    for (int k = 0; k < r; ++k) sum += std::fabs(C[(size_t)j * kOrbRank + k]);
    if (!(sum <= kOrbGain)) return 0;
  }
  return r;
}

// The chains (bit mask) to look for a plan of: the general form is long enough for the
// rank that the chain's R vector (host, `ld` apart) shows at least.  R is looked at
// through kLook random functionals p of its images under kLook random symmetries,
// p.S_j^T R = (S_j p).R with S_j p from the context's creation.  This keeps the probe and
// the wait for it away from perturbations of no symmetry and from calls at the line
// (64 dots, 3 us at 381 modes, for 50 us).
unsigned orbit_candidates(const Ctx* c, int nc, int prec, const double* R, long ld) {
  if (!orbit_sized(c, prec)) return 0;
  const Orbit& o = c->orb;
  const int n = c->n, rows = std::min(o.nsym, kLook);
  const double full = estimate_us(c, (double)c->N * o.nsym, prec);
  unsigned mask = 0;
  for (int ch = 0; ch < nc; ++ch) {
    double Q[kLook][kLook];
    int r = 0;
    for (int j = 0; j < rows; ++j) {
      double* v = Q[r];
      for (int i = 0; i < kLook; ++i)
        v[i] = dot(o.look.data() + ((size_t)j * kLook + i) * n, R + ch * ld, n);
      const double whole = dot(v, v, kLook);
      for (int k = 0; k < r; ++k) {
        const double t = dot(v, Q[k], kLook);
        for (int m = 0; m < kLook; ++m) v[m] -= t * Q[k][m];
      }
      const double rest = dot(v, v, kLook);
      if (!(rest > 1e-12 * whole)) continue;   // (NaN: left to the probe)
      const double inv = 1.0 / std::sqrt(rest);
      for (int m = 0; m < kLook; ++m) v[m] *= inv;
      ++r;
    }
    if (r <= kOrbRank && full - estimate_us(c, (double)c->N * std::max(r, 1), prec) > kOrbWorthUs)
      mask |= 1u << ch;
  }
  return mask;
}

// the split images of the configurations; false = no room
static bool split_ready(Ctx* c, int prec) {
  Orbit& o = c->orb;
  if (!o.sub) {
    Ctx* s = new Ctx();
    s->device = c->device;
    s->stream = c->stream;
    s->n = c->n;
    s->np = c->np;
    s->N = c->N;
    s->n_syms = 1;
    s->M = c->N;
    s->Mp = o.Mp;
    s->n_eff = c->n_eff;
    s->row_lo = 0;
    s->row_hi = c->N;
    s->U = o.U;
    s->F = o.F;
    s->rho_img = o.rho;
    s->fy = c->fy;
    s->fpsi = c->fpsi;
    o.sub = s;
  }
  if (ensure_split(o.sub, prec) == 0) return true;
  (void)hipGetLastError();
  free_split(o.sub);
  return false;
}

// whether what the passes of a plan in this precision need is there (again)
bool orbit_ready(Ctx* c, int prec, hipStream_t s) {
  return c->orb.usable && ensure(c, s) && (prec == PREC_FP64 || split_ready(c, prec));
}

// Plan of nc chains (waits for the stream): the chains of `mask` that have a small orbit
// take the form (p.ok: some do), the others the general one.  x null: the averages of
// the padded inputs in c->R1, c->Y1.  Else a run from the packed vectors x (device):
// the relation holds for R and for each of the two pair sectors.
int orbit_plan(Ctx* c, int nc, unsigned mask, int prec, const double* x, hipStream_t s,
               OrbPlan& p) {
  Orbit& o = c->orb;
  p.ok = false;
  if (!ensure(c, s)) return 0;
  const int ncol = (c->n + 15) / 16, rows4 = o.rows * 4, ns = o.nsym;
  std::vector<int> piv;
  std::vector<double> C, Call;
  const int nm = x ? 2 * nc : nc;   // matrices
  if (x) {
    const long nn = (long)c->np * c->np;
    hipLaunchKernelGGL(orb_unpack, dim3((unsigned)((nn + 255) / 256), nm), dim3(256), 0, s, x, c->n,
                       c->np, (const int*)nullptr, 0, o.Yb, o.Rb);
  }
  hipLaunchKernelGGL(orb_probe, dim3(o.rows / 16, ncol, nm), dim3(256), 0, s, o.pu, o.pf,
                     x ? o.Yb : c->Y1, x ? o.Rb : c->R1, c->fy, c->fpsi, c->np, round_up(c->n, 16),
                     o.rows, o.ppart);
  hipLaunchKernelGGL(orb_probe_sum, dim3((rows4 + 255) / 256, nm), dim3(256), 0, s, o.ppart, ncol,
                     rows4, o.pout);
  TDS_CHECK_HIP(hipGetLastError());
  TDS_CHECK_HIP(hipStreamSynchronize(s));
  // chain by chain: rank and relation
  p.nc = nc;
  p.prec = prec;
  p.chains = p.others.n = p.rank = 0;
  std::vector<int> ranks(nc, 0);
  std::vector<std::vector<int>> pivots(nc);
  Call.assign((size_t)nc * ns * kOrbRank, 0.0);
  const double full = estimate_us(c, (double)c->N * ns, prec);
  for (int ch = 0; ch < nc; ++ch) {
    const double *m0 = o.pout + (size_t)(x ? 2 * ch : ch) * rows4, *m1 = m0 + rows4;
    // s3, s4 of the vector (R or R1), s1, s2 of each matrix (A and B, or Y1)
    std::vector<Dots> dots = {{m0, 2}, {m0, 3}, {m0, 0}, {m0, 1}};
    if (x) dots.insert(dots.end(), {{m1, 0}, {m1, 1}});
    const int r = mask >> ch & 1 ? relation(dots, ns, piv, C) : 0;
    if (r && full - estimate_us(c, (double)c->N * r, prec) > kOrbWorthUs) {
      ranks[ch] = r;
      pivots[ch] = piv;
      std::copy(C.begin(), C.end(), Call.begin() + (size_t)ch * ns * kOrbRank);
      p.rank = std::max(p.rank, r);
      ++p.chains;
    } else {
      p.others.at[p.others.n++] = ch;
    }
  }
  if (p.chains == 0) return 0;
  if (prec != PREC_FP64 && !split_ready(c, prec)) return 0;
  if (p.others.n && !p.general) {   // what the other chains leave, before it is spread
    const size_t count = kMaxChains * ((size_t)c->n + (size_t)c->n * c->n);
    if (hipMalloc((void**)&p.general, sizeof(double) * count) != hipSuccess) {
      (void)hipGetLastError();
      p.general = nullptr;
      return 0;
    }
  }
  // rounds of whole chains, at most kOrbPairs pairs each; of the clean-up, whose
  // matrices are the two sectors of each chain
  std::vector<int2> pairs, clean;
  std::vector<int4> mats, cmats;
  auto deal = [&](int sectors, std::vector<OrbPlan::Round>& rounds, std::vector<int2>& pr,
                  std::vector<int4>& mt) {
    rounds.clear();
    for (int ch = 0; ch < nc; ++ch) {
      if (!ranks[ch]) continue;
      if (rounds.empty() || rounds.back().count + sectors * ranks[ch] > kOrbPairs)
        rounds.push_back({(int)mt.size(), 0, (int)pr.size(), 0});
      OrbPlan::Round& rd = rounds.back();
      for (int sec = 0; sec < sectors; ++sec) {
        const int m = sectors * ch + sec;
        mt.push_back(int4{rd.count, ranks[ch], ch, m});
        for (int q : pivots[ch]) pr.push_back(int2{m, q});
        rd.count += ranks[ch];
        ++rd.mats;
      }
    }
  };
  deal(1, p.rounds, pairs, mats);
  deal(2, p.clean_rounds, clean, cmats);
  const size_t b0 = sizeof(int4) * (mats.size() + cmats.size()),
               b1 = sizeof(int2) * (pairs.size() + clean.size()), b2 = sizeof(double) * Call.size();
  const size_t need = b0 + b1 + b2;
  if (p.cap < need) {
    if (p.dev) (void)hipFree(p.dev);
    p.dev = nullptr;
    p.cap = 0;
    const size_t most = sizeof(int4) * 3 * kMaxChains + sizeof(int2) * 3 * kMaxChains * kOrbRank +
                        sizeof(double) * kMaxChains * (size_t)ns * kOrbRank;
    TDS_CHECK_HIP(hipMalloc(&p.dev, std::max(most, need)));
    p.cap = std::max(most, need);
  }
  p.host.resize(need);
  char* h = p.host.data();
  std::copy(mats.begin(), mats.end(), reinterpret_cast<int4*>(h));
  std::copy(cmats.begin(), cmats.end(), reinterpret_cast<int4*>(h) + mats.size());
  std::copy(Call.begin(), Call.end(), reinterpret_cast<double*>(h + b0));
  std::copy(pairs.begin(), pairs.end(), reinterpret_cast<int2*>(h + b0 + b2));
  std::copy(clean.begin(), clean.end(), reinterpret_cast<int2*>(h + b0 + b2) + pairs.size());
  TDS_CHECK_HIP(hipMemcpyAsync(p.dev, h, need, hipMemcpyHostToDevice, s));
  char* d = static_cast<char*>(p.dev);
  p.mats = reinterpret_cast<int4*>(d);
  p.cmats = p.mats + mats.size();
  p.C = reinterpret_cast<double*>(d + b0);
  p.pairs = reinterpret_cast<int2*>(d + b0 + b2);
  p.clean = p.pairs + pairs.size();
  p.ok = true;
  return 0;
}

static OrbPanels panels(const Ctx* c) {
  const Orbit& o = c->orb;
  return OrbPanels{o.start, o.npanel, o.nsym, o.S, o.ST};
}

// the perturbed averages of the plan's chains with an orbit (inputs in c->R1, c->Y1)
static int run_orbits(Ctx* c, const OrbPlan& p, int apply_d4, double* f_dev, double* d2v_dev,
                      hipStream_t s) {
  Orbit& o = c->orb;
  const int n = c->n, np = c->np, ks = orb_ksplit(c);
  const OrbPanels pn = panels(c);
  for (const OrbPlan::Round& rd : p.rounds) {
    const int P = rd.count;
    hipLaunchKernelGGL(orb_in, dim3(o.npanel * o.npanel, P), dim3(256), 0, s, pn, p.pairs + rd.pair,
                       c->Y1, c->R1, np, (const int*)nullptr, 0, o.Y1, o.R1);
    if (p.prec != PREC_FP64) {
      // the split kernels on the configurations, in groups of 6 pairs (they take three
      // at a time).  128 atoms x 20000, 9 pairs: 0.40 ms for 2.0 in FP64; against FP64
      // results the error is below that of the split average over the images (d2v
      // 1e-7 for 7e-7 in FP16x2, 1.3e-6 for 1.5e-6 in BF16x2 at 12000 configurations)
      for (int p0 = 0; p0 < P; p0 += 6) {
        o.sub->R1 = o.R1 + (long)p0 * np;
        o.sub->Y1 = o.Y1 + (long)p0 * np * np;
        o.sub->f_out = o.f + (long)p0 * np;
        o.sub->d2v_out = o.z + (long)p0 * np * np;
        const int rc = launch_pa_split(o.sub, std::min(6, P - p0), apply_d4, p.prec, s, nullptr);
        if (rc) return rc;
      }
    } else {
      const F64Rows rows{o.U, o.F, o.rho, o.Mp};
      launch_weights_f64(rows, n, np, P, o.Y1, o.R1, c->fy, c->fpsi, apply_d4, 0, (c->N + 63) / 64,
                         0, c->N, o.coef, s);
      // as many pairs at once as the context's partial sums have room for (it holds
      // kMaxChains ksplit of them, ksplit at least 8, ks at most 24)
      const long ke = round_up_l(c->N, 8), rps = round_up_l((ke + ks - 1) / ks, 8);
      const int most = kMaxChains * c->ksplit / ks;
      for (int p0 = 0; p0 < P; p0 += most) {
        const int g = std::min(most, P - p0);
        launch_outer_f64(rows, n, np, g, o.coef + (long)p0 * o.Mp * 4, c->fy, ks, 0, ke, rps, 0,
                         c->zpart, c->fpart, s);
        launch_reduce_f64(n, np, g, ks, c->zpart, c->fpart, o.z + (long)p0 * np * np,
                          o.f + (long)p0 * np, 1.0 / c->n_eff, s);
      }
    }
    const auto out = p.rank <= 3 ? orb_out<true, 3> : orb_out<true, kOrbRank>;
    hipLaunchKernelGGL(out, dim3(o.npanel * (o.npanel + 3) / 2, rd.mats), dim3(512), 0, s, pn,
                       p.mats + rd.mat, p.C, o.z, o.f, c->fy, n, np, 1.0 / o.nsym,
                       1.0 / (c->n_eff * o.nsym), (const int*)nullptr, 0, (const int*)nullptr,
                       f_dev, d2v_dev);
    TDS_CHECK_HIP(hipGetLastError());
  }
  return 0;
}

// dst[k] = src[at[k]] (GATHER; in place too: at[k] >= k, and an element is moved by one
// thread) or dst[at[k]] = src[k], `per` doubles per chain
template <bool GATHER>
__global__ void orb_move(const double* src, double* dst, OrbPlan::List l, long per) {
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= per) return;
  for (int k = 0; k < l.n; ++k)
    dst[(GATHER ? k : l.at[k]) * per + e] = src[(GATHER ? l.at[k] : k) * per + e];
}

// the perturbed averages of the plan's chains (inputs in c->R1, c->Y1): those with an
// orbit, then the others, which c->R1, c->Y1 are packed for
int run_pa_orbit(Ctx* c, const OrbPlan& p, int apply_d4, double* f_dev, double* d2v_dev,
                 hipStream_t s) {
  int rc = run_orbits(c, p, apply_d4, f_dev, d2v_dev, s);
  if (rc || p.others.n == 0) return rc;
  const long n = c->n, np = c->np;
  auto blocks = [](long count) { return dim3((unsigned)((count + 255) / 256)); };
  hipLaunchKernelGGL(orb_move<true>, blocks(np), dim3(256), 0, s, c->R1, c->R1, p.others, np);
  hipLaunchKernelGGL(orb_move<true>, blocks(np * np), dim3(256), 0, s, c->Y1, c->Y1, p.others,
                     np * np);
  double *f = p.general, *d = p.general + kMaxChains * n;
  rc = run_pa(c, p.others.n, apply_d4, p.prec, f, d, s);
  if (rc) return rc;
  hipLaunchKernelGGL(orb_move<false>, blocks(n), dim3(256), 0, s, f, f_dev, p.others, n);
  hipLaunchKernelGGL(orb_move<false>, blocks(n * n), dim3(256), 0, s, d, d2v_dev, p.others, n * n);
  TDS_CHECK_HIP(hipGetLastError());
  return 0;
}

// project the packed vectors x of the plan's chains on their sector, on every
// kOrbClean-th step (kk: the chains' common step counter on the device)
int orbit_clean(Ctx* c, const OrbPlan& p, double* x, const int* kk, const int* active,
                hipStream_t s) {
  Orbit& o = c->orb;
  const int n = c->n, np = c->np;
  const long nn = (long)np * np;
  const OrbPanels pn = panels(c);
  hipLaunchKernelGGL(orb_unpack, dim3((unsigned)((nn + 255) / 256), 2 * p.nc), dim3(256), 0, s, x,
                     n, np, kk, kOrbClean, o.Yb, o.Rb);
  for (const OrbPlan::Round& r : p.clean_rounds) {
    hipLaunchKernelGGL(orb_in, dim3(o.npanel * o.npanel, r.count), dim3(256), 0, s, pn,
                       p.clean + r.pair, o.Yb, o.Rb, np, kk, kOrbClean, o.Y1, o.R1);
    const auto out = p.rank <= 3 ? orb_out<false, 3> : orb_out<false, kOrbRank>;
    hipLaunchKernelGGL(out, dim3(o.npanel * (o.npanel + 3) / 2, r.mats), dim3(512), 0, s, pn,
                       p.cmats + r.mat, p.C, o.Y1, o.R1, c->fy, n, np, 1.0 / o.nsym, 1.0 / o.nsym,
                       kk, kOrbClean, active, (double*)nullptr, x);
  }
  TDS_CHECK_HIP(hipGetLastError());
  return 0;
}

}  // namespace tdscha
