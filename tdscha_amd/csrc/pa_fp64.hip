// FP64 ensemble-averaged D3/D4 application on MFMA (v_mfma_f64_4x4x4_4b_f64).
//
// The per-image algebra of CModules/LanczosFunctions.c:2082-2754 is regrouped
// into three passes over the device-resident symmetric image ensemble
// (rows = images b = i*N_sym + j, columns = modes):
//
//   weights_f64   V = U . Y1 (tiled GEMM, K = modes) with a fused row-dot
//                 epilogue: s1 = u.Y1.u, s2 = u.Y1.g, s3 = a.R1, s4 = f.R1
//                 -> per image c1, c2 (d2v weights) and alpha, beta (force
//                 weights).
//   outer_f64     Z = U^T B with B = c1 F + (c2/2) fY U  (split-K GEMM over
//                 the images, LDS-staged image tiles), and on the diagonal
//                 tiles the force average sum alpha F + beta fY U.
//   reduce        d2v = fY Z + (fY Z)^T, f = sum of partials, scaled by
//                 1/(N_eff N_sym); fixed summation order (deterministic).
//
// Both GEMMs are bound by the FP64 matrix rate.  The 4x4x4 instruction (four
// independent 4x4x4 products) sustains 72 TF/s with constant operands on
// MI355X, at one wave per SIMD already (70-72 with both operands read from LDS
// each step); the 16x16x4 one 35 TF/s at one wave per SIMD and 49 TF/s at eight
// in the same loop.  Measured at 381 modes, 960,000 images, 3 chains: weights
// 14.0 ms, outer 14.1 ms (60 TF/s each; with the 16x16x4 instruction and
// register prefetch 18.6 and 17.4 ms), at 159 modes and 240,000 images 0.88 and
// 0.82 ms (2.35 and 1.94 ms with 128-column tiles).
//
// Operand layout of the 4x4x4 MFMA (one double per lane, block q = lane / 4 % 4):
//   A[i][k]: i = lane % 4, k = lane / 16;  B[k][j]: j = lane % 4, k = lane / 16
//   D[i][j]: j = lane % 4, i = lane / 16
// The four blocks of A hold 16 rows (row 4 q + i of a group: lane % 16).  B holds
// either the same 4 columns in all four blocks (its lanes read one LDS address:
// a broadcast), or 16 columns, rotated by r blocks (a DPP row rotation) in four
// MFMAs so that block q meets the columns of block q - r.  FP64 vector
// instructions take matrix time here, so a B that is built (the outer product)
// is built once per value and rotated: built four-fold for the broadcast form
// the outer product ran at 44 TF/s instead of 57.
#include <algorithm>
#include <type_traits>

#include "common.hpp"

namespace tdscha {

// ---------------------------------------------------------------------------
// image expansion: U[b, m] = sum_k S_{blk(m)}[j, pos(m), k] X[i, modes_blk[k]]
// ---------------------------------------------------------------------------
__global__ void expand_images(const double* __restrict__ X, const double* __restrict__ Y,
                              const double* __restrict__ rho, const int* __restrict__ mode_block,
                              const int* __restrict__ mode_pos, const int* __restrict__ block_dim,
                              const int* __restrict__ block_moff, const long* __restrict__ block_soff,
                              const int* __restrict__ block_modes, const double* __restrict__ syms,
                              int n, int np, int n_syms, long M, double* __restrict__ U,
                              double* __restrict__ F, double* __restrict__ rho_img) {
  const long row = blockIdx.x;
  const int m = threadIdx.x + blockIdx.y * blockDim.x;
  if (m >= np) return;
  double su = 0.0, sf = 0.0;
  if (row < M && m < n) {
    const long i = row / n_syms;
    const int j = (int)(row % n_syms);
    const int b = mode_block[m];
    const int d = block_dim[b];
    const double* S = syms + block_soff[b] + ((long)j * d + mode_pos[m]) * d;
    const int* modes = block_modes + block_moff[b];
    const double* x = X + i * n;
    const double* y = Y + i * n;
    for (int k = 0; k < d; ++k) {
      const double s = S[k];
      su += s * x[modes[k]];
      sf += s * y[modes[k]];
    }
  }
  U[row * np + m] = su;
  F[row * np + m] = sf;
  if (m == 0) rho_img[row] = (row < M) ? rho[row / n_syms] : 0.0;
}

// ---------------------------------------------------------------------------
// Work-group order of both GEMMs: the hardware deals work-groups to the 8
// XCDs in turn (id % 8), so the chains of one tile get ids 8 apart and run on
// one XCD at about the same time, sharing its L2 for the image rows.
//
// Tiles: n modes are covered by ceil(n / 128) equal column tiles of 16 CB
// columns (CB = 1 .. 8), so that little is computed for padding (159 modes: two
// tiles of 80 columns, where whole 128-column tiles would do 1.6 times the
// work of a GEMM side and 2.6 times that of the outer product).
// ---------------------------------------------------------------------------
// CB consecutive doubles from p[o] on (16-byte pieces where CB is even).  The
// LDS reads of both kernels form each address with one index: the compiler
// knows which LDS array a read may touch only through short pointer
// chains, and otherwise waits for every copy in flight.
template <int CB>
static __device__ __forceinline__ void read_run(const double* p, long o, double (&v)[CB]) {
  if constexpr (CB % 2 == 0) {
#pragma unroll
    for (int c = 0; c < CB; c += 2) {
      const double2 t = *reinterpret_cast<const double2*>(p + (o + c));
      v[c] = t.x;
      v[c + 1] = t.y;
    }
  } else {
#pragma unroll
    for (int c = 0; c < CB; ++c) v[c] = p[o + c];
  }
}

// LDS addresses of the copies are formed in the LDS address space: a generic
// pointer at a constant offset would count as any array
typedef __attribute__((address_space(3))) double* lds_d;
static __device__ __forceinline__ void copy16(const double* g, lds_d l) {
  __builtin_amdgcn_global_load_lds((gbl_ptr_t)g, (lds_ptr_t)l, 16, 0, 0);
}

// acc[i][r] += A_i x B, 16 rows per i: block q of lane's column group q - r
template <int NA>
static __device__ __forceinline__ void mfma_rot(const double (&a)[NA], double b,
                                                double (&acc)[NA][4]) {
  const double b1 = rot4<1>(b), b2 = rot4<2>(b), b3 = rot4<3>(b);
#pragma unroll
  for (int i = 0; i < NA; ++i) acc[i][0] = mfma4(a[i], b, acc[i][0]);
#pragma unroll
  for (int i = 0; i < NA; ++i) acc[i][1] = mfma4(a[i], b1, acc[i][1]);
#pragma unroll
  for (int i = 0; i < NA; ++i) acc[i][2] = mfma4(a[i], b2, acc[i][2]);
#pragma unroll
  for (int i = 0; i < NA; ++i) acc[i][3] = mfma4(a[i], b3, acc[i][3]);
}

// Both kernels run 4 waves per work-group, two work-groups per CU (3 of the outer
// product up to CB = 5), and stream their K chunks through a ring of 3 LDS slots
// (separate arrays, slot fixed at compile time by a 3-fold unroll) filled by
// direct-to-LDS copies issued two chunks ahead; with the next chunk held in
// registers (one chunk ahead) the latency of the loads showed (50 and 34 TF/s).

// weights: one work-group = 64 image rows, column tiles of 16 CB one after the
// other (wave w: columns 4 CB w .. of the tile for all 64 rows), K in chunks of
// 16 modes.  A lane reads two successive modes of a row at once (16 bytes): within 8 modes the first MFMA takes the even ones and the
// second the odd ones, in A and B alike.  The 16-byte pieces of a row are
// stored XOR-ed with the row (the copies permute their source), so that the 8
// rows a read serves per cycle sit in 8 distinct bank groups.  The first chunks
// of the next column tile are requested before a tile's epilogue.
constexpr int WA_KC = 16;

template <int CB>
__global__ __launch_bounds__(256, 2) void weights_f64(
    const double* __restrict__ U, const double* __restrict__ F,
    const double* __restrict__ Y1all, const double* __restrict__ R1all,
    const double* __restrict__ fy, const double* __restrict__ fpsi,
    const double* __restrict__ rho_img, int np, int nk, int ntile, long Mp, int apply_d4,
    long tile0, long tile1, long row_lo, long row_hi, int nc, double* __restrict__ coef_all) {
  constexpr int W = 16 * CB;
  constexpr int kCY = (2 * CB + 3) / 4;   // copies of Y1 per wave and chunk
  constexpr int kLoads = 2 + kCY;
  const int xcd = blockIdx.x & 7;
  const int jj = blockIdx.x >> 3;
  const int chain = jj % nc;
  const long tile = tile0 + (long)(jj / nc) * 8 + xcd;
  if (tile >= tile1) return;   // whole work-group, before any barrier
  const double* Y1 = Y1all + (long)chain * np * np;
  const double* R1 = R1all + (long)chain * np;
  double* coef = coef_all + (long)chain * Mp * 4;
  const long r0 = tile * 64;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4, lq = lane & 3;
  const int drow = (lane & 12) + lg;   // row of a 16-row group this lane's results belong to

  constexpr int kU = 64 * WA_KC, kSlot = kU + WA_KC * W;
  __shared__ __align__(16) double s0[kSlot];
  __shared__ __align__(16) double s1[kSlot];
  __shared__ __align__(16) double s2[kSlot];
  static_assert(1024 <= kSlot, "the row-dot partials fit a slot");
  double(*const red)[64][4] = reinterpret_cast<double(*)[64][4]>(s2);   // [4][64][4]

  // copy chunk kc of column tile c0, 64 pieces of 16 bytes per copy, dealt to
  // the waves (every wave and lane takes part in each, so that the number of
  // copies in flight is known; those beyond the last repeat it): 8 copies of 8
  // U rows (128 bytes of a row each), 2 CB copies of Y1
  const double* pu = U + (r0 + 16 * wave + (lane >> 3)) * np + 2 * ((lane & 7) ^ (lane >> 3));
  int yoff[kCY];
#pragma unroll
  for (int e = 0; e < kCY; ++e) {
    const int p = 64 * min(wave + 4 * e, 2 * CB - 1) + lane;
    yoff[e] = p / (W / 2) * np + 2 * (p % (W / 2));
  }
  auto issue = [&](lds_d slot, int c0, int kc) {
    const int k0 = kc * WA_KC;
    copy16(pu + k0, slot + 16 * wave * WA_KC);
    copy16(pu + 8L * np + k0, slot + (16 * wave + 8) * WA_KC);
    const double* py = Y1 + (long)k0 * np + c0;
#pragma unroll
    for (int e = 0; e < kCY; ++e)
      copy16(py + yoff[e], slot + kU + 128 * min(wave + 4 * e, 2 * CB - 1));
  };

  double acc[4][CB];
  auto compute = [&](const double* cur) {
#pragma unroll
    for (int k8 = 0; k8 < WA_KC; k8 += 8) {
      double2 a[4];
#pragma unroll
      for (int rb = 0; rb < 4; ++rb)
        a[rb] = *reinterpret_cast<const double2*>(
            cur + ((16 * rb + lr) * WA_KC + 2 * ((k8 / 2 + lg) ^ (lr & 7))));
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        double b[CB];
        read_run<CB>(cur, kU + (k8 + 2 * lg + t) * W + 4 * CB * wave + CB * lq, b);
#pragma unroll
        for (int rb = 0; rb < 4; ++rb)
#pragma unroll
          for (int cb = 0; cb < CB; ++cb)
            acc[rb][cb] = mfma4(t ? a[rb].y : a[rb].x, b[cb], acc[rb][cb]);
      }
    }
  };
  // chunk kc: its copies (all but the youngest kLoads) have landed and every
  // wave is done with chunk kc - 1, whose slot takes chunk kc + 2
  auto step = [&](const double* cur, double* nxt, int c0, int kc) {
    TDS_WAIT_VMCNT(kLoads);
    lds_barrier();
    issue((lds_d)nxt, c0, kc + 2);
    compute(cur);
  };
  // the last two chunks
  auto tail = [&](const double* a, const double* b) {
    TDS_WAIT_VMCNT(kLoads);
    lds_barrier();
    compute(a);
    TDS_WAIT_VMCNT(0);
    lds_barrier();
    compute(b);
  };

  // tid = 4 row + quantity: running row-dot sums over the column tiles
  const int urow = tid >> 2;
  double rowsum = 0.0;
  const int nkc = nk / WA_KC;
  issue((lds_d)s0, 0, 0);
  issue((lds_d)s1, 0, 1);
  for (int c0 = 0; c0 < ntile * W; c0 += W) {
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < CB; ++b) acc[a][b] = 0.0;
    int kc = 0;
    for (; kc + 5 <= nkc; kc += 3) {
      step(s0, s2, c0, kc);
      step(s1, s0, c0, kc + 1);
      step(s2, s1, c0, kc + 2);
    }
    if (nkc - kc == 2) {
      tail(s0, s1);
    } else if (nkc - kc == 3) {
      step(s0, s2, c0, kc);
      tail(s1, s2);
    } else {
      step(s0, s2, c0, kc);
      step(s1, s0, c0, kc + 1);
      tail(s2, s0);
    }
    lds_barrier();   // every slot is free
    if (c0 + W < ntile * W) {
      issue((lds_d)s0, c0 + W, 0);
      issue((lds_d)s1, c0 + W, 1);
    }

    // fused epilogue: row dots over this lane's CB columns, then over the four
    // lanes of the row
    const int col = c0 + 4 * CB * wave + CB * lq;
    double fyr[CB], fpc[CB], r1c[CB];
    read_run<CB>(fy, col, fyr);
    read_run<CB>(fpsi, col, fpc);
    read_run<CB>(R1, col, r1c);
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) fyr[cb] *= r1c[cb];
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) {
      const long o = (r0 + 16 * rb + drow) * np + col;
      double u[CB], f[CB];
      read_run<CB>(U, o, u);
      read_run<CB>(F, o, f);
      double p[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) {
        p[0] += acc[rb][cb] * u[cb];
        p[1] += acc[rb][cb] * (f[cb] * fpc[cb]);
        p[2] += u[cb] * fyr[cb];
        p[3] += f[cb] * r1c[cb];
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        p[q] += __shfl_xor(p[q], 1);
        p[q] += __shfl_xor(p[q], 2);
      }
      red[wave][16 * rb + drow][lq] = lq < 2 ? (lq ? p[1] : p[0]) : (lq == 2 ? p[2] : p[3]);
    }
    lds_barrier();
    rowsum += (red[0][urow][lq] + red[1][urow][lq]) + (red[2][urow][lq] + red[3][urow][lq]);
    // (slot 2 is filled again after the next tile's first barrier)
  }
  // the row's four lanes share its sums; lane q writes coefficient q
  const int base = lane & 60;
  const double s_1 = __shfl(rowsum, base);       // u.Y1.u
  const double s_2 = __shfl(rowsum, base + 1);   // u.Y1.g  (Y1 symmetrised on upload)
  const double s_3 = __shfl(rowsum, base + 2);   // a.R1
  const double s_4 = __shfl(rowsum, base + 3);   // f.R1
  const long row = r0 + urow;
  // images outside [row_lo, row_hi) carry no weight (image-range calls)
  const double rho = (row >= row_lo && row < row_hi) ? rho_img[row] : 0.0;
  const double c1 = rho * (-s_3 / 3.0 + apply_d4 * s_1 / 8.0);
  const double c2 = rho * (-s_4 / 3.0 + apply_d4 * s_2 / 4.0);
  coef[row * 4 + lq] = lq < 2 ? (lq ? c2 : c1) : (lq == 2 ? -rho * s_1 / 6.0 : -rho * s_2 / 3.0);
}

// ---------------------------------------------------------------------------
// outer: split-K Z[mu, nu] = sum_b U[b, mu] B[b, nu] over a range of images,
// T x T tiles (T = 16 CB), wave w on all T rows and the columns 4 CB w .., chunks
// of 8 images.  A slot holds the images' U of the mu columns, F and (off the
// diagonal) U of the nu columns and the coefficients; a wave builds the B values
// of its own columns in registers as it reads them, 16 columns at a time in the
// rotated form and the CB % 4 groups of 4 that remain in the broadcast form.
// ---------------------------------------------------------------------------
constexpr int WB_KC = 8;

template <int CB>
__global__ __launch_bounds__(256, CB > 5 ? 2 : 3) void outer_f64(
    const double* __restrict__ U, const double* __restrict__ F,
    const double* __restrict__ coef_all, const double* __restrict__ fy, int np, long Mp,
    int ksplit, int ntile, long kbase, long kend, long rows_per_split, int accumulate, int nc,
    double* __restrict__ zpart_all, double* __restrict__ fpart_all) {
  constexpr int T = 16 * CB;
  constexpr int NF = CB / 4, NQ = CB % 4;   // rotated 16-column and broadcast 4-column operands
  const int xcd = blockIdx.x & 7;
  const int jj = blockIdx.x >> 3;
  const int chain = jj % nc;
  const int rest = jj / nc;
  const int t2 = ntile * ntile;
  const int tile = rest % t2;
  const int ks = xcd + 8 * (rest / t2);
  const int tm = tile / ntile, tn = tile % ntile;
  const double* coef = coef_all + (long)chain * Mp * 4;
  const int zl = ntile * T;   // partials hold the tiles only
  double* zpart = zpart_all + ((long)chain * ksplit + ks) * zl * zl;
  double* fpart = fpart_all + ((long)chain * ksplit + ks) * np;
  const int mu0 = tm * T, nu0 = tn * T;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int lr = lane & 15, lg = lane >> 4, lq = lane & 3, lb = (lane >> 2) & 3;

  constexpr int kM = WB_KC * T, kSlot = 3 * kM + 128;
  __shared__ __align__(16) double s0[kSlot];
  __shared__ __align__(16) double s1[kSlot];
  __shared__ __align__(16) double s2[kSlot];

  double acc[NF > 0 ? NF : 1][CB][4], aq[NQ > 0 ? NQ : 1][CB];
#pragma unroll
  for (int i = 0; i < CB; ++i) {
#pragma unroll
    for (int g = 0; g < NF; ++g) acc[g][i][0] = acc[g][i][1] = acc[g][i][2] = acc[g][i][3] = 0.0;
#pragma unroll
    for (int g = 0; g < NQ; ++g) aq[g][i] = 0.0;
  }

  const long kb = kbase + (long)ks * rows_per_split;
  const long ke = kb + rows_per_split < kend ? kb + rows_per_split : kend;
  const int nch = ke > kb ? (int)((ke - kb) / WB_KC) : 0;
  // this lane's B columns: 16 g + lr of the rotated operands, 4 g + lq of the others
  const int wcol = 4 * CB * wave + lr, qcol = 4 * CB * wave + 16 * NF + lq;
  double hf[NF > 0 ? NF : 1], hq[NQ > 0 ? NQ : 1], fa[NF + 1], fb[NF + 1];
#pragma unroll
  for (int g = 0; g < NF; ++g) hf[g] = 0.5 * fy[nu0 + wcol + 16 * g];
#pragma unroll
  for (int g = 0; g < NQ; ++g) hq[g] = 0.5 * fy[nu0 + qcol + 4 * g];
#pragma unroll
  for (int g = 0; g <= NF; ++g) fa[g] = fb[g] = 0.0;   // sums of alpha f, beta u (diagonal tiles)
  // column of the tile whose f sum a lane holds in fa[NF]: 16 NF + lr of the wave's 4 CB
  const int lcol = 4 * CB * wave + 16 * NF + (lr < 4 * NQ ? lr : 0);

  auto run = [&](auto is_diag) {
    constexpr bool DIAG = decltype(is_diag)::value;
    constexpr int kC = (CB + 3) / 4;                  // copies per matrix, wave and chunk
    constexpr int kLoads = kC * (DIAG ? 2 : 3) + 1;
    constexpr int oUn = DIAG ? 0 : 2 * kM;            // U of the nu columns
    // 64 pieces of 16 bytes per copy, CB copies per matrix, dealt to the waves
    // (every wave and lane takes part in each, so that the number of copies in
    // flight is known; those beyond the last repeat it)
    int off[kC];
#pragma unroll
    for (int e = 0; e < kC; ++e) {
      const int p = 64 * min(wave + 4 * e, CB - 1) + lane;
      off[e] = p / (T / 2) * np + 2 * (p % (T / 2));
    }
    const int coff = 2 * (lane & 15);   // 8 images of 4 coefficients, four times over
    auto issue = [&](lds_d slot, int ch) {
      const long row = kb + (long)ch * WB_KC;
      const double* pu = U + row * np;
      const double* pf = F + row * np + nu0;
#pragma unroll
      for (int e = 0; e < kC; ++e) {
        const lds_d d = slot + 128 * min(wave + 4 * e, CB - 1);
        copy16(pu + mu0 + off[e], d);
        copy16(pf + off[e], d + kM);
        if (!DIAG) copy16(pu + nu0 + off[e], d + 2 * kM);
      }
      copy16(coef + row * 4 + coff, slot + 3 * kM);
    };
    // chunk ch: its copies (all but the youngest kLoads) have landed and every
    // wave is done with chunk ch - 1, whose slot takes chunk ch + 2 (the last
    // one again beyond the end)
    auto step = [&](const double* cur, double* nxt, int ch) {
      TDS_WAIT_VMCNT(kLoads);
      lds_barrier();
      issue((lds_d)nxt, min(ch + 2, nch - 1));
#pragma unroll
      for (int k4 = 0; k4 < WB_KC; k4 += 4) {
        const int k = k4 + lg;
        double a[CB];
        // rows 16 i + lane % 16, or (CB even) rows 32 i + 2 (lane % 16) + 0, 1
        if constexpr (CB % 2 == 0) {
#pragma unroll
          for (int i = 0; i < CB; i += 2) {
            const double2 t = *reinterpret_cast<const double2*>(cur + (k * T + 16 * i + 2 * lr));
            a[i] = t.x;
            a[i + 1] = t.y;
          }
        } else {
#pragma unroll
          for (int i = 0; i < CB; ++i) a[i] = cur[k * T + 16 * i + lr];
        }
        const int of = kM + k * T, on = oUn + k * T;
        const double2 c12 = *reinterpret_cast<const double2*>(cur + (3 * kM + 4 * k));
        double2 ab;
        if constexpr (DIAG) ab = *reinterpret_cast<const double2*>(cur + (3 * kM + 4 * k + 2));
#pragma unroll
        for (int g = 0; g < NF; ++g) {
          const double f = cur[of + wcol + 16 * g], u = cur[on + wcol + 16 * g];
          mfma_rot<CB>(a, c12.x * f + c12.y * (hf[g] * u), acc[g]);
          if constexpr (DIAG) {
            fa[g] += ab.x * f;
            fb[g] += ab.y * u;
          }
        }
#pragma unroll
        for (int g = 0; g < NQ; ++g) {
          const double b =
              c12.x * cur[of + qcol + 4 * g] + c12.y * (hq[g] * cur[on + qcol + 4 * g]);
#pragma unroll
          for (int i = 0; i < CB; ++i) aq[g][i] = mfma4(a[i], b, aq[g][i]);
        }
        if constexpr (DIAG && NQ > 0) {
          fa[NF] += ab.x * cur[of + lcol];
          fb[NF] += ab.y * cur[on + lcol];
        }
      }
    };
    issue((lds_d)s0, 0);
    issue((lds_d)s1, min(1, nch - 1));
    for (int ch = 0;;) {
      step(s0, s2, ch);
      if (++ch == nch) break;
      step(s1, s0, ch);
      if (++ch == nch) break;
      step(s2, s1, ch);
      if (++ch == nch) break;
    }
    TDS_WAIT_VMCNT(0);   // the copies past the end land before the LDS is released
  };
  if (nch > 0) {
    if (tm == tn)
      run(std::true_type{});
    else
      run(std::false_type{});
  }

  // write the partial tile; accumulate: add to the partial of earlier image
  // chunks (each element has one writer, chunks run in order)
  const int drow = 4 * lb + lg;
#pragma unroll
  for (int i = 0; i < CB; ++i) {
    const int mu = mu0 + (CB % 2 ? 16 * i + drow : 16 * (i & ~1) + 2 * drow + (i & 1));
    double* z = zpart + (long)mu * zl + nu0 + 4 * CB * wave + lq;
#pragma unroll
    for (int g = 0; g < NF; ++g)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        double* p = z + 16 * g + 4 * ((lb - r) & 3);
        *p = (accumulate ? *p : 0.0) + acc[g][i][r];
      }
#pragma unroll
    for (int g = 0; g < NQ; ++g) {
      double* p = z + 16 * NF + 4 * g;
      *p = (accumulate ? *p : 0.0) + aq[g][i];
    }
  }
  if (tm == tn) {
#pragma unroll
    for (int g = 0; g < NF + (NQ > 0); ++g) {
      const int c = g < NF ? wcol + 16 * g : lcol;
      double v = fa[g] + fy[nu0 + c] * fb[g];
      v += __shfl_xor(v, 16);
      v += __shfl_xor(v, 32);
      if (lg == 0 && (g < NF || lr < 4 * NQ)) {
        double* p = fpart + nu0 + c;
        *p = (accumulate ? *p : 0.0) + v;
      }
    }
  }
}

// sum the K-split partials in a fixed order, rows and columns below n: 64
// elements per work-group, the partials in 4 or 16 slices of 8 loads in flight each,
// combined in LDS; grid (ceil(n / 64), n + 1, chains), the last row the f sums
template <int SL>
__global__ __launch_bounds__(64 * SL) void reduce_ksplit(const double* __restrict__ zpart_all,
                                                         const double* __restrict__ fpart_all,
                                                         int n, int np, int zl, int ksplit,
                                                         double* __restrict__ zsum_all,
                                                         double* __restrict__ f_all, double norm) {
  const int chain = blockIdx.z, row = blockIdx.y;
  const int t = threadIdx.x & 63, c = blockIdx.x * 64 + t, sl = threadIdx.x >> 6;
  const bool isf = row == n;
  const long stride = isf ? np : (long)zl * zl;
  const double* p = isf ? fpart_all + (long)chain * ksplit * np + c
                        : zpart_all + (long)chain * ksplit * stride + (long)row * zl + c;
  const int per = (ksplit + SL - 1) / SL;
  const int lo = sl * per, hi = lo + per < ksplit ? lo + per : ksplit;
  double s = 0.0;
  if (c < n) {
    int k = lo;
    for (; k + 8 <= hi; k += 8) {
      double v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = p[(k + j) * stride];
#pragma unroll
      for (int j = 0; j < 8; ++j) s += v[j];
    }
    for (; k < hi; ++k) s += p[k * stride];
  }
  __shared__ double red[SL][64];
  red[sl][t] = s;
  __syncthreads();
  if (sl == 0 && c < n) {
    double v = 0.0;
#pragma unroll
    for (int q = 0; q < SL; q += 4)
      v += (red[q][t] + red[q + 1][t]) + (red[q + 2][t] + red[q + 3][t]);
    if (isf)
      f_all[(long)chain * np + c] = v * norm;
    else
      zsum_all[(long)chain * np * np + (long)row * np + c] = v;
  }
}

// column tiles of n modes: ceil(n / 128) of them, 16 CB columns each
F64Tiles f64_tiles(int n) {
  const int t = (n + kTile - 1) / kTile;
  return {t, ((n + t - 1) / t + 15) / 16};
}

template <typename Fn>
static void with_cb(int cb, Fn fn) {
  switch (cb) {
    case 1: fn(std::integral_constant<int, 1>{}); break;
    case 2: fn(std::integral_constant<int, 2>{}); break;
    case 3: fn(std::integral_constant<int, 3>{}); break;
    case 4: fn(std::integral_constant<int, 4>{}); break;
    case 5: fn(std::integral_constant<int, 5>{}); break;
    case 6: fn(std::integral_constant<int, 6>{}); break;
    case 7: fn(std::integral_constant<int, 7>{}); break;
    default: fn(std::integral_constant<int, 8>{}); break;
  }
}

// rows [64 tile0, 64 tile1) of U, F; coefficients of images outside
// [row_lo, row_hi) are zero
void launch_weights_f64(const F64Rows& r, int n, int np, int nc, const double* Y1,
                        const double* R1, const double* fy, const double* fpsi, int apply_d4,
                        long tile0, long tile1, long row_lo, long row_hi, double* coef,
                        hipStream_t s) {
  const F64Tiles t = f64_tiles(n);
  const int nk = std::max(2 * WA_KC, round_up(n, WA_KC));   // the ring starts with two chunks
  // tiles dealt 8 at a time (one per XCD), every chain of a tile on its XCD
  const long g = round_up_l(tile1 - tile0, 8) * nc;
  with_cb(t.cb, [&](auto cb) {
    hipLaunchKernelGGL(weights_f64<decltype(cb)::value>, dim3((unsigned)g), dim3(256), 0, s, r.U,
                       r.F, Y1, R1, fy, fpsi, r.rho, np, nk, t.ntile, r.Mp,
                       apply_d4, tile0, tile1, row_lo, row_hi, nc, coef);
  });
}

void launch_outer_f64(const F64Rows& r, int n, int np, int nc, const double* coef,
                      const double* fy, int ksplit, long kb, long ke, long rps, int accumulate,
                      double* zpart, double* fpart, hipStream_t s) {
  const F64Tiles t = f64_tiles(n);
  const long g = (long)t.ntile * t.ntile * ksplit * nc;
  with_cb(t.cb, [&](auto cb) {
    hipLaunchKernelGGL(outer_f64<decltype(cb)::value>, dim3((unsigned)g), dim3(256), 0, s, r.U,
                       r.F, coef, fy, np, r.Mp, ksplit, t.ntile, kb, ke, rps, accumulate, nc,
                       zpart, fpart);
  });
}

void launch_reduce_f64(int n, int np, int nc, int ksplit, const double* zpart,
                       const double* fpart, double* zsum, double* f, double norm, hipStream_t s) {
  const F64Tiles t = f64_tiles(n);
  const int zl = t.ntile * 16 * t.cb;
  const dim3 g((n + 63) / 64, n + 1, nc);
  // a single tile has few work-groups and many splits
  if (t.ntile == 1)
    hipLaunchKernelGGL(reduce_ksplit<16>, g, dim3(1024), 0, s, zpart, fpart, n, np, zl, ksplit,
                       zsum, f, norm);
  else
    hipLaunchKernelGGL(reduce_ksplit<4>, g, dim3(256), 0, s, zpart, fpart, n, np, zl, ksplit,
                       zsum, f, norm);
}

// weights and K-split partials of c->R1/c->Y1
void launch_sums_fp64(Ctx* c, int nc, int apply_d4, hipStream_t s, hipEvent_t* ev) {
  const F64Rows rows{c->U, c->F, c->rho_img, c->Mp};
  // image range [row_lo, row_hi): whole 64-row tiles of the weights kernel
  // (rows outside the range get zero coefficients), and the outer GEMM's K
  // range from the 8-row step below row_lo to the step above row_hi
  const long t0 = c->row_lo / 64, t1 = (c->row_hi + 63) / 64;
  if (ev) (void)hipEventRecord(ev[0], s);
  launch_weights_f64(rows, c->n, c->np, nc, c->Y1, c->R1, c->fy, c->fpsi, apply_d4, t0, t1,
                     c->row_lo, c->row_hi, c->coef, s);
  if (ev) (void)hipEventRecord(ev[1], s);
  const long kb = c->row_lo / WB_KC * WB_KC;
  const long ke = round_up_l(c->row_hi, WB_KC);
  const long rps = round_up_l((ke - kb + c->ksplit - 1) / c->ksplit, WB_KC);
  launch_outer_f64(rows, c->n, c->np, nc, c->coef, c->fy, c->ksplit, kb, ke, rps, 0, c->zpart,
                   c->fpart, s);
  if (ev) (void)hipEventRecord(ev[2], s);
}

int launch_pa_fp64(Ctx* c, int nc, int apply_d4, hipStream_t s, hipEvent_t* ev) {
  launch_sums_fp64(c, nc, apply_d4, s, ev);
  // zsum -> c->d2v_out (padded), normalised f -> c->f_out
  launch_reduce_f64(c->n, c->np, nc, c->ksplit, c->zpart, c->fpart, c->d2v_out, c->f_out,
                    1.0 / (c->n_eff * c->n_syms), s);
  if (ev) (void)hipEventRecord(ev[3], s);
  return 0;
}

}  // namespace tdscha
