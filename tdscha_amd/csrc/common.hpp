// Shared definitions for the tdscha_amd HIP library (gfx950 / CDNA4).
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstdio>
#include <string>
#include <utility>
#include <vector>

namespace tdscha {

// ---------------------------------------------------------------- errors
void set_error(const std::string& msg);
const char* last_error();

#define TDS_CHECK_HIP(expr)                                                   \
  do {                                                                        \
    hipError_t _e = (expr);                                                   \
    if (_e != hipSuccess) {                                                   \
      ::tdscha::set_error(std::string(#expr) + ": " + hipGetErrorString(_e)); \
      return -1;                                                              \
    }                                                                         \
  } while (0)

#define TDS_REQUIRE(cond, code, msg)            \
  do {                                          \
    if (!(cond)) {                              \
      ::tdscha::set_error(msg);                 \
      return (code);                            \
    }                                           \
  } while (0)

// ------------------------------------------------------------ constants
constexpr double RY_TO_K = 157887.32400374097;
constexpr int kTile = 128;      // column tile of the weighted outer-product GEMM
constexpr int kRowTile = 64;    // image rows per workgroup of the weights GEMM
constexpr int kMaxChains = 8;   // perturbations applied in one batched call
constexpr int kPartBlocks = 1024;  // blocks of the grid-wide maxima in the split prep

inline int round_up(int x, int m) { return (x + m - 1) / m * m; }
inline long round_up_l(long x, long m) { return (x + m - 1) / m * m; }

// MFMA operand vector types
// direct global -> LDS copy of 16 bytes per lane: lane i's bytes land at
// lds_base + 16 i (lds_base is wave-uniform)
typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef __attribute__((address_space(1))) void* gbl_ptr_t;
__device__ __forceinline__ void dma16(const void* g, void* lds_base) {
  __builtin_amdgcn_global_load_lds((gbl_ptr_t)g, (lds_ptr_t)lds_base, 16, 0, 0);
}

// s_waitcnt vmcnt(N) (expcnt and lgkmcnt not waited), gfx9 encoding
#define TDS_WAIT_VMCNT(N) \
  __builtin_amdgcn_s_waitcnt(((N) & 15) | (((N) >> 4) << 14) | 0x0F70)

// Work-group barrier without a memory fence.  The direct-to-LDS copies are
// completed explicitly (vmcnt) before it; this waits for the wave's own LDS
// reads and writes (lgkmcnt(0)), and the empty asm statements keep the
// compiler from moving memory accesses across it.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_s_waitcnt(0xC07F);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// FP64 matrix products of 4 x 4 x 4 blocks
__device__ __forceinline__ double mfma4(double a, double b, double c) {
  return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}

// v of the lane 4 R lanes before, cyclic within a row of 16 lanes
template <int R>
__device__ __forceinline__ double rot4(double v) {
  if constexpr (R == 0) return v;
  constexpr int ctrl = 0x120 + 4 * R;   // row_ror:4R
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), ctrl, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), ctrl, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// acc += A B for a 16 x 16 block, 4 of the K index: A[i][k] i = lane % 16,
// B[k][j] j = lane % 16, k = lane / 16; acc[r] of a lane is the element of row
// 4 q + lane / 16, column 4 ((q - r) % 4) + lane % 4 (q = lane / 4 % 4)
__device__ __forceinline__ void mma16(double a, double b, double (&acc)[4]) {
  acc[0] = mfma4(a, b, acc[0]);
  acc[1] = mfma4(a, rot4<1>(b), acc[1]);
  acc[2] = mfma4(a, rot4<2>(b), acc[2]);
  acc[3] = mfma4(a, rot4<3>(b), acc[3]);
}

// Arrays carved from one allocation (256-byte aligned): add() each, allocate total()
// bytes, assign() the base.
class Carve {
 public:
  template <typename T>
  void add(T** p, size_t count) {
    parts_.push_back({reinterpret_cast<void**>(p), total_});
    total_ += (sizeof(T) * count + 255) / 256 * 256;
  }
  size_t total() const { return total_; }
  void assign(void* base) const {
    for (const auto& q : parts_) *q.first = static_cast<char*>(base) + q.second;
  }

 private:
  std::vector<std::pair<void**, size_t>> parts_;
  size_t total_ = 0;
};

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

enum Precision { PREC_FP64 = 0, PREC_FP16X2 = 1, PREC_BF16X2 = 2 };

// Per-precision image storage for the split-precision kernels.
struct SplitStore {
  void* Uh = nullptr;   // image-major blocks, hi part of the scaled U (weights A operand)
  void* Ul = nullptr;   //   lo part
  float* FA = nullptr;  // image-major FP32 blocks of F (weights epilogue)
  float* UA32 = nullptr;  // image-major FP32 blocks of U (weights epilogue)
  void* UhT = nullptr;  // mode-major blocks, hi part of the scaled U (outer GEMM)
  void* UlT = nullptr;  //   lo part
  float* XT = nullptr;  // mode-major FP32 blocks of F (outer B build)
  float* YT = nullptr;  // mode-major FP32 blocks of fY U / 2 (outer B build)
  double* su = nullptr;  // [np] power-of-two column scale of U
  double* sf = nullptr;  // [np] power-of-two column scale of F
  double* umax = nullptr;  // [np] max |U| per column (unscaled)
  double* fmax = nullptr;  // [np] max |F| per column (unscaled)
  float* colw = nullptr;   // [3, np] 1/su, 1/sf, fpsi in FP32 (weights epilogue)
  bool ready = false;
};

// Host calls up to this size pass their vectors through pinned memory that the kernels
// access: a copy each way is a launch of its own (4 to 5 us on the device, 16 atoms:
// 82 -> 40 us per call).  Longer vectors are copied.
constexpr size_t kPinned = 65536;

// Orbit form of the averages (orbit.hip)
constexpr int kProbe = 8;            // probe configurations of the rank search
constexpr int kOrbRank = 6;          // largest orbit of a chain
constexpr int kOrbPairs = 24;        // rotated perturbations of one pass
constexpr double kOrbTol = 1e-13;    // accuracy of the relation
constexpr double kOrbGain = 16.0;    // largest sum of its factors
constexpr int kOrbClean = 2;         // Lanczos steps between projections on the sector
// least time that the form saves (microseconds, estimated, one chain; the kernels take
// 1.5 to 2 times the estimate at these sizes): the search, a wait for the host of about
// 40 us and the rotations cost a call of one chain 150 to 200.  Averages of one IR
// vector, host arrays: 54 atoms x 2500 (estimate 209) general 434 us, orbit 247; 128
// atoms x 450 (217) about 570, 460; just below the line, 54 x 2050 (172) and 128 x 360
// (174), the general form takes 365 and 530.
constexpr double kOrbWorthUs = 175.0;

struct OrbPlan {
  bool ok = false;         // some chain takes the form
  int prec = 0;            // of its averages
  int nc = 0, chains = 0, rank = 0;   // chains, those with an orbit, their largest rank
  struct List {
    int n, at[kMaxChains];
  };
  List others = {};        // the chains without, in the general form
  struct Round {           // a pass: its first matrix and their number, its pairs
    int mat, mats, pair, count;
  };
  std::vector<Round> rounds, clean_rounds;   // of the averages, of the clean-up
  std::vector<char> host;
  double* general = nullptr;   // [kMaxChains, n], [kMaxChains, n, n] averages of `others`
  void* dev = nullptr;
  size_t cap = 0;
  int4 *mats = nullptr, *cmats = nullptr;
  int2 *pairs = nullptr, *clean = nullptr;
  double* C = nullptr;
};

struct Ctx;

struct Orbit {
  bool usable = false;     // tables built
  int chains = 0;          // chains of the last call or run that took the form
  // found by the first Lanczos run (-1: not yet)
  int group = -1;          // the symmetries are closed under multiplication
  int trans = -1;          // the translation average commutes with them
  int nsym = 1, npanel = 0, rows = 0;
  long Mp = 0;
  std::vector<double> syms;               // host copy of the symmetry blocks
  std::vector<int> gens;                  // generators of the group
  std::vector<double> look;               // [8][8][n] S_j p of orbit_candidates
  double* arena = nullptr;                // holds start, S, ST, pu, pf (and U, F, rho)
  size_t arena_bytes = 0;
  int* start = nullptr;                   // [npanel + 1]
  double *S = nullptr, *ST = nullptr;     // [npanel, nsym, 32, 32] panels of S_j, transposed
  double *U = nullptr, *F = nullptr, *rho = nullptr;       // [Mp, np] the configurations
  double *pu = nullptr, *pf = nullptr, *pones = nullptr;   // [rows, np] probe images
  double* work = nullptr;                 // holds the workspaces below
  double *ppart = nullptr;                // partial sums of the probe
  double* pout = nullptr;                 // pinned host memory: its results
  double *R1 = nullptr, *Y1 = nullptr;    // [kOrbPairs, np(, np)] rotated inputs
  double *Rb = nullptr, *Yb = nullptr;    // [2 kMaxChains, np(, np)] unpacked vectors
  double *coef = nullptr, *z = nullptr, *f = nullptr;
  // the configurations as a context of their own, with what the split precisions need
  // (made at the first plan in one of them); its inputs and outputs are set per pass
  Ctx* sub = nullptr;
  OrbPlan plan[1];                        // of the synchronous entries
};

// ------------------------------------------------------------- context
struct Ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  // problem
  int n = 0;      // modes
  int np = 0;     // padded modes (multiple of kTile)
  int N = 0;      // configurations
  int n_syms = 0;
  long M = 0;     // images N * n_syms
  long Mp = 0;    // padded images (multiple of the K split granule)
  double T = 0;
  double n_eff = 0;
  // image range of the next perturbed-average pass, [row_lo, row_hi) in
  // image order b = i * n_syms + j (default: every image)
  long row_lo = 0;
  long row_hi = 0;
  // symmetric image ensemble, device resident
  double* U = nullptr;      // [Mp, np] S_j x_i
  double* F = nullptr;      // [Mp, np] S_j y_i
  double* rho_img = nullptr;// [Mp]
  double* fy = nullptr;     // [np]
  double* fpsi = nullptr;   // [np]
  double* w = nullptr;      // [np]
  // pinned host memory that the kernels read and write directly, for calls whose
  // vectors take at most kPinned bytes each way (null: no such call)
  char* pinned = nullptr;   // [2 kPinned]: in, out
  // per-call buffers
  double* R1 = nullptr;     // [kMaxChains, np]
  double* Y1 = nullptr;     // [kMaxChains, np, np]
  double* coef = nullptr;   // [kMaxChains, Mp, 4] (c1, c2, alpha, beta)
  double* zpart = nullptr;  // [kMaxChains, ksplit] partial tiles of the outer GEMM
  double* fpart = nullptr;  // [kMaxChains, ksplit, np]
  double* f_out = nullptr;  // [kMaxChains, np]
  double* d2v_out = nullptr;// [kMaxChains, np, np]
  int ksplit = 0;
  // split precision
  SplitStore split[3];
  void* Y1h = nullptr;      // [kMaxChains, np, np] (16-bit)
  void* Y1l = nullptr;
  double* ysc = nullptr;    // [kMaxChains] power-of-two scale of split Y1
  double* ysc3 = nullptr;   // [kMaxChains] scale of the folded fY R1 column
  double* bsc = nullptr;    // [kMaxChains, np] column scale of split B
  double* pmax = nullptr;   // [kMaxChains, kPartBlocks, 2] per-block maxima of the split prep
  float* epi = nullptr;     // [kMaxChains, 2, np] fY R1 and R1 (weights epilogue)
  float* coef32 = nullptr;  // [Mp/16, kMaxChains, 4, 16] FP32 coefficients for the outer GEMM
  double* wpart = nullptr;  // [kMaxChains, np/128, Mp, 4] weights row-dot partials
  int ksplit_s = 0;          // K split of the split-precision outer GEMM
  float* zpart32 = nullptr;  // [kMaxChains, ksplit_s, np, np] raw FP32 partial tiles
  double* fpart_s = nullptr; // [kMaxChains, ksplit_s, np]
  double* sbsc = nullptr;    // [kMaxChains, np] B column scales of the last call
  // Wigner / harmonic helpers
  double* pair_ca = nullptr;   // [npairs]
  double* pair_cb = nullptr;
  double* pair_sm = nullptr;
  double* pair_sp = nullptr;
  double* pair_harm_a = nullptr;
  double* pair_harm_b = nullptr;
  int* pair_row = nullptr;
  int* pair_col = nullptr;
  // standard representation helpers
  double* std_coef = nullptr;  // [8, npairs] harmonic 2x2 block coefficients
  double* inv_coef = nullptr;  // [4, npairs] inverse harmonic 2x2 blocks (preconditioner)
  double* yw = nullptr;        // [np] Y_w
  double* reaw = nullptr;      // [np] ReA_w
  // gamma-only translational projector
  int n_cells = 0;
  int n_cart = 0;
  double* pols = nullptr;      // [n_cart, n]
  int* inv_perms = nullptr;    // [n_cells, n_cart]
  // translation group orbits (when the permutations form a group): dof J
  // lies in the orbit of rep_dof[jrep[J]], reached by inv_perms[ju[J]]
  int n_rep = 0;
  int* rep_dof = nullptr;      // [n_rep]
  int* jrep = nullptr;         // [n_cart]
  int* ju = nullptr;           // [n_cart]
  double* rep_sum = nullptr;   // [kMaxChains, n_rep, n_cart]
  double* tproj = nullptr;     // [n, n]
  double* cart_tmp = nullptr;  // [kMaxChains, n_cart, n_cart] x2
  double* cart_tmp2 = nullptr;
  double* mode_tmp = nullptr;  // [kMaxChains, n, n_cart]
  // scratch for the anharmonic wrapper
  double* psi_dev = nullptr;   // [kMaxChains, len_psi] x2
  double* psi_out_dev = nullptr;
  double* f_fin = nullptr;     // [kMaxChains, n] perturbed averages (normalised)
  double* d2v_fin = nullptr;   // [kMaxChains, n, n]
  double* f_proj = nullptr;    // [kMaxChains, n] translation-projected f
  double* stage_in = nullptr;  // [kMaxChains, n + n*n] host<->device staging
  double* stage_out = nullptr;
  // host-side copies of the symmetry description
  std::vector<int> block_dim, block_off, block_modes, sym_block_id;
  // operator-rotation form (flag TDSCHA_CTX_ROTATE_OPERATORS): U, F hold the
  // configurations themselves (n_syms = 1 for the kernels) and every pass is
  // run on rotated perturbations S_j^T R1, S_j^T Y1 S_j, its results rotated
  // back and summed over the rot_nsym symmetries
  bool rotate = false;
  int rot_nsym = 1;
  int rt_dmax = 0;             // largest block
  int* rt_cols = nullptr;      // [dmax, n] modes of each mode's block (position-major)
  int* rt_d = nullptr;         // [n] size of each mode's block
  double* rt_sr = nullptr;     // [rot_nsym, dmax, n] S_j[m, cols(m)[t]]   (row m of S_j)
  double* rt_sc = nullptr;     // [rot_nsym, dmax, n] S_j[cols(m)[t], m]   (column m)
  int* rt_bs = nullptr;        // [n] first mode of each mode's block (panel kernels)
  int* rt_pstart = nullptr;    // [rt_npanel + 1] first mode of each panel, then np
  int rt_npanel = 0, rt_nreal = 0;
  bool rt_panels = false;      // every block consecutive modes, at most 24: panel kernels
  double* R1_base = nullptr;   // [kMaxChains, np] unrotated padded inputs of a call
  double* Y1_base = nullptr;   // [kMaxChains, np, np]
  double* rot_t1 = nullptr;    // [kMaxChains, np, np] rotation intermediates
  double* rot_t2 = nullptr;
  double* rot_f = nullptr;     // [kMaxChains, np]
  Orbit orb;
};

int ensure_split(Ctx* c, int prec);

void orbit_plan_free(OrbPlan& p);
bool orbit_sized(const Ctx* c, int prec);
unsigned orbit_candidates(const Ctx* c, int nc, int prec, const double* R, long ld);
int orbit_sector(Ctx* c, bool* ok);
int orbit_plan(Ctx* c, int nc, unsigned mask, int prec, const double* x, hipStream_t s,
               OrbPlan& p);
bool orbit_ready(Ctx* c, int prec, hipStream_t s);
hipError_t dev_alloc(Ctx* c, void** p, size_t bytes);
template <typename T>
hipError_t dev_alloc(Ctx* c, T** p, size_t bytes) {
  return dev_alloc(c, reinterpret_cast<void**>(p), bytes);
}
int run_pa(Ctx* c, int nc, int apply_d4, int prec, double* f_dev, double* d2v_dev, hipStream_t s);
int run_pa_orbit(Ctx* c, const OrbPlan& p, int apply_d4, double* f_dev, double* d2v_dev,
                 hipStream_t s);
int orbit_clean(Ctx* c, const OrbPlan& p, double* x, const int* kk, const int* active,
                hipStream_t s);

// FP64 GEMM launches (pa_fp64.hip), shared by every caller of the kernels
struct F64Tiles {
  int ntile;  // column tiles
  int cb;     // columns of a tile / 16
};
F64Tiles f64_tiles(int n);
struct F64Rows {
  const double* U;    // [Mp, np] image rows
  const double* F;    // [Mp, np]
  const double* rho;  // [Mp]
  long Mp;
};
void launch_weights_f64(const F64Rows& r, int n, int np, int nc, const double* Y1,
                        const double* R1, const double* fy, const double* fpsi, int apply_d4,
                        long tile0, long tile1, long row_lo, long row_hi, double* coef,
                        hipStream_t s);
void launch_outer_f64(const F64Rows& r, int n, int np, int nc, const double* coef,
                      const double* fy, int ksplit, long kb, long ke, long rps, int accumulate,
                      double* zpart, double* fpart, hipStream_t s);
void launch_reduce_f64(int n, int np, int nc, int ksplit, const double* zpart,
                       const double* fpart, double* zsum, double* f, double norm, hipStream_t s);
void launch_sums_fp64(Ctx* c, int nc, int apply_d4, hipStream_t s, hipEvent_t* ev);
// One tile of modes (the image form): sums and output in one launch up to 256 partials.
// Its work-groups read whole 8 x 8 blocks of every partial (45 modes: 64 partials
// 5.0 us, 512 13.3); sums and symmetrisation as two kernels take about 10 us.
inline bool finish_in_one(const Ctx* c, int prec) {
  return prec == PREC_FP64 && !c->rotate && f64_tiles(c->n).ntile == 1 && c->ksplit <= 256;
}
void launch_finish_averages(Ctx* c, int nc, double* f, double* d2v, hipStream_t s);

}  // namespace tdscha
