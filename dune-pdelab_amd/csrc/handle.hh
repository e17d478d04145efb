// handle.hh -- the state behind one pdelab_gpu_gridoperator handle (internal to the
// library) and the per-degree apply launcher shared by its translation units.
#ifndef PDELAB_HANDLE_HH
#define PDELAB_HANDLE_HH

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/pdelab_gpu.h"
#include "block_jacobi.hh"
#include "dg_kernels.hh"
#include "dg_load.hh"
#include "dg_mfma.hh"
#include "dg_tables.hh"
#include "dg_velocity.hh"
#include "output.hh"

using namespace pdelab_amd;

// Block Jacobi data of one operator (J or J^T): fast-diagonalisation entries or dense
// transposed inverse blocks, per cell or per boundary type.
struct BlockJacobiData {
  bool fdm = false, per_cell = false;
  bool valid64 = false, valid32 = false;
  long long entries = 0, esize = 0;
  double* d64 = nullptr;
  float* d32 = nullptr;
  // row-major copies of per-type dense blocks (bj_typed_kernel)
  double* rm64 = nullptr;
  float* rm32 = nullptr;
};

// Constants of the apply kernels on the device, one allocation.
struct DeviceTables {
  // constant-coefficient line matrices: [0] J, [1] J^T
  LineMats<double> lm64[2];
  LineMats<float> lm32[2];
  MfmaTab mfma[4];  // matrix-core apply: J, J^T, then their convection parts (cell-wise kappa)
};

struct pdelab_gpu_gridoperator {
  pdelab_config cfg;
  int device = 0;
  hipStream_t stream = nullptr;
  std::string err;
  Tables1D tab;
  DGArgs<double> a64;
  DGArgs<float> a32;
  LoadArgs la;
  GradArgs ga;
  long long ncells = 0, nloc = 0, N = 0;
  int n1 = 2;
  bool conv = false, vark = false;
  double* d_kappa = nullptr;
  float* d_kappa32 = nullptr;
  double* d_fc64 = nullptr;  // per-cell face coefficients (FC values per cell) of kappa
  float* d_fc32 = nullptr;
  double* d_fw64 = nullptr;  // per-cell kappa and face weights of the matrix-core apply
  double* d_R0 = nullptr;
  bool R0_valid = false;
  double* d_src = nullptr;
  double* d_ftab = nullptr;
  double* d_gtab = nullptr;
  double* d_diag = nullptr;
  double* d_dinv = nullptr;
  float* d_dinv32 = nullptr;
  bool diag_valid = false;
  double* w64[8] = {nullptr};
  float* w32[8] = {nullptr};
  void *d_small = nullptr, *h_small = nullptr;  // hold the partials, scalars and states below
  double* d_part64 = nullptr;
  float* d_part32 = nullptr;
  double* d_scal64 = nullptr;
  float* d_scal32 = nullptr;
  double* h_scal64 = nullptr;
  float* h_scal32 = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  hipEvent_t evk[2] = {nullptr, nullptr};  // of the Krylov loop's copies of the state
  double* d_applydot = nullptr;  // per-workgroup partials of the fused apply dot
  int* d_state = nullptr;        // device Krylov loop: {stopped (CG: the iteration), aborted, iteration, -}
  double* d_dstate = nullptr;    // {defect, def0, reduction, -}
  int* h_state = nullptr;        // pinned mirrors (the state's twice)
  double* h_dstate = nullptr;
  double* d_bscal = nullptr;     // device BiCGSTAB loop: {rho, rho_new, alpha, omega, beta}
  DeviceTables* d_tab = nullptr;  // constants of the apply kernels
  MfmaX mfma_x[4];
  bool sym[2] = {false, false};  // J / J^T have the structure of line_op_sym
  // apply kernel: 0 the row kernel (x-row chunks), 1 the general kernel (chunks of consecutive cells)
  int apply_variant = 0;
  // [0] J, [1] J^T, [2] J with dense inverse blocks (block SOR), [3] the diagonal blocks of J
  // themselves (iterative block Jacobi)
  BlockJacobiData bj[4];
  IBJOptions ibj_opt{1e-5, 100, 1, 1.0};
  void* d_ibj_stat = nullptr;  // int error code at 0, unsigned long long iteration sum at 8
  // reaction shift of the one-step stage operators: the kernels apply J + shift M
  double shift = 0.0;
  double prec_shift = 0.0;  // shift for which the cached diagonal and block Jacobi data hold
  double* os[4] = {nullptr, nullptr, nullptr, nullptr};  // one-step work vectors
  // flexible GMRES of the mixed-precision solve: the Arnoldi basis V (kFgmresRestart + 1
  // vectors) and the preconditioned directions Z (kFgmresRestart vectors), FP64
  static constexpr int kFgmresRestart = 10;
  double* fg[2 * kFgmresRestart + 1] = {nullptr};
  void* d_bjpart = nullptr;  // per-workgroup partials of the block Jacobi application
  // block SOR: cells ordered by hyperplane x + y + z, hyperplane s at
  // d_sor_order[sor_first[s] .. sor_first[s + 1]); relaxation factor omega
  int* d_sor_order = nullptr;
  std::vector<int> sor_first;
  double sor_omega = 1.0;
  // velocity field b(x) tabulated at the quadrature points (replaces the constant b of cfg):
  // device layouts of dg_velocity.hh, FP64 and FP32
  bool varb = false;
  double* d_bv64 = nullptr;
  double* d_bf64 = nullptr;
  float* d_bv32 = nullptr;
  float* d_bf32 = nullptr;
  VelArgs<double> va64;
  VelArgs<float> va32;
  VelArgs<double>* d_va64 = nullptr;  // device copy for the cell-block set-up
  MfmaVelTab* d_mfma_vel = nullptr;   // constants of the matrix-core apply with the field
  double* d_sortmp64 = nullptr;       // block SOR with a field: the right-hand side less the couplings
  float* d_sortmp32 = nullptr;
};

using H = pdelab_gpu_gridoperator;

#define HIPCHK(h, expr)                                                              \
  do {                                                                               \
    hipError_t e_ = (expr);                                                          \
    if (e_ != hipSuccess) {                                                          \
      (h)->err = std::string(#expr " failed: ") + hipGetErrorString(e_);             \
      return PDELAB_ERR_HIP;                                                         \
    }                                                                                \
  } while (0)

#define CHK(...)                     \
  do {                               \
    int s_ = (__VA_ARGS__);          \
    if (s_ != PDELAB_OK) return s_;  \
  } while (0)

inline long long apply_cpb(const H* h) {
  return h->n1 == 2 ? ApplyShape<2>::CPB : (h->n1 == 3 ? ApplyShape<3>::CPB : ApplyShape<4>::CPB);
}

// Whether an apply launch that the matrix cores do not take (FP32, Q1, see mfma_kernel) takes the
// row kernel (chunks of x-rows) rather than the general kernel (chunks of consecutive cells). Rows
// that split into whole chunks always do. The partial last chunk of a row is moved back to overlap
// the previous one (nx > CPB), and its overlapping lanes do work that is not stored, so such grids
// take the row kernel only for the constant-coefficient symmetric operator, where it is fastest
// (0.78 of the general kernel's time at Q3, 0.90 at Q2), with at most 1/8 (Q3) or 1/16 (Q2) of the
// row's lanes wasted. Decided per launch: set_kappa may change the operator after creation.
inline bool row_kernel(const H* h) {
  if (h->apply_variant != 0) return false;
  const long long cpb = apply_cpb(h), nx = h->a64.n[0];
  const long long span = (nx + cpb - 1) / cpb * cpb;
  if (span == nx) return true;
  if (nx < cpb || h->n1 == 2 || h->vark || h->conv || !h->sym[0] || !h->sym[1]) return false;
  return (span - nx) * (h->n1 == 4 ? 8 : 16) <= span;
}

// Chunks of one apply launch: the row kernel takes ceil(nx / CPB) chunks of every x-row,
// the general kernel ceil(ncells / CPB) chunks of consecutive cells.
inline long long apply_blocks_of(const H* h, bool row) {
  const long long cpb = apply_cpb(h);
  if (!row) return (h->ncells + cpb - 1) / cpb;
  return (h->a64.n[0] + cpb - 1) / cpb * h->a64.n[1] * h->a64.n[2];
}
inline long long apply_blocks(const H* h) { return apply_blocks_of(h, row_kernel(h)); }

// z-chunks walked by one workgroup of the row apply, for constant-coefficient symmetric
// operators (measured faster there; slower with cell-wise kappa): 2 at Q3; 8 at Q2, or 4
// where nz is a multiple of 4 but not of 8; else 1. The launch and the count of fused-dot
// partials both use it.
inline int apply_walk(const H* h) {
  if (!row_kernel(h) || h->vark || h->conv || !h->sym[0] || !h->sym[1]) return 1;
  const long long nz = h->a64.n[2];
  if (h->n1 == 4) return nz % 2 == 0 ? 2 : 1;
  if (h->n1 == 3) return nz % 8 == 0 ? 8 : (nz % 4 == 0 ? 4 : 1);
  return 1;
}

// The coefficient form of a matrix-core launch (dg_mfma.hh)
inline int mfma_kind(const H* h, bool vel) {
  if (!h->vark) return vel || (h->sym[0] && h->sym[1]) ? MFMA_CONST : MFMA_CONV;
  if (h->conv || !h->a64.weightsOn || (vel && h->a64.aniso)) return MFMA_GENERAL;
  return h->a64.aniso ? MFMA_TENSOR : MFMA_WEIGHT;
}

// Whether the matrix-core kernel (dg_mfma.hh) can take an FP64 apply: Q2 and Q3, planes of at least
// four cells (a wave's group) whose byte offsets stay below 4 GiB. A Q1 cell would fill an eighth of
// the 4x4x4 blocks.
inline bool mfma_shape(const H* h) {
  const long long np = (long long)h->a64.n[0] * h->a64.n[1];
  return h->apply_variant == 0 && h->n1 >= 3 && np >= 4 && np * h->nloc * 8 < (1LL << 32);
}
// Workgroups of a plane (16 cells each). Beyond about a thousand steps of workgroups along z a launch is
// bound by its work, below by a wave's latency, where this kernel is always the faster one.
inline long long mfma_wgs(const H* h) { return ((long long)h->a64.n[0] * h->a64.n[1] + 15) / 16; }

// Whether it does. us, row or general kernel -> matrix cores: 64^3 Q3 78.6 -> 61.6, convection 105.5 ->
// 66.3, lognormal kappa 117.5 -> 71.7; 96^3 Q2 145.1 -> 116.6, 204.2 -> 128.9, 265.0 -> 160.2; 83x61x71 Q2
// lognormal 116.8 -> 65.6; 100^3 Q3 337.5 -> 258.7; 32^3 Q2 7.5 -> 5.0; 24^3 Q3 5.8 -> 4.5. The other two
// kernels are the faster ones for
// * cell-wise kappa with convection or weightsOff, whose lane matrices are combined from nine
//   tables per face and step: 64^3 Q2 62 and 74 against 100, 96^3 Q3 445 and 463 against 604; small
//   grids 7.8 -> 6.0 (8^3 Q2);
// * planes that leave much of their last workgroup's 16 cells idle: 2x2x8192 Q2 9.5 against 19.3,
//   17x1x8192 Q2 25.6 against 33.6. The share of busy cells at which that ends depends on the
//   degree and the coefficient (Q2 constant 13 of 16, since there the others come closest);
// * one plane of 128^2 cells or more, where each start serves a single step: 512x512x1 Q2 32 against 44 us
//   (two planes 62 against 70), Q3 55 against 60; if rows split into whole chunks also with a diagonal
//   tensor (57 against 66, J^T at Q3 105 against 125) and with cell-wise kappa at Q2 (56 against 60; at Q3
//   y = J z 96 against 99, but J^T 110 against 102). Convection stays here (52 -> 44, Q3 95 -> 58).
// fused: r += R(x), where the other kernels need a second pass over three vectors. That moves the lines:
// 512x512x1 Q2 61 -> 54 us, 6x6x8192 Q2 77 -> 64; cell-wise kappa with convection 64^3 Q3 192 -> 166, 32^3 Q2
// 21 -> 17 (48^3 Q2 52 against 55).
inline bool mfma_kernel(const H* h, bool fused = false) {
  if (!mfma_shape(h)) return false;
  const int kind = mfma_kind(h, false);
  const bool q2 = h->n1 == 3;
  const long long wgs = mfma_wgs(h), np = (long long)h->a64.n[0] * h->a64.n[1], nz = h->a64.n[2], steps = wgs * nz;
  if (kind == MFMA_GENERAL) return steps < (fused ? 2500 : 256) || (fused && !q2 && nz > 1 && np >= 13 * wgs);
  const long long busy = kind == MFMA_CONV ? (q2 ? 8 : 6) : (q2 && kind == MFMA_CONST ? 13 : 9);
  if (steps > 1024 && np < (fused ? std::min(busy, 7LL) : busy) * wgs) return false;
  if (!fused && np >= 128 * 128 && nz <= (q2 && kind == MFMA_CONST ? 2 : 1)) {
    if (kind == MFMA_CONST) return false;
    if (kind == MFMA_TENSOR || (q2 && kind == MFMA_WEIGHT)) return !row_kernel(h);
  }
  return true;
}

// Whether its velocity-field form does: up to four points per direction (Q2 with intorderadd 0..3, Q3
// with 0 or 1), the field's in-plane byte offsets below 4 GiB. It replaces two kernels and is the
// slower one only on the thinnest planes: 2x2x8192 Q2 59 against 47 us, with a diagonal tensor or
// weightsOff 91 against 50 (Q3 116 against 85; 4x2x8192 92 against 90).
inline bool mfma_vel_kernel(const H* h) {
  const long long np = (long long)h->a64.n[0] * h->a64.n[1], m = h->tab.m;
  if (!mfma_shape(h) || m > 4 || !(h->vark || (h->sym[0] && h->sym[1])) || np * 6 * m * m * m * 8 >= (1LL << 32)) return false;
  const long long busy = mfma_kind(h, true) == MFMA_GENERAL ? 8 : (h->n1 == 3 ? 6 : 4);
  return mfma_wgs(h) * h->a64.n[2] <= 1024 || np >= busy * mfma_wgs(h);
}

// One launch of the matrix-core apply: workgroups of four waves of four cells cover a plane,
// zsegs of them a column. A wave's start (its first planes and constants) costs about two
// steps, so walks are long: up to 32 steps, 8 or more where that still gives 1024 workgroups
// (four waves per SIMD), and shorter only for 512 workgroups. Walks of 4 / 8 / 16 / 32 steps:
// 64^3 Q3 72 / 63 / 62 / 61 us, 64^3 Q2 - / 34.2 / 33.8 / 36.9 us; of 1 / 2 / 4: 32^3 Q2 7.5 / 7.0 /
// 6.9 us.
// Wide planes are walked in strips of 8 workgroups along x (mfma_strip): the 128 workgroups that an XCD
// holds are 2048 consecutive cells, whose y-neighbours its L2 keeps only if that is many rows.
// 2048x64x32 Q3 1693 -> 1034 us (row kernel 1240), 1024x32x32 Q3 362 -> 246 (row kernel 323), 512x128x32
// Q3 681 -> 503 (624), 2048x64x32 Q2 719 -> 534, 384x128x32 Q3 412 -> 382; 256x256 gains 5 % at Q3 and loses
// 1 % at 200x200; fewer than 8 planes lose up to 15 % at Q2.
struct MfmaGrid {
  long long wgs;  // workgroups of a plane
  int zsegs, zw;
  unsigned prow;  // workgroups of a row where the plane is walked in strips, else 0
};
inline MfmaGrid mfma_grid(const H* h) {
  const long long nx = h->a64.n[0], nz = h->a64.n[2];
  MfmaGrid g;
  g.wgs = mfma_wgs(h);
  auto cover = [&](long long target) { return (target + g.wgs - 1) / g.wgs; };
  const long long segs = std::max({(nz + 31) / 32, std::min(cover(1024), (nz + 7) / 8), std::min(cover(512), nz)});
  g.zw = (int)((nz + segs - 1) / segs);
  g.zsegs = (int)((nz + g.zw - 1) / g.zw);
  g.prow = nx > 256 && h->a64.n[1] > 1 && nz >= 8 ? (unsigned)((nx + 15) / 16) : 0u;
  return g;
}
inline long long mfma_blocks(const H* h) {
  const MfmaGrid g = mfma_grid(h);
  return g.wgs * g.zsegs;
}

inline int fail(H* h, int code, const std::string& msg) {
  if (h) h->err = msg;
  return code;
}

inline int grid_for(long long n) {
  long long b = (n + 255) / 256;
  return (int)std::max(1LL, std::min(b, 4096LL * 8));
}

// per-cell face coefficients and operator arguments of the precision T
template <typename T>
inline const T* fc_for(H* h);
template <>
inline const double* fc_for<double>(H* h) { return h->d_fc64; }
template <>
inline const float* fc_for<float>(H* h) { return h->d_fc32; }
template <typename T>
inline const DGArgs<T>& args_for(H* h);
template <>
inline const DGArgs<double>& args_for<double>(H* h) { return h->a64; }
template <>
inline const DGArgs<float>& args_for<float>(H* h) { return h->a32; }

template <typename T>
inline const LineMats<T>* line_mats(H* h, bool trans);
template <>
inline const LineMats<double>* line_mats<double>(H* h, bool trans) { return h->d_tab->lm64 + (trans ? 1 : 0); }
template <>
inline const LineMats<float>* line_mats<float>(H* h, bool trans) { return h->d_tab->lm32 + (trans ? 1 : 0); }

// y (+)= J z (or J^T z) on the handle's stream for Q_{N1-1}: mode 0 y = J z, 1 y += J z,
// 2 y = J z with the fused z.(Jz) partials in dotp. Defined in apply_q<N1-1>.hip.
template <int N1, typename T>
int launch_apply_n(H* h, const T* z, T* y, const T* fc, const DGArgs<T>& a, bool trans, int mode, T* dotp,
                   const int* stop);

// The FP64 apply on the matrix cores (apply_mfma.hip; modes as above and, with a vector w,
// 3: w.y partials, 4: (w.y, y.y) partials, 5: y += J z + w) and its constants, from the 1D
// matrices of J and J^T without reaction and their convection parts.
int launch_apply_mfma(H* h, const double* z, double* y, bool trans, int mode, double* dotp, const int* stop,
                      const double* w = nullptr);
void mfma_setup(H* h, const DGArgs<long double>& al, const LineMats<long double> (&m)[2],
                const LineMats<long double> (&mconv)[2], MfmaTab (&t)[4]);
MfmaArgs mfma_args(const H* h, bool trans);
// The same with the velocity field's terms (apply_mfma_vel.hip), and their constants.
int launch_apply_mfma_vel(H* h, const double* z, double* y, bool trans, bool accum, const int* stop);
int mfma_vel_setup(H* h);
int mfma_weights(H* h);  // d_fw64 from the current face coefficients

// Block Jacobi (block_jacobi.hip): data set-up for the given precision (64 or 32),
// invalidation when kappa changes, the launches (BJ_PREC / BJ_ADD / BJ_CGR / BJ_CGD / BJ_CGX, see
// block_jacobi.hh; the partials go to d_bjpart, their count to *nparts) and the
// diagonal blocks themselves (ncells * nloc^2, row-major).
int bj_prepare(H* h, bool trans, int precision);
void bj_invalidate(H* h);
void bj_free(H* h);
template <typename T, typename A>
int bj_launch(H* h, bool trans, int mode, BJVec<T, A> v, int* nparts);
// Whether the CG loop lets the p update apply W^{-1} again (BJ_CGD, BJ_CGX) instead of storing z.
bool bj_cg_recompute(const H* h, bool trans);
int bj_block_diagonal(H* h, bool trans, double* blocks);
// Block SOR (block_sor.hh): data set-up (dense blocks of J) and one sweep, from v = 0
// (v = W^{-1} d, the solvers) or in place from the v given (inplace); the kernels store
// nothing when *stop is set.
int sor_prepare(H* h, int precision);
template <typename T>
int sor_launch(H* h, const T* d, T* v, const int* stop, bool inplace);
// Iterative block Jacobi (bj_iter_kernel): the diagonal blocks of J, and one application
// v = W^{-1} d (v += W^{-1} d with add); the block solvers' error code goes to *err (kept at
// the first nonzero), their iteration sum is added to *iters when non-null.
int ibj_prepare(H* h, int precision);
template <typename T>
int ibj_launch(H* h, const T* d, T* v, int* err, unsigned long long* iters, const int* stop, bool add);
// Assembled Jacobian in the 7-point block pattern (jacobian.hh) and its apply y = A z.
int jac_assemble(H* h, bool trans, double* blocks, long long* cols);
int jac_block_apply(H* h, const double* blocks, const long long* cols, const double* z, double* y);
// Velocity field (velocity.hip): set or clear the tabulated b(x) (host arrays in the layout of
// pdelab_gpu_set_velocity_field), add its convection terms y += C z or y += C^T z (nothing
// stored when *stop is set) and their diagonal, free the data.
int vel_set(H* h, const double* b_vol, const double* b_face);
template <typename T>
int vel_launch(H* h, const T* z, T* y, const int* stop, bool trans);
int vel_diag(H* h, double* diag);
void vel_free(H* h);
// Block SOR with a velocity field: *out = d less the convection couplings of the cells of
// hyperplane d_sor_order[first .. first + count) (lower neighbours; all with inplace).
template <typename T>
int vel_sor_rhs(H* h, const T* d, const T* v, int first, int count, bool inplace, const T** out);

#endif
