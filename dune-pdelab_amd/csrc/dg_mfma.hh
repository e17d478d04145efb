// dg_mfma.hh -- FP64 apply y (+)= J z (J^T z) of the Q2 and Q3 DG operator on the matrix
// cores (v_mfma_f64_4x4x4_4b: four independent 4x4x4 products per wave).
//
// One wave holds four consecutive cells of an xy-plane, one per block of the instruction,
// and walks them along z. Within a block the 16 lanes are a grid over two of the cell's
// three index directions and a lane's registers run over x, so a lane's x-line is
// contiguous in memory. With data D[lane%4][lane/16] the instruction contracts the
// lane/16 index with a 4x4 matrix L held one entry per lane (row lane%4, column lane/16):
//   L as the first operand:  out keeps lane%4, lane/16 becomes the new index;
//   L as the second operand: the contracted index moves to lane%4, the other to lane/16.
// Two lane layouts are used, T0 (lane%4 = y, lane/16 = z) and T1 (lane%4 = z, lane/16 = y):
//   s_z  T0 -> T1   own, lower and upper neighbour, second operand
//   s_y  T1 -> T1   own, lower and upper neighbour, first operand
//   s_x  T1         register lines; the neighbours' trace and derivative come from the
//                   adjacent blocks by DPP row shifts, from memory at the wave's two ends
//   M_x in registers, M_y T1 -> T0, M_z T0 -> T0, then a contiguous store.
// The T0 and T1 readings of a cell are strided in memory: as global loads each instruction
// touches 32 (T0) or 64 (T1) 64-byte segments for 1 KB, and the L1 then serves one segment per
// cycle and bounds the kernel. The wave therefore moves its four consecutive cells (one
// contiguous run) with fully coalesced loads and stores and changes layout through an LDS
// region of its own: no workgroup barrier, the next step's loads in flight during a step.
// A boundary face replaces its cell's matrices, so cell-wise coefficients, convection,
// transposition and partial rows (any nx: a block whose row ends ignores its neighbour)
// take the same path. Q2 pads the 4x4 blocks with zeros. mfma_kernel() says which calls come here.
//
// Measured (y = J z, three states in turn, row kernel -> this one): 64^3 Q3 76.2 -> 61.6 us (268 MB,
// 4.4 TB/s), lognormal kappa 117 -> 72 us; 96^3 Q2 145 -> 118 us, convection 204 -> 129 us. At 64^3 Q3 it
// reads 1.33x and writes 1.0x the algorithmic bytes, 1.17x in all, runs at 41 % of the FP64 rate with 10
// waves per CU, and no unit is busy for more than 40 % of the time: the latency of a step's loads, products
// and layout changes bounds it. At Q2 9/16 of the matrix lanes are padding.
// With a velocity field (before: the apply with b = 0, then a kernel of one cell per wave and
// seven barrier phases over LDS): 64^3 Q2 296 -> 107 us (340 MB, 3.2 TB/s), 40^3 Q3 145 -> 46 us, with
// cell-wise kappa 141 -> 66 us. Two waves per SIMD hold 170 to 256 registers (of the Q3 instances six
// spill 20 to 72 bytes all the same: cell-wise kappa, and diagonal tensors or weightsOff in y +=); three
// spilled everywhere and were slower (112 us). Bound by the latency of a step's chain of 93 (Q2) or 120
// products.
#ifndef PDELAB_DG_MFMA_HH
#define PDELAB_DG_MFMA_HH

#include <hip/hip_runtime.h>

#include <type_traits>

#include "block_reduce.hh"
#include "dg_kernels.hh"

namespace pdelab_amd {

// Constants of one operator (J or J^T). Lane matrices: entry (i, k) at 4 i + k, zero padded.
// [0] is the y direction, [1] z. Constant kappa: the whole 1D matrices; cell-wise kappa:
// own/dlo/dhi/nlo/nhi (and A, P, Q of the x-lines) hold the convection part only.
struct MfmaTab {
  double own[2][16], dlo[2][16], dhi[2][16], nlo[2][16], nhi[2][16];
  double M[16];
  // cell-wise kappa: own = S (kappa K + whi U1 + P (U2, U3) - wlo U4), neighbours
  // S (wlo X1 + P X2 + whi X3) below and S (P X4 + whi X5 + wlo X6) above
  double K[16], U[4][16], X[6][16];
  // the same for weightsOn and isotropic kappa, whose face has one weight w (P = 2 alphak w):
  // own = S (kappa K + w WL + w' WU), neighbours S w NL and S w' NU, boundary faces S kappa (BL, BU)
  double WL[16], WU[16], NL[16], NU[16], BL[2][16], BU[2][16];
  // x-lines: s = A u + Pl vl + Ql dl + Pr vr + Qr dr, corrections Dlo u, Dhi u at the boundary
  double A[4][4], Pl[4], Ql[4], Pr[4], Qr[4];
  double Dlo[4][4], Dhi[4][4];
};

// x-line constants held in scalar registers through the walk. The basis is symmetric about
// 1/2: the derivative functionals satisfy d0[j] = -d1[n-1-j], A and the mass M are
// centro-symmetric, and the upper face's vectors are the lower face's reversed (P) and
// reversed with the sign changed (Q). (A, P, Q) = (M^-1 A_x + V c, neighbour value, neighbour
// derivative) for the constant symmetric operator, (M^-1 K, M^-1 e0, M^-1 d0) for cell-wise kappa.
struct MfmaX {
  double d1[4], M[4][4], A[4][4], P[4], Q[4];
};

// Constants of the velocity field's terms for M points per direction. Lane matrices as above:
// LB, LD point by node, WB = (w B)^T, WDy = vs_1 (w D)^T, WDz = vs_2 (w D)^T node by point; scalars
// for the x-lines, indexed [point][node]: B, D, BW = w B, DW = vs_0 w D. vs = -|K| / h, area = |K| / h.
struct MfmaVelTab {
  double LB[16], LD[16], WB[16], WDy[16], WDz[16];
  double B[4][4], D[4][4], BW[4][4], DW[4][4];
};

struct MfmaArgs {
  int nx, ny, nz;
  unsigned np;     // cells of a plane
  int zw, zsegs;   // z-steps of a wave, waves per column
  unsigned prow, prows;  // workgroups of a row (rounded up) and such rows of a plane, if walked in strips; else 0
  double vc;       // reaction V c
  // cell-wise kappa: S per direction, face signs (1, theta) of J or (-theta, -1) of J^T,
  // Dirichlet penalty factor, boundary types
  double S[3], fg, fh, alphak;
  int weightsOn, bc[6];
  MfmaX x;
  // velocity field at the quadrature points (layout of dg_velocity.hh), or null
  const double *bv, *bf;
  const MfmaVelTab* vt;
  double vs[3], area[3];
};

// Constant kappa, symmetric line operator (no convection); cell-wise kappa with one weight per
// face (weightsOn, no convection; rows of kappa and w of the lower x, y, z face), the same for
// a diagonal tensor (rows of a_x, a_y, a_z and the weights; the same arithmetic, so that
// diag(kappa, kappa, kappa) gives the bits of kappa); cell-wise kappa in general (weightsOff,
// convection; the FC values per cell of the row kernel); constant kappa with convection.
enum { MFMA_CONST = 0, MFMA_WEIGHT = 1, MFMA_GENERAL = 2, MFMA_CONV = 3, MFMA_TENSOR = 4 };
constexpr int mfma_row(bool tensor) { return tensor ? 6 : 4; }  // values of a cell's row

// Waves per SIMD the register allocation aims at without a velocity field: no vector register goes to
// scratch. (With 96 bytes of it the face-weight Q3 kernel took 97 instead of 76 us at 64^3, and 72 bytes
// cost the fused-dot Q2 one 5 of 17 us at 32^3. Up to 130 scalar registers are parked in vector lanes.)
template <int N1, int KIND, int MODE>
constexpr int mfma_waves() {
  if (KIND == MFMA_GENERAL) return 2;
  if (KIND == MFMA_TENSOR) return N1 == 4 ? 2 : 3;
  if (KIND == MFMA_WEIGHT && N1 == 4) return MODE < 3 ? 3 : 2;
  return KIND == MFMA_WEIGHT || N1 == 4 ? 3 : 4;
}

// w of each face: the common weight omega kappa of both sides, half the harmonic average
__global__ __launch_bounds__(256) static void mfma_weight_kernel(const double* __restrict__ fc, double* __restrict__ fw,
                                                                 long long ncells, int tensor) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncells) return;
  const int k = tensor ? 3 : 1;
  double* f = fw + mfma_row(tensor) * c;
  for (int d = 0; d < k; ++d) f[d] = fc[FC * c + d];
#pragma unroll
  for (int d = 0; d < 3; ++d) f[k + d] = fc[FC * c + FCF + 3 * d + 1];
}

typedef double mfma_d2 __attribute__((ext_vector_type(2), aligned(8)));  // in a vector: 8-byte aligned
typedef double mfma_a2 __attribute__((ext_vector_type(2)));              // in LDS

__device__ __forceinline__ double mfma4(double a, double b, double c) {
  return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}

// Global and constant address spaces by name: a pointer that passed through per_step would
// otherwise be generic, and its loads flat.
typedef const double __attribute__((address_space(1))) * mfma_gp;
typedef double __attribute__((address_space(1))) * mfma_gpw;
typedef const MfmaTab __attribute__((address_space(4))) * mfma_tp;

// A uniform pointer whose loads and address arithmetic the compiler may not move out of the
// loop step: a vector base stays a scalar register pair plus a 32-bit lane offset, and the
// x-line constants of the operators without the symmetric form, which exceed the scalar
// registers, are loaded again each step instead of being parked in vector lanes (one
// v_readlane per 32 bits and use).
template <typename Q, typename P>
__device__ __forceinline__ Q per_step(P p) {
  unsigned long long v = reinterpret_cast<unsigned long long>(p);
  asm volatile("" : "+s"(v));
  return (Q)v;
}

// A lane offset kept as 32 bits up to its use: widened outside the loop it would take two
// registers and a 64-bit addition per access.
__device__ __forceinline__ unsigned here(unsigned off) {
  asm volatile("" : "+v"(off));
  return off;
}

// Staging of a wave's four cells: each lane moves PER elements per set, element lane + 64 p of
// NE (Q3: 16-byte pairs, Q2: doubles, since a cell of 27 is no whole number of pairs).
// LDS slots: Q2 linear; Q3 pairs permuted within a cell so that the 16 lanes of a quarter wave
// touch the 16 distinct pair positions of the 64 banks in the T0, the T1 and the linear
// pattern alike. pair (b, z, y, h): position bits h^b0, y0^z1, y1^z0, z0^b1, then z1, b.
template <int N1>
struct MfmaStage {
  static constexpr int NL = N1 * N1 * N1;
  static constexpr int NE = N1 == 4 ? 128 : 108, NX = N1 == 4 ? 64 : 54;  // elements of a set, of the two end cells
  static constexpr int ES = N1 == 4 ? 16 : 8;                              // bytes of an element
  static constexpr int BUF = 4 * NL, XBUF = 2 * NL;                        // doubles
  static constexpr int WAVE = 4 * BUF + XBUF;  // own, next (alternating), lower y, upper y, ends
  using E = typename std::conditional<N1 == 4, mfma_d2, double>::type;
  __device__ static __forceinline__ int slot(int b, int zz, int yy) {  // double offset of an x-line
    if constexpr (N1 == 4) {
      const int lo = (b & 1) | (((yy & 1) ^ (zz >> 1)) << 1) | (((yy >> 1) ^ (zz & 1)) << 2) |
                     (((zz & 1) ^ (b >> 1)) << 3);
      return 2 * (32 * b + 16 * (zz >> 1) + lo);
    } else {
      return NL * b + 3 * yy + 9 * zz;
    }
  }
  __device__ static __forceinline__ int eslot(int q) {  // double offset of element q of a set
    if constexpr (N1 == 4) return slot(q >> 5, (q >> 3) & 3, (q >> 1) & 3) ^ (2 * (q & 1));
    else return q;
  }
  __device__ static __forceinline__ int cell(int q) { return N1 == 4 ? q >> 5 : q / NL; }
  // x-line at slot a of a buffer
  __device__ static __forceinline__ void line(const double* __restrict__ buf, int a, double (&u)[N1]) {
    if constexpr (N1 == 4) {
      const mfma_a2 v = *reinterpret_cast<const mfma_a2*>(buf + a), w = *reinterpret_cast<const mfma_a2*>(buf + (a ^ 2));
      u[0] = v.x; u[1] = v.y; u[2] = w.x; u[3] = w.y;
    } else {
      u[0] = buf[a]; u[1] = buf[a + 1]; u[2] = buf[a + 2];
    }
  }
  __device__ static __forceinline__ void put_line(double* __restrict__ buf, int a, const double (&u)[N1]) {
    if constexpr (N1 == 4) {
      *reinterpret_cast<mfma_a2*>(buf + a) = mfma_a2{u[0], u[1]};
      *reinterpret_cast<mfma_a2*>(buf + (a ^ 2)) = mfma_a2{u[2], u[3]};
    } else {
      buf[a] = u[0]; buf[a + 1] = u[1]; buf[a + 2] = u[2];
    }
  }
  __device__ static __forceinline__ void put(double* __restrict__ buf, int a, const E& v) {
    if constexpr (N1 == 4) *reinterpret_cast<mfma_a2*>(buf + a) = v;
    else buf[a] = v;
  }
  __device__ static __forceinline__ E get(const double* __restrict__ buf, int a) {
    if constexpr (N1 == 4) return *reinterpret_cast<const mfma_a2*>(buf + a);
    else return buf[a];
  }
  __device__ static __forceinline__ double dot(const E& u, const E& v) {
    if constexpr (N1 == 4) return u.x * v.x + u.y * v.y;
    else return u * v;
  }
  __device__ static __forceinline__ E load(mfma_gp base, unsigned off) {
    typedef const E __attribute__((address_space(1))) * EP;
    return *(EP)((const char __attribute__((address_space(1)))*)base + here(off));
  }
  __device__ static __forceinline__ void store(mfma_gpw base, unsigned off, const E& v) {
    typedef E __attribute__((address_space(1))) * EP;
    *(EP)((char __attribute__((address_space(1)))*)base + here(off)) = v;
  }
};

// Position in the plane of workgroup w: in memory order, or (prow > 0) in strips of kMfmaStrip workgroups
// along x, row after row. A row of workgroups is a row of cells rounded up, so that the strip drifts by
// less than a workgroup per row where 16 does not divide nx; what is left of the plane follows in order.
constexpr unsigned kMfmaStrip = 8;
__host__ __device__ __forceinline__ unsigned mfma_strip(unsigned w, unsigned prow, unsigned prows) {
  if (prow == 0 || w >= prow * prows) return w;
  const unsigned full = prow / kMfmaStrip * kMfmaStrip;
  if (w < full * prows) {
    const unsigned s = w / (kMfmaStrip * prows), r = w % (kMfmaStrip * prows);
    return r / kMfmaStrip * prow + s * kMfmaStrip + r % kMfmaStrip;
  }
  const unsigned r = w - full * prows, width = prow - full;
  return r / width * prow + full + r % width;
}

// Orders a wave's LDS writes before its later reads (the LDS serves one wave's accesses in
// order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// src of the lane `4` below (row_shr) or above (row_shl) within each row of 16 lanes, i.e.
// of the same lane of the previous / next block; old where there is none
template <int CTRL>
__device__ __forceinline__ double dpp_block(double old, double src) {
  const long long o = __double_as_longlong(old), s = __double_as_longlong(src);
  const int lo = __builtin_amdgcn_update_dpp((int)o, (int)s, CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(o >> 32), (int)(s >> 32), CTRL, 0xf, 0xf, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
constexpr int kPrevBlock = 0x114, kNextBlock = 0x104;

// src of lane 2 / 3 of the quad in lanes 0 / 1 (and 2 / 3)
__device__ __forceinline__ double dpp_upper_pair(double src) {
  const long long s = __double_as_longlong(src);
  const int lo = __builtin_amdgcn_mov_dpp((int)s, 0xee, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_mov_dpp((int)(s >> 32), 0xee, 0xf, 0xf, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// MODE 0: y = J z, 1: y += J z, 2: y = J z and partials of z . (J z), one per workgroup. With a
// second vector w (wvec), read as y is in mode 1:
// 3: y = J z and partials of w . y, 4: y = J z and partials of (w . y, y . y), 5: y += J z + w.
// (A pass of its own reads y back. 96^3 Q2: a dot 74 us, here 35 more; 64^3 Q3 lognormal residual:
// apply and axpy 154 us, mode 5 110 us, 4.9 TB/s.)
// VEL 1 (J), 2 (J^T): adds the convection terms of the velocity field at M points per direction
// (dg_velocity.hh states them). They too are 4x4x4 products: z at the points by contracting x
// in registers, z (T0 -> T1) and y; the products with b; and the tests back, y (T1 -> T0) and z.
// The traces of the y faces are gathered into one product, own lower / own upper / lower
// neighbour's / upper neighbour's along lane%4 (T1 -> lane/16 = z), interpolated, upwinded with a
// quad permutation and tested back; the z faces likewise from T0, the x faces per register.
template <int N1, int KIND, int MODE, int VEL = 0, int M = N1>
__global__ __launch_bounds__(256, (VEL ? 2 : mfma_waves<N1, KIND, MODE>())) void dg_mfma_kernel(const double* __restrict__ z, double* __restrict__ y,
                                                      const double* __restrict__ fc, const MfmaTab* __restrict__ tab,
                                                      const MfmaArgs a, unsigned nblocks, double* __restrict__ dotp,
                                                      const int* __restrict__ stop,
                                                      const double* __restrict__ wvec = nullptr) {
  // a device-side Krylov loop that has stopped: read here, obeyed once the first loads are on
  // their way (the flag and they come from beyond the L2, which other XCDs' kernels have written)
  const int stopped = stop ? *stop : 0;
  using SG = MfmaStage<N1>;
  using E = typename SG::E;
  constexpr int NL = SG::NL;
  constexpr unsigned CB = NL * sizeof(double);
  constexpr bool WT = KIND == MFMA_WEIGHT || KIND == MFMA_TENSOR;  // face weights
  constexpr bool RY = MODE == 1 || MODE == 5, RW = MODE >= 3;      // y or w is read
  constexpr bool ADD = !WT;                                        // the tables' line matrices take part
  constexpr int FW = mfma_row(KIND == MFMA_TENSOR), FK = FW - 3;
  __shared__ __attribute__((aligned(16))) double lds[4 * SG::WAVE];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i4 = lane & 3, blk = (lane >> 2) & 3, k4 = lane >> 4;
  double* const W = lds + wave * SG::WAVE;
  double *const BYL = W + 2 * SG::BUF, *const BYR = W + 3 * SG::BUF, *const BX = W + 4 * SG::BUF;
  const bool act = N1 == 4 || (i4 < N1 && k4 < N1);
  const unsigned lb = (unsigned)xcd_logical_block(blockIdx.x, nblocks);
  const unsigned gq = nblocks / (unsigned)a.zsegs, zs = lb / gq;
  const unsigned c4 = 4u * (mfma_strip(lb % gq, a.prow, a.prows) * 4u + wave);  // first cell of the group
  const unsigned cs = min(c4, a.np - 4u);  // the last group is moved back to end with the plane
  const unsigned cc = cs + blk, nx = (unsigned)a.nx;
  const bool valid = cc >= c4;  // false for cells of the previous group (and past the plane): not stored
  const unsigned gx = cc % nx;
  const bool lox = gx > 0, hix = gx < nx - 1u, loy = cc >= nx, hiy = cc + nx < a.np;
  const bool ld_xe = (blk == 0 && lox) || (blk == 3 && hix);
  // padding lanes of Q2 read the line of a neighbouring lane: their matrix rows and columns are zero
  const int p4 = N1 == 4 ? i4 : min(i4, N1 - 1), r4 = N1 == 4 ? k4 : min(k4, N1 - 1);
  const int a0 = SG::slot(blk, r4, p4), a1 = SG::slot(blk, p4, r4);             // T0, T1
  const int ax = SG::slot(blk == 0 ? 0 : 1, p4, r4);                             // T1 in the end cells
  // staged elements: slots and byte offsets within a plane (below 4 GiB); where a neighbour does
  // not exist the own element is read (and the value dropped below)
  const bool two = N1 == 4 || lane < SG::NE - 64, ldx = N1 == 4 || lane < SG::NX;
  int se[2];
  unsigned ow[2], oyl[2], oyr[2];
  bool st[2];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int q = min(lane + 64 * p, SG::NE - 1);
    const unsigned c = cs + SG::cell(q);
    se[p] = SG::eslot(q);
    ow[p] = cs * CB + q * SG::ES;
    oyl[p] = ow[p] - (c >= nx ? nx * CB : 0u);
    oyr[p] = ow[p] + (c + nx < a.np ? nx * CB : 0u);
    st[p] = c >= c4;
  }
  int sx;
  unsigned ox;
  {
    const int q = min(lane, SG::NX - 1), e = SG::cell(q), r = q - e * (SG::NX / 2);
    sx = SG::eslot(q);
    const unsigned c = e == 0 ? (cs > 0 ? cs - 1u : 0u) : min(cs + 4u, a.np - 1u);
    ox = c * CB + r * SG::ES;
  }
  const size_t plane = (size_t)a.np * NL;
  const int k0 = (int)zs * a.zw, k1 = min(k0 + a.zw, a.nz);
  const int me = 4 * i4 + k4;
  const double Mm = tab->M[me];
  double Ly = 0, Nyl = 0, Nyr = 0, Lzi = 0, Nzl = 0, Nzr = 0;
  double wK = 0, wWL = 0, wWU = 0, wNL = 0, wNU = 0, wKy = 0, bzl = 0, bzu = 0;
  if constexpr (ADD) {
    Ly = tab->own[0][me];
    if (!loy) Ly += tab->dlo[0][me];
    if (!hiy) Ly += tab->dhi[0][me];
    Nyl = loy ? tab->nlo[0][me] : 0.0;
    Nyr = hiy ? tab->nhi[0][me] : 0.0;
    Lzi = tab->own[1][me];
    Nzl = tab->nlo[1][me];
    Nzr = tab->nhi[1][me];
  }
  if constexpr (WT) {
    wK = tab->K[me];
    wWL = tab->WL[me];
    wWU = tab->WU[me];
    wNL = tab->NL[me];
    wNU = tab->NU[me];
    wKy = wK;  // with the boundary faces of the cell's row, which scale with kappa too
    if (!loy) wKy += tab->BL[0][me];
    if (!hiy) wKy += tab->BU[0][me];
  }
  // corrections of the own z matrix at the ends of the column
  if (k0 == 0) bzl = WT ? tab->BL[1][me] : tab->dlo[1][me];
  if (k1 == a.nz) bzu = WT ? tab->BU[1][me] : tab->dhi[1][me];
  // MFMA_GENERAL: coefficients of a face: own side's weight, neighbour's weight, penalty; a
  // Dirichlet boundary face has own weight kappa, penalty alphak kappa and no neighbour
  struct Face {
    double wo, wn, P;
  };
  auto lower = [&](const double* f, int d, bool has, double k, Face& F) {
    F.wn = has ? f[FCF + 3 * d] : 0.0;
    F.wo = has ? f[FCF + 3 * d + 1] : 0.0;
    F.P = has ? f[FCF + 3 * d + 2] : 0.0;
    if (!has && a.bc[2 * d] == BC_DIRICHLET) {
      F.wo = k;
      F.P = a.alphak * (a.weightsOn ? k : 1.0);
    }
  };
  auto upper = [&](const double* f, int d, bool has, size_t stride, double k, Face& F) {
    const double* fn = f + (has ? stride * FC : 0);
    F.wo = has ? fn[FCF + 3 * d] : 0.0;
    F.wn = has ? fn[FCF + 3 * d + 1] : 0.0;
    F.P = has ? fn[FCF + 3 * d + 2] : 0.0;
    if (!has && a.bc[2 * d + 1] == BC_DIRICHLET) {
      F.wo = k;
      F.P = a.alphak * (a.weightsOn ? k : 1.0);
    }
  };
  // lane matrices of a direction: own, lower and upper neighbour
  auto mats = [&](double S, double k, const Face& l, const Face& u, double& Lm, double& Nl, double& Nr) {
    Lm = S * (k * tab->K[me] + l.wo * tab->U[0][me] + l.P * tab->U[1][me] + u.P * tab->U[2][me] - u.wo * tab->U[3][me]);
    Nl = S * (l.wn * tab->X[0][me] + l.P * tab->X[1][me] + l.wo * tab->X[2][me]);
    Nr = S * (u.P * tab->X[3][me] + u.wn * tab->X[4][me] + u.wo * tab->X[5][me]);
  };
  // the lower z-neighbour's matrix at step kz > 0
  auto lower_z = [&](int kz) {
    const double* f = fc + ((size_t)kz * a.np + cc) * FC + FCF + 6;
    return a.S[2] * (f[0] * tab->X[0][me] + f[2] * tab->X[1][me] + f[1] * tab->X[2][me]) + Nzl;
  };
  // in flight for the next step: elements of the next plane, the y-neighbours and the end cells,
  // of y and w, and the face weights. They are issued in one batch and waited for together:
  // loads complete in order, so a load issued later would have to wait for these.
  E rn[2], rl[2], rr[2], rx, ry[2], rw[2];
  double fk[3] = {0, 0, 0}, fx = 0, fy = 0, fxu = 0, fyu = 0, fzu = 0;
  auto fetch = [&](const double* base, const unsigned (&o)[2], E (&v)[2]) {
    const mfma_gp b = per_step<mfma_gp>(base);
    v[0] = SG::load(b, o[0]);
    if (two) v[1] = SG::load(b, o[1]);
  };
  auto fetch_step = [&](int kz) {
    const double* zk = z + (size_t)kz * plane;
    fetch(zk + (kz + 1 < a.nz ? plane : 0), ow, rn);  // at the top the own cells (their matrix is zero)
    fetch(zk, oyl, rl);
    fetch(zk, oyr, rr);
    if (ldx) rx = SG::load(per_step<mfma_gp>(zk), ox);
    if constexpr (RY) fetch(y + (size_t)kz * plane, ow, ry);
    if constexpr (RW) fetch(wvec + (size_t)kz * plane, ow, rw);
    if constexpr (WT) {
      const mfma_gp f = per_step<mfma_gp>(fc + (size_t)kz * a.np * FW);
      const unsigned of = cc * (unsigned)(FW * 8);
      auto at = [&](mfma_gp q, unsigned o) { return *(mfma_gp)((const char __attribute__((address_space(1)))*)q + here(o)); };
#pragma unroll
      for (int d = 0; d < 3; ++d) fk[d] = d < FK ? at(f, of + 8 * d) : fk[0];
      fx = at(f, of + 8 * FK);
      fy = at(f, of + 8 * FK + 8);
      fxu = at(f, of + (hix ? FW * 8 : 0u) + 8 * FK);
      fyu = at(f, of + (hiy ? nx * (FW * 8) : 0u) + 8 * FK + 8);
      fzu = at(kz + 1 < a.nz ? f + (size_t)a.np * FW : f, of + 8 * FK + 16);
    }
  };
  auto put = [&](double* buf, const E (&v)[2]) {
    SG::put(buf, se[0], v[0]);
    if (two) SG::put(buf, se[1], v[1]);
  };
  // ---- velocity field
  constexpr int M2 = M * M, M3 = M2 * M, VM = VEL ? M : 1, VN = VEL ? N1 : 1;
  double LB = 0, LD = 0, WB = 0, WDy = 0, WDz = 0, Po = 0, Pl = 0, Pu = 0, Eo = 0, say = 0, saz = 0;
  double b0[VM], b1[VM], b2[VM], by[VM], bz[VM], bxl = 0, bxu = 0;  // the field at this step's points
  double tz[VN];  // the lower z-neighbour's trace part
  unsigned ov = 0, ofx = 0, ofy = 0;
  bool outy = false;
  // boundary sides with a convection term
  auto takes = [&](int side) -> int { return int(a.bc[side] == BC_DIRICHLET) | int(a.bc[side] == BC_OUTFLOW); };
  if constexpr (VEL != 0) {
    LB = a.vt->LB[me];
    WB = a.vt->WB[me];
    if constexpr (VEL == 1) {
      WDy = a.vt->WDy[me];
      WDz = a.vt->WDz[me];
    } else {
      LD = a.vt->LD[me];
    }
    // gather: own lower, own upper, lower neighbour's, upper neighbour's trace; scatter: its transpose
    Po = (i4 == 0 && k4 == 0) || (i4 == 1 && k4 == N1 - 1) ? 1.0 : 0.0;
    Pl = i4 == 2 && k4 == N1 - 1 ? 1.0 : 0.0;
    Pu = i4 == 3 && k4 == 0 ? 1.0 : 0.0;
    Eo = (i4 == 0 && k4 == 0) || (i4 == N1 - 1 && k4 == 1) ? 1.0 : 0.0;
    // signed face areas of the lane's y and z face (lower, upper); zero where the face has no term
    // (here and below as selects: hipcc 7.2 dropped the assignment of nested short-circuit branches)
    const bool lo = i4 == 0, up = i4 == 1;
    const double sl = (int(loy) | takes(2)) ? -a.area[1] : 0.0, su = (int(hiy) | takes(3)) ? a.area[1] : 0.0;
    say = lo ? sl : (up ? su : 0.0);
    outy = (lo ? int(!loy) & int(a.bc[2] == BC_OUTFLOW) : up ? int(!hiy) & int(a.bc[3] == BC_OUTFLOW) : 0) != 0;
    saz = i4 == 0 ? -a.area[2] : (i4 == 1 ? a.area[2] : 0.0);
    const int qi = min(i4, M - 1), qk = min(k4, M - 1);
    ov = (cc * (3 * M3) + M * (qk + M * qi)) * 8u;              // volume, T1: lane%4 = z point, lane/16 = y point
    ofx = (cc * (6 * M2) + qi + M * qk) * 8u;                   // x faces, T0: lane%4 = y point, lane/16 = z point
    ofy = (cc * (6 * M2) + (2 + (i4 & 1)) * M2 + M * qk) * 8u;  // y faces: lane%4 = side; the z faces 2 M2 further
  }
  auto load_field = [&](int kz) {
    if constexpr (VEL != 0) {
      const mfma_gp bv = per_step<mfma_gp>(a.bv + (size_t)kz * a.np * (3 * M3));
      const mfma_gp bf = per_step<mfma_gp>(a.bf + (size_t)kz * a.np * (6 * M2));
      auto row = [&](mfma_gp base, unsigned off, double (&v)[VM]) {
        const mfma_gp q = (mfma_gp)((const char __attribute__((address_space(1)))*)base + here(off));
#pragma unroll
        for (int e = 0; e < M; ++e) v[e] = q[e];
      };
      row(bv, ov, b0);
      row(bv, ov + M3 * 8, b1);
      row(bv, ov + 2 * M3 * 8, b2);
      row(bf, ofy, by);
      row(bf, ofy + 2 * M2 * 8, bz);
      const mfma_gp q = (mfma_gp)((const char __attribute__((address_space(1)))*)bf + here(ofx));
      bxl = q[0];
      bxu = q[M2];
    }
  };
  // upwinded flux of a face point: sa the signed area (the weights come with the test)
  auto flux = [&](double own, double nb, double b, double sa, bool out) {
    const double cf = sa * b;
    const bool in = (int(out) | int(cf >= 0.0)) != 0;
    if constexpr (VEL == 2) return in ? cf * (out ? own : own - nb) : 0.0;
    return cf * (in ? own : nb);
  };
  // o (T0) += the convection terms of the step's cells: own lines uz (T0) and u (T1), the upper
  // plane's zr (T0), the x-neighbours' traces vl, vr (T1)
  auto convect = [&](int kz, const double (&uz)[N1], const double (&zr)[N1], const double (&u)[N1], double vl, double vr,
                     double (&o)[N1]) {
    if constexpr (VEL != 0) {
      typedef const MfmaVelTab __attribute__((address_space(4))) * tp;
      const bool loz = kz > 0, hiz = kz < a.nz - 1;
      // x faces
      {
        const double ol = mfma4(LB, mfma4(u[0], LB, 0.0), 0.0), ou = mfma4(LB, mfma4(u[N1 - 1], LB, 0.0), 0.0);
        const double nl = mfma4(LB, mfma4(vl, LB, 0.0), 0.0), nu = mfma4(LB, mfma4(vr, LB, 0.0), 0.0);
        const double sl = (int(lox) | takes(0)) ? -a.area[0] : 0.0, su = (int(hix) | takes(1)) ? a.area[0] : 0.0;
        const double fl = flux(ol, nl, bxl, sl, (int(!lox) & int(a.bc[0] == BC_OUTFLOW)) != 0);
        const double fu = flux(ou, nu, bxu, su, (int(!hix) & int(a.bc[1] == BC_OUTFLOW)) != 0);
        o[0] = mfma4(mfma4(fl, WB, 0.0), WB, o[0]);
        o[N1 - 1] = mfma4(mfma4(fu, WB, 0.0), WB, o[N1 - 1]);
      }
      // gathered traces t[x] (lane%4 = side, lane/16 = the other direction): the points, the flux,
      // the test along x and that direction; returns g[x] (lane%4 = the other direction, lane/16 = side)
      auto face = [&](const double (&t)[N1], const double (&b)[VM], double sa, bool out, double (&g)[N1]) {
        const tp v = per_step<tp>(a.vt);
        double f[VM];
#pragma unroll
        for (int q = 0; q < M; ++q) {
          double w = 0;
#pragma unroll
          for (int e = 0; e < N1; ++e) w += v->B[q][e] * t[e];
          w = mfma4(LB, w, 0.0);
          f[q] = flux(w, dpp_upper_pair(w), b[q], sa, out);
        }
#pragma unroll
        for (int e = 0; e < N1; ++e) {
          double w = 0;
#pragma unroll
          for (int q = 0; q < M; ++q) w += v->BW[q][e] * f[q];
          g[e] = mfma4(w, WB, 0.0);
        }
      };
      {
        double t[N1], g[N1], n[N1];
        SG::line(BYL, a1, n);
#pragma unroll
        for (int e = 0; e < N1; ++e) t[e] = mfma4(n[e], loy ? Pl : 0.0, mfma4(u[e], Po, 0.0));
        SG::line(BYR, a1, n);
#pragma unroll
        for (int e = 0; e < N1; ++e) t[e] = mfma4(n[e], hiy ? Pu : 0.0, t[e]);
        face(t, by, say, outy, g);
#pragma unroll
        for (int e = 0; e < N1; ++e) o[e] = mfma4(g[e], Eo, o[e]);
      }
      {
        double t[N1], g[N1];
        const double pu = hiz ? Pu : 0.0;
#pragma unroll
        for (int e = 0; e < N1; ++e) {
          t[e] = mfma4(zr[e], pu, mfma4(uz[e], Po, tz[e]));
          tz[e] = mfma4(uz[e], Pl, 0.0);
        }
        const int lo = int(i4 == 0) & int(!loz), up = int(i4 == 1) & int(!hiz);
        const double sa = (lo & (1 - takes(4))) | (up & (1 - takes(5))) ? 0.0 : saz;
        const bool out = ((lo & int(a.bc[4] == BC_OUTFLOW)) | (up & int(a.bc[5] == BC_OUTFLOW))) != 0;
        face(t, bz, sa, out, g);
#pragma unroll
        for (int e = 0; e < N1; ++e) o[e] = mfma4(Eo, g[e], o[e]);
      }
      // volume
      const tp v = per_step<tp>(a.vt);
      if constexpr (VEL == 1) {
        double p0[VM], p1[VM], p2[VM];
#pragma unroll
        for (int q = 0; q < M; ++q) {
          double w = 0;
#pragma unroll
          for (int e = 0; e < N1; ++e) w += v->B[q][e] * uz[e];
          w = mfma4(LB, mfma4(w, LB, 0.0), 0.0);
          p0[q] = b0[q] * w;
          p1[q] = b1[q] * w;
          p2[q] = b2[q] * w;
        }
        const tp r = per_step<tp>(a.vt);
#pragma unroll
        for (int e = 0; e < N1; ++e) {
          double w0 = 0, w1 = 0, w2 = 0;
#pragma unroll
          for (int q = 0; q < M; ++q) {
            w0 += r->DW[q][e] * p0[q];
            w1 += r->BW[q][e] * p1[q];
            w2 += r->BW[q][e] * p2[q];
          }
          const double tB = mfma4(w1, WDy, mfma4(w0, WB, 0.0)), tD = mfma4(w2, WB, 0.0);
          o[e] = mfma4(WDz, tD, mfma4(WB, tB, o[e]));
        }
      } else {
        double p[VM];
#pragma unroll
        for (int q = 0; q < M; ++q) {
          double w = 0, d = 0;
#pragma unroll
          for (int e = 0; e < N1; ++e) {
            w += v->B[q][e] * uz[e];
            d += v->D[q][e] * uz[e];
          }
          const double zB = mfma4(w, LB, 0.0);
          const double gx = mfma4(LB, mfma4(d, LB, 0.0), 0.0), gy = mfma4(LD, zB, 0.0);
          const double gz = mfma4(LB, mfma4(w, LD, 0.0), 0.0);
          p[q] = a.vs[0] * b0[q] * gx + a.vs[1] * b1[q] * gy + a.vs[2] * b2[q] * gz;
        }
        const tp r = per_step<tp>(a.vt);
#pragma unroll
        for (int e = 0; e < N1; ++e) {
          double w = 0;
#pragma unroll
          for (int q = 0; q < M; ++q) w += r->BW[q][e] * p[q];
          o[e] = mfma4(WB, mfma4(w, WB, 0.0), o[e]);
        }
      }
    }
  };
  double ua[N1], ub[N1], sn[N1];  // own T0 lines of even / odd steps, lower z-neighbour's part of s
  double wz = 0;                  // face weights: that of the lower z face
  {
    E r0[2], rz[2];
    fetch(z + (size_t)k0 * plane, ow, r0);
    if (k0 > 0) fetch(z + (size_t)(k0 - 1) * plane, ow, rz);
    if constexpr (WT) wz = fc[((size_t)k0 * a.np + cc) * FW + FK + 2];
    fetch_step(k0);
    if (stopped) return;
    put(W, r0);
    if (k0 > 0) put(BYL, rz);
  }
  wave_lds_fence();
  SG::line(W, a0, ua);
#pragma unroll
  for (int e = 0; e < N1; ++e) sn[e] = 0;
  if constexpr (VEL != 0) {
#pragma unroll
    for (int e = 0; e < N1; ++e) tz[e] = 0;
  }
  if (k0 > 0) {
    double zl[N1], Nl = Nzl;
    SG::line(BYL, a0, zl);
    if constexpr (WT) Nl = a.S[2] * wz * wNL;
    if constexpr (KIND == MFMA_GENERAL) Nl = lower_z(k0);
#pragma unroll
    for (int e = 0; e < N1; ++e) sn[e] = mfma4(zl[e], Nl, 0.0);
    if constexpr (VEL != 0) {
#pragma unroll
      for (int e = 0; e < N1; ++e) tz[e] = mfma4(zl[e], Pl, 0.0);
    }
  }
  // entry (i, j) of a centro-symmetric matrix, read at the lexicographically first position
  auto centro = [](const double(&m)[4][4], int i, int j) {
    const bool keep = i * N1 + j <= (N1 - 1 - i) * N1 + (N1 - 1 - j);
    return m[keep ? i : N1 - 1 - i][keep ? j : N1 - 1 - j];
  };
  double pq = 0, qq = 0;  // this lane's shares of the dots
  // one z-step: own cells in B0 (T0 lines uz), the next plane's to B1 (T0 lines zr)
  auto step = [&](int kz, double* B0, double* B1, double (&uz)[N1], double (&zr)[N1]) {
    const bool loz = kz > 0, hiz = kz < a.nz - 1;
    load_field(kz);  // older than the next step's loads: waited for without them
    wave_lds_fence();
    put(B1, rn);
    put(BYL, rl);
    put(BYR, rr);
    if (ldx) SG::put(BX, sx, rx);
    const double kx = fk[0], ky = fk[1], kz_ = fk[2], wxl = fx, wyl = fy, wxu = hix ? fxu : 0.0, wyu = hiy ? fyu : 0.0, wzu = hiz ? fzu : 0.0;
    E yo[2], wo[2];
    if constexpr (RY) {
      yo[0] = ry[0];
      yo[1] = ry[1];
    }
    if constexpr (MODE == 5) {
      yo[0] += rw[0];
      if (two) yo[1] += rw[1];
    } else if constexpr (RW) {
      wo[0] = rw[0];
      wo[1] = rw[1];
    }
    if (kz + 1 < k1) fetch_step(kz + 1);
    wave_lds_fence();
    double u[N1], yn[N1], s[N1];
    SG::line(B1, a0, zr);
    SG::line(B0, a1, u);
    if constexpr (KIND == MFMA_CONST || KIND == MFMA_CONV) {
      double Lz = Lzi;
      if (!loz) Lz += bzl;
      if (!hiz) Lz += bzu;
      const double Nr = hiz ? Nzr : 0.0;
      double w[N1];  // the y direction is summed by itself
#pragma unroll
      for (int e = 0; e < N1; ++e) s[e] = mfma4(uz[e], Lz, sn[e]);
#pragma unroll
      for (int e = 0; e < N1; ++e) sn[e] = mfma4(uz[e], Nzl, 0.0);
#pragma unroll
      for (int e = 0; e < N1; ++e) s[e] = mfma4(zr[e], Nr, s[e]);
#pragma unroll
      for (int e = 0; e < N1; ++e) w[e] = mfma4(Ly, u[e], 0.0);
      SG::line(BYL, a1, yn);
#pragma unroll
      for (int e = 0; e < N1; ++e) w[e] = mfma4(Nyl, yn[e], w[e]);
      SG::line(BYR, a1, yn);
#pragma unroll
      for (int e = 0; e < N1; ++e) s[e] += mfma4(Nyr, yn[e], w[e]);
    }
    if constexpr (WT) {
      const double sy = a.S[1], sz = a.S[2];
      const double zk_ = sz * kz_, zwu = sz * wzu;
      double Lm = zk_ * wK + (sz * wz) * wWL + zwu * wWU;
      if (!loz) Lm += zk_ * bzl;
      if (!hiz) Lm += zk_ * bzu;
      const double Nr = zwu * wNU, Nn = zwu * wNL;
#pragma unroll
      for (int e = 0; e < N1; ++e) s[e] = mfma4(uz[e], Lm, sn[e]);
#pragma unroll
      for (int e = 0; e < N1; ++e) sn[e] = mfma4(uz[e], Nn, 0.0);
#pragma unroll
      for (int e = 0; e < N1; ++e) s[e] = mfma4(zr[e], Nr, s[e]);
      const double yk = sy * ky, yw = sy * wyl, ywu = sy * wyu;
      Lm = yk * wKy + yw * wWL + ywu * wWU;
#pragma unroll
      for (int e = 0; e < N1; ++e) s[e] = mfma4(Lm, u[e], s[e]);
      SG::line(BYL, a1, yn);
      const double Nl = yw * wNL, Nu = ywu * wNU;
#pragma unroll
      for (int e = 0; e < N1; ++e) s[e] = mfma4(Nl, yn[e], s[e]);
      SG::line(BYR, a1, yn);
#pragma unroll
      for (int e = 0; e < N1; ++e) s[e] = mfma4(Nu, yn[e], s[e]);
      wz = wzu;
    }
    double kg = 0, xwl = 0, xwh = 0, xP = 0, ywl = 0, ywh = 0, yP = 0;  // x faces: lower (whi, P, wlo), upper
    if constexpr (KIND == MFMA_GENERAL) {
      const double* f = fc + ((size_t)kz * a.np + cc) * FC;
      Face lo, up;
      double Lm, Nl, Nr;
      lower(f, 2, loz, f[2], lo);
      upper(f, 2, hiz, a.np, f[2], up);
      mats(a.S[2], f[2], lo, up, Lm, Nl, Nr);
      Lm += Lzi + (loz ? 0.0 : bzl) + (hiz ? 0.0 : bzu);
      Nr = hiz ? Nr + Nzr : 0.0;
      const double Nn = hiz ? lower_z(kz + 1) : 0.0;
#pragma unroll
      for (int e = 0; e < N1; ++e) {
        s[e] = mfma4(uz[e], Lm, sn[e]);
        sn[e] = mfma4(uz[e], Nn, 0.0);
        s[e] = mfma4(zr[e], Nr, s[e]);
      }
      lower(f, 1, loy, f[1], lo);
      upper(f, 1, hiy, a.nx, f[1], up);
      mats(a.S[1], f[1], lo, up, Lm, Nl, Nr);
      Lm += Ly;
      Nl = loy ? Nl + Nyl : 0.0;
      Nr = hiy ? Nr + Nyr : 0.0;
#pragma unroll
      for (int e = 0; e < N1; ++e) s[e] = mfma4(Lm, u[e], s[e]);
      SG::line(BYL, a1, yn);
#pragma unroll
      for (int e = 0; e < N1; ++e) s[e] = mfma4(Nl, yn[e], s[e]);
      SG::line(BYR, a1, yn);
#pragma unroll
      for (int e = 0; e < N1; ++e) s[e] = mfma4(Nr, yn[e], s[e]);
      kg = f[0];
      lower(f, 0, lox, kg, lo);
      upper(f, 0, hix, 1, kg, up);
      xwh = lo.wo;
      xwl = lo.wn;
      xP = lo.P;
      ywl = up.wo;
      ywh = up.wn;
      yP = up.P;
    }
    // x-lines: trace and derivative of the neighbours, those of the wave's ends from xe
    const MfmaX& X = a.x;
    double der0 = 0, der1 = 0, ed = 0, ev = 0;
#pragma unroll
    for (int e = 0; e < N1; ++e) {
      der0 -= X.d1[N1 - 1 - e] * u[e];
      der1 += X.d1[e] * u[e];
    }
    if (ld_xe) {
      double e0 = 0, e1 = 0, xe[N1];
      SG::line(BX, ax, xe);
#pragma unroll
      for (int e = 0; e < N1; ++e) {
        e0 -= X.d1[N1 - 1 - e] * xe[e];
        e1 += X.d1[e] * xe[e];
      }
      ed = blk == 0 ? e1 : e0;
      ev = blk == 0 ? xe[N1 - 1] : xe[0];
    }
    double vl = dpp_block<kPrevBlock>(ev, u[N1 - 1]), dl = dpp_block<kPrevBlock>(ed, der1);
    double vr = dpp_block<kNextBlock>(ev, u[0]), dr = dpp_block<kNextBlock>(ed, der0);
    // row ends: no neighbour, boundary corrections
    double bl0 = 0, bl1 = 0, bu0 = 0, bu1 = 0;  // face weights: boundary parts of ce0, cd0, ce1, cd1
    if (!lox) {
      vl = dl = 0;
      if constexpr (ADD) {
        const mfma_tp t = per_step<mfma_tp>(tab);
#pragma unroll
        for (int i = 0; i < N1; ++i)
#pragma unroll
          for (int j = 0; j < N1; ++j) s[i] += t->Dlo[i][j] * u[j];
      } else if (a.bc[0] == BC_DIRICHLET) {
        bl0 = a.S[0] * kx * (a.fg * der0 + a.alphak * u[0]);
        bl1 = -a.S[0] * kx * a.fh * u[0];
      }
    }
    if (!hix) {
      vr = dr = 0;
      if constexpr (ADD) {
        const mfma_tp t = per_step<mfma_tp>(tab);
#pragma unroll
        for (int i = 0; i < N1; ++i)
#pragma unroll
          for (int j = 0; j < N1; ++j) s[i] += t->Dhi[i][j] * u[j];
      } else if (a.bc[1] == BC_DIRICHLET) {
        bu0 = a.S[0] * kx * (a.alphak * u[N1 - 1] - a.fg * der1);
        bu1 = a.S[0] * kx * a.fh * u[N1 - 1];
      }
    }
    if constexpr (WT || KIND == MFMA_GENERAL) {
      double sk, ce0, cd0, ce1, cd1;
      if constexpr (WT) {
        const double Sx = a.S[0], sw = Sx * wxl, su = Sx * wxu, p2 = 2.0 * a.alphak;
        const double J0 = vl - u[0], J1 = u[N1 - 1] - vr;
        sk = Sx * kx;
        ce0 = sw * (a.fg * (dl + der0) - p2 * J0) + bl0;
        cd0 = sw * a.fh * J0 + bl1;
        ce1 = su * (p2 * J1 - a.fg * (der1 + dr)) + bu0;
        cd1 = su * a.fh * J1 + bu1;
      } else {
        const double J0 = vl - u[0], G0 = xwl * dl + xwh * der0;
        const double J1 = u[N1 - 1] - vr, G1 = ywl * der1 + ywh * dr;
        const double Sx = a.S[0];
        sk = Sx * kg;
        ce0 = Sx * (a.fg * G0 - xP * J0);
        cd0 = Sx * a.fh * xwh * J0;
        ce1 = Sx * (yP * J1 - a.fg * G1);
        cd1 = Sx * a.fh * ywl * J1;
      }
#pragma unroll
      for (int i = 0; i < N1; ++i) {
        double kv = 0;
#pragma unroll
        for (int j = 0; j < N1; ++j) kv += centro(X.A, i, j) * u[j];
        s[i] += sk * kv + ce0 * X.P[i] + cd0 * X.Q[i] + ce1 * X.P[N1 - 1 - i] - cd1 * X.Q[N1 - 1 - i] + a.vc * u[i];
      }
    }
    if constexpr (KIND == MFMA_CONST) {
#pragma unroll
      for (int i = 0; i < N1; ++i) {
#pragma unroll
        for (int j = 0; j < N1; ++j) s[i] += centro(X.A, i, j) * u[j];
        s[i] += X.P[i] * vl;
        s[i] += X.Q[i] * dl;
        s[i] += X.P[N1 - 1 - i] * vr;
        s[i] -= X.Q[N1 - 1 - i] * dr;
      }
    }
    if constexpr (KIND == MFMA_CONV || KIND == MFMA_GENERAL) {
      const mfma_tp t = per_step<mfma_tp>(tab);
#pragma unroll
      for (int i = 0; i < N1; ++i) {
        if constexpr (KIND == MFMA_CONV) s[i] += a.vc * u[i];
#pragma unroll
        for (int j = 0; j < N1; ++j) s[i] += t->A[i][j] * u[j];
        s[i] += t->Pl[i] * vl;
        s[i] += t->Ql[i] * dl;
        s[i] += t->Pr[i] * vr;
        s[i] += t->Qr[i] * dr;
      }
    }
    // mass: x in registers, y (T1 -> T0), z
    double o[N1];
#pragma unroll
    for (int i = 0; i < N1; ++i) {
      double v = 0;
#pragma unroll
      for (int j = 0; j < N1; ++j) v += X.M[mass_canon<N1>(i, j) / N1][mass_canon<N1>(i, j) % N1] * s[j];
      o[i] = mfma4(v, Mm, 0.0);
    }
#pragma unroll
    for (int i = 0; i < N1; ++i) o[i] = mfma4(Mm, o[i], 0.0);
    convect(kz, uz, zr, u, vl, vr, o);
    if constexpr (MODE == 2) {  // the own lines again, from LDS: held through the step they would spill
      double v[N1];
      SG::line(B0, a0, v);
      if (act && valid) {
#pragma unroll
        for (int i = 0; i < N1; ++i) pq += v[i] * o[i];
      }
    }
    // back to memory order through the lower y-neighbours' buffer (read above)
    wave_lds_fence();
    if (act) SG::put_line(BYL, a0, o);
    wave_lds_fence();
    {
      const mfma_gpw yc = per_step<mfma_gpw>(y + (size_t)kz * plane);
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        if ((p == 0 || two) && st[p]) {
          E v = SG::get(BYL, se[p]);
          if constexpr (MODE == 3 || MODE == 4) pq += SG::dot(wo[p], v);
          if constexpr (MODE == 4) qq += SG::dot(v, v);
          if constexpr (RY) v += yo[p];
          SG::store(yc, ow[p], v);
        }
      }
    }
  };
  double* const W1 = W + SG::BUF;
  int kz = k0;
  for (; kz + 1 < k1; kz += 2) {
    step(kz, W, W1, ua, ub);
    step(kz + 1, W1, W, ub, ua);
  }
  if (kz < k1) step(kz, W, W1, ua, ub);
  if constexpr (MODE == 2 || MODE == 3) {
    double v[1] = {pq};
    block_sum_reuse<4, double, 1>(v, lds);
    if (threadIdx.x == 0) dotp[blockIdx.x] = v[0];
  }
  if constexpr (MODE == 4) {
    double v[2] = {pq, qq};
    block_sum_reuse<4, double, 2>(v, lds);
    if (threadIdx.x == 0) {
      dotp[2 * blockIdx.x] = v[0];
      dotp[2 * blockIdx.x + 1] = v[1];
    }
  }
}

}  // namespace pdelab_amd

#endif
