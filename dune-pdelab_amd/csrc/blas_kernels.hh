// blas_kernels.hh -- vector backend kernels (ISTL::BlockVector dot / two_norm / axpy,
// R:dune/pdelab/backend/istl/vector.hh:249-282) and the fused Krylov updates.
//
// Reductions are deterministic: a fixed grid of kRedBlocks blocks walks the vector
// with a fixed stride, each block reduces in a fixed tree (wave64 shuffles, then LDS)
// and one block sums the per-block partials in order. Results are therefore
// bitwise reproducible run to run.
#ifndef PDELAB_BLAS_KERNELS_HH
#define PDELAB_BLAS_KERNELS_HH

#include <hip/hip_runtime.h>

#include "block_reduce.hh"
#include "stream_io.hh"

namespace pdelab_amd {

// Block-wide sum of NR accumulators; result valid in thread 0.
template <typename A, int NR>
__device__ __forceinline__ void block_sum(A (&v)[NR]) {
  __shared__ A red[NR][kRedThreads / 64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < NR; ++j) {
    v[j] = wave_sum(v[j]);
    if (lane == 0) red[j][wid] = v[j];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int j = 0; j < NR; ++j) {
      A s = red[j][0];
      for (int w = 1; w < kRedThreads / 64; ++w) s += red[j][w];
      v[j] = s;
    }
  }
}

// Elements in flight per thread and stream of the reducing vector kernels: with one, the 1024
// workgroups cannot cover the memory latency (x.y of 23.9M floats, 191 MB: 51 us, with four 29 us,
// 6.5 TB/s).
constexpr int kVecUnroll = 4;

// partial[b] = block b's share of x.y, or partial[2 b + j] its shares of (x.y, y.y) (NR = 2)
template <typename T, typename A, int NR>
__global__ __launch_bounds__(kRedThreads) void dot_partial_kernel(const T* __restrict__ x, const T* __restrict__ y,
                                                                  long long n, A* __restrict__ partial) {
  A v[NR];
#pragma unroll
  for (int j = 0; j < NR; ++j) v[j] = A(0);
  constexpr long long S = (long long)kRedBlocks * kRedThreads;
  for (long long i0 = (long long)blockIdx.x * kRedThreads + threadIdx.x; i0 < n; i0 += kVecUnroll * S) {
    T xv[kVecUnroll], yv[kVecUnroll];
#pragma unroll
    for (int u = 0; u < kVecUnroll; ++u) {
      const long long i = i0 + u * S;
      xv[u] = yv[u] = T(0);
      if (i < n) {
        xv[u] = x[i];
        yv[u] = y[i];
      }
    }
#pragma unroll
    for (int u = 0; u < kVecUnroll; ++u) {
      v[0] += (A)xv[u] * (A)yv[u];
      if constexpr (NR == 2) v[1] += (A)yv[u] * (A)yv[u];
    }
  }
  block_sum<A, NR>(v);
  if (threadIdx.x == 0)
#pragma unroll
    for (int j = 0; j < NR; ++j) partial[NR * blockIdx.x + j] = v[j];
}

// Single-workgroup sums of per-workgroup partials (up to tens of thousands of them):
// kFinalThreads threads, each with four independent accumulators so that four loads
// per thread are in flight, then the workgroup tree. The order is fixed.
constexpr int kFinalThreads = 1024;

template <typename A, int NR>
__device__ __forceinline__ void strided_partial_sum(const A* __restrict__ partial, int nb, A (&v)[NR]) {
  A a[4][NR];
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int j = 0; j < NR; ++j) a[u][j] = A(0);
  int b = threadIdx.x;
  for (; b + 3 * kFinalThreads < nb; b += 4 * kFinalThreads)
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int j = 0; j < NR; ++j) a[u][j] += partial[(b + u * kFinalThreads) * NR + j];
  for (; b < nb; b += kFinalThreads)
#pragma unroll
    for (int j = 0; j < NR; ++j) a[0][j] += partial[b * NR + j];
#pragma unroll
  for (int j = 0; j < NR; ++j) v[j] = (a[0][j] + a[1][j]) + (a[2][j] + a[3][j]);
  block_sum_n<kFinalThreads, A, NR>(v);
}

// out[j] = sum_b partial[b*NR + j]   (one workgroup of kFinalThreads threads)
template <typename A, int NR>
__global__ __launch_bounds__(kFinalThreads) void final_reduce_kernel(const A* __restrict__ partial, int nb,
                                                                     A* __restrict__ out,
                                                                     const int* __restrict__ stop) {
  if (stop && *stop) return;  // a device-side Krylov loop has already stopped
  A v[NR];
  strided_partial_sum<A, NR>(partial, nb, v);
  if (threadIdx.x == 0)
#pragma unroll
    for (int j = 0; j < NR; ++j) out[j] = v[j];
}

template <typename T>
__global__ __launch_bounds__(256) void axpy_kernel(long long n, T a, const T* __restrict__ x, T* __restrict__ y) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    y[i] += a * x[i];
}

template <typename T>
__global__ __launch_bounds__(256) void scale_kernel(long long n, T a, T* __restrict__ x) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    x[i] *= a;
}

template <typename T>
__global__ __launch_bounds__(256) void fill_kernel(long long n, T a, T* __restrict__ x) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    x[i] = a;
}

template <typename S, typename D>
__global__ __launch_bounds__(256) void convert_kernel(long long n, const S* __restrict__ x, D* __restrict__ y) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    y[i] = (D)x[i];
}

// x -= (double) z32   (refinement update)
__global__ __launch_bounds__(256) void sub_f32_kernel(long long n, const float* __restrict__ z, double* __restrict__ x) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    x[i] -= (double)z[i];
}

// y32 = (float)(s x64): the refinement residual handed to the FP32 solve at unit norm
__global__ __launch_bounds__(256) void scale_to_f32_kernel(long long n, double s, const double* __restrict__ x,
                                                           float* __restrict__ y) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    y[i] = (float)(s * x[i]);
}

// x -= s (double) z32   (refinement update of a correction computed at scale 1/s)
__global__ __launch_bounds__(256) void sub_scaled_f32_kernel(long long n, double s, const float* __restrict__ z,
                                                             double* __restrict__ x) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    x[i] -= s * (double)z[i];
}

// kappa = exp(log kappa) in FP64 and FP32
__global__ __launch_bounds__(256) void exp_kernel(long long n, const double* __restrict__ logk, double* __restrict__ k64,
                                                  float* __restrict__ k32) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const double v = exp(logk[i]);
    k64[i] = v;
    k32[i] = (float)v;
  }
}

// dinv = 1 / d
template <typename T>
__global__ __launch_bounds__(256) void invert_kernel(long long n, const double* __restrict__ d, T* __restrict__ dinv) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    dinv[i] = (T)(1.0 / d[i]);
}

// y = dinv .* x  (SeqJac with one step and relaxation 1 from a zero start, or the
// identity when dinv == nullptr); also returns partials of y . x
template <typename T, typename A>
__global__ __launch_bounds__(kRedThreads) void prec_dot_kernel(long long n, const T* __restrict__ dinv,
                                                               const T* __restrict__ x, T* __restrict__ y,
                                                               A* __restrict__ partial) {
  A v[1] = {A(0)};
  for (long long i = (long long)blockIdx.x * kRedThreads + threadIdx.x; i < n; i += (long long)kRedBlocks * kRedThreads) {
    const T xi = x[i];
    const T yi = dinv ? dinv[i] * xi : xi;
    y[i] = yi;
    v[0] += (A)yi * (A)xi;
  }
  block_sum<A, 1>(v);
  if (threadIdx.x == 0) partial[blockIdx.x] = v[0];
}

// Device-side CG iteration (dune-istl CGSolver::apply, R:dune/istl/solvers.hh): the apply with
// the fused p.q partials, the update of r with the partials of (r.r, z.r), and the update of x
// and p. The sums in between are finished by single-workgroup launches (cg_pq_kernel,
// cg_check_kernel) or, where the partials are few, by every workgroup of the kernel that needs
// them: a launch costs 3 to 6 us with its gap, summing a thousand partials in each of a
// thousand workgroups 1 to 2 us. state = {iteration that stopped the loop or 0, aborted, iteration};
// dstate = {defect, def0, reduction}. Every kernel of an iteration after the one that stopped
// the loop returns at once.
// Scalar slots of the step lengths: the single-workgroup kernels divide once, and the
// vector kernels read the quotients (an FP64 division per wave cost ~10 us per launch).
constexpr int kSlotLambda = 8, kSlotBeta = 9;

// Most partials of one sum that the workgroups of a vector kernel add up themselves, and most
// elements for which the x/p update does so: its grid is exact above, 65536 workgroups at 2^24.
// us per iteration, point Jacobi, separate launches -> folded: 16^3 Q2 18.6 -> 13.1, 32^3 Q2 30.7 ->
// 27.4, 48^3 Q2 71.5 -> 61.1, 64^3 Q2 (7.1M) 132.9 -> 122.8; 64^3 Q3 (16.8M) with only p.q folded
// 306.3 -> 297.1, with the check folded too 307.3.
constexpr int kFoldPartials = 2048;
constexpr long long kFoldElements = 1LL << 23;

// The sums of the partials, by every workgroup alike (kRedThreads threads): all threads of all
// workgroups get the same bits.
template <typename A, int NR>
__device__ __forceinline__ void group_partial_sum(const A* __restrict__ partial, int nb, A (&v)[NR]) {
  __shared__ A red[NR][kRedThreads / 64];
#pragma unroll
  for (int j = 0; j < NR; ++j) v[j] = A(0);
  for (int b0 = threadIdx.x; b0 < nb; b0 += 4 * kRedThreads) {
    A a[4][NR];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int j = 0; j < NR; ++j) a[u][j] = b0 + u * kRedThreads < nb ? partial[(b0 + u * kRedThreads) * NR + j] : A(0);
#pragma unroll
    for (int j = 0; j < NR; ++j) v[j] += (a[0][j] + a[1][j]) + (a[2][j] + a[3][j]);
  }
#pragma unroll
  for (int j = 0; j < NR; ++j) {
    v[j] = wave_sum(v[j]);
    if ((threadIdx.x & 63) == 0) red[j][threadIdx.x >> 6] = v[j];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < NR; ++j) {
    A s = red[j][0];
#pragma unroll
    for (int w = 1; w < kRedThreads / 64; ++w) s += red[j][w];
    v[j] = s;
  }
}

// scal[0] = p.q from the apply's partials, scal[kSlotLambda] = lambda = scal[slot_rho] / p.q
template <typename A>
__global__ __launch_bounds__(kFinalThreads) void cg_pq_kernel(const A* __restrict__ partial, int nb,
                                                            A* __restrict__ scal, int slot_rho,
                                                            const int* __restrict__ stop) {
  if (*stop) return;
  A v[1];
  strided_partial_sum<A, 1>(partial, nb, v);
  if (threadIdx.x == 0) {
    scal[0] = v[0];
    scal[kSlotLambda] = scal[slot_rho] / v[0];
  }
}

// Which of an iteration's vectors are left in the 256 MB memory-side cache. dinv, read once, streams past
// it unless all five vectors fit (CG_ALL); q and z, which the next kernels read again, stay with p while
// these three fit (CG_KEEP); else only p, for the apply (CG_STREAM). x streams in cg_xpupdate_kernel;
// cg_xpcheck_kernel, for vectors of up to 2^23 elements, leaves all of its own. Each line's times are of one
// card and one run (the first solve has taken 501 to 537 ms on different cards). Mixed solve at 64^3 Q3
// lognormal (67 MB per vector): z and q streamed, dinv cached 519 ms, z and q kept, dinv streamed 505 ms,
// dinv cached as well 535 ms. FP64 CG at 64^3 Q3 (134 MB): dinv cached 829 ms, streamed 766 ms; with z and q
// kept 839 ms. At 72^3 Q2 (81 MB) 281, 273 and 290 ms. Mixed solve at 64^3 Q2 (28 MB): all cached 152 ms, as
// before 157 ms.
enum { CG_STREAM = 0, CG_KEEP = 1, CG_ALL = 2 };
constexpr int cg_cache(long long bytes) {
  return 5 * bytes <= 224LL << 20 ? CG_ALL : (3 * bytes <= 224LL << 20 ? CG_KEEP : CG_STREAM);
}
template <bool STREAM, typename V>
__device__ __forceinline__ V ld_vec(const V* p) {
  if constexpr (STREAM) return ld_stream<V>(p);
  else return *p;
}

// z = W^{-1} r: z -= lambda dinv q (r -= lambda q without a preconditioner); partials of r.r and
// z.r with r = z / dinv, two per workgroup. The loop carries z in r's place, so that the x/p update
// reads one vector, not r and dinv: FP32 64^3 Q3 (67 MB per vector) x/p 57.9 -> 51.3 us, this kernel
// 39.1 -> 39.5 us; FP64 CG at 64^3 Q3 297 -> 276 us per iteration. FOLD: lambda from the npq
// partials of p.q at pq (and scal[0], scal[kSlotLambda] set, as cg_pq_kernel does), else from
// scal[kSlotLambda].
template <typename T, typename A, bool FOLD, int CACHE>
__global__ __launch_bounds__(kRedThreads) void cg_rupdate_kernel(long long n, T* __restrict__ z, const T* __restrict__ q,
                                                                 const T* __restrict__ dinv, A* __restrict__ scal,
                                                                 A* __restrict__ partial, const int* __restrict__ state,
                                                                 const A* __restrict__ pq, int npq, int slot_rho) {
  if (state[0]) return;
  A v[2] = {A(0), A(0)};
  const long long S = (long long)gridDim.x * kRedThreads;
  T zv[kVecUnroll], qv[kVecUnroll], dv[kVecUnroll];
  auto load = [&](long long i0) {
#pragma unroll
    for (int u = 0; u < kVecUnroll; ++u) {
      const long long i = i0 + u * S;
      zv[u] = qv[u] = T(0);
      dv[u] = T(1);
      if (i < n) {  // z is stored cached for the x/p update that follows
        zv[u] = ld_vec<CACHE == CG_STREAM>(z + i);
        qv[u] = ld_vec<CACHE == CG_STREAM>(q + i);
        if (dinv) dv[u] = ld_vec<CACHE != CG_ALL>(dinv + i);
      }
    }
  };
  const long long first = (long long)blockIdx.x * kRedThreads + threadIdx.x;
  load(first);  // on their way while lambda is formed
  T lambda;
  if constexpr (FOLD) {
    A s[1];
    const A rho = scal[slot_rho];
    group_partial_sum<A, 1>(pq, npq, s);
    const A lam = rho / s[0];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      scal[0] = s[0];
      scal[kSlotLambda] = lam;
    }
    lambda = (T)lam;
  } else lambda = (T)scal[kSlotLambda];
  for (long long i0 = first; i0 < n;) {
#pragma unroll
    for (int u = 0; u < kVecUnroll; ++u) {
      const long long i = i0 + u * S;
      if (i < n) {
        const T zi = zv[u] - lambda * (dv[u] * qv[u]);
        z[i] = zi;
        const T ri = dinv ? zi / dv[u] : zi;
        v[0] += (A)ri * (A)ri;
        v[1] += (A)zi * (A)ri;
      }
    }
    i0 += kVecUnroll * S;
    if (i0 < n) load(i0);
  }
  block_sum_n<kRedThreads, A, 2>(v);
  if (threadIdx.x == 0) {
    partial[2 * blockIdx.x] = v[0];
    partial[2 * blockIdx.x + 1] = v[1];
  }
}

// IterativeSolver::Iteration::step of iteration it: records the defect and the iteration and
// raises the stop flag on convergence (def < reduction def0 or def < 1e-30) or on a non-finite
// defect. `stops` is the decision alone.
__device__ __forceinline__ bool cg_stops(double def, const double* __restrict__ dstate) {
  return !isfinite(def) || def < dstate[1] * dstate[2] || def < 1e-30;
}
__device__ __forceinline__ void cg_record(double def, int it, int* __restrict__ state, double* __restrict__ dstate) {
  state[2] = it;
  dstate[0] = def;
  if (!isfinite(def)) state[1] = 1;
  if (cg_stops(def, dstate)) state[0] = it;
}

// The step on the device by one workgroup: reduces the partials of (r.r, z.r) into out[0..1] and
// writes beta = z.r / rho_old.
template <typename A>
__global__ __launch_bounds__(kFinalThreads) void cg_check_kernel(const A* __restrict__ partial, int nb,
                                                               A* __restrict__ out, int* __restrict__ state,
                                                               double* __restrict__ dstate, int it,
                                                               const A* __restrict__ rho_old, A* __restrict__ beta) {
  if (state[0]) return;
  A v[2];
  strided_partial_sum<A, 2>(partial, nb, v);
  if (threadIdx.x == 0) {
    out[0] = v[0];
    out[1] = v[1];
    *beta = v[1] / *rho_old;
    cg_record(sqrt((double)v[0]), it, state, dstate);
  }
}

// x += lambda p (lambda = scal[kSlotLambda]), then p = z + beta p with beta = scal[kSlotBeta]; on
// the iteration that stopped the loop only x is updated (dune-istl leaves the loop after the
// defect check).
// Elements per thread of the x/p update: one double, or two contiguous floats (8 B per
// lane and stream either way).
template <typename T>
constexpr int xp_ept() { return sizeof(T) == 4 ? 2 : 1; }

template <typename T, typename A, bool KEEP>
__global__ __launch_bounds__(256) void cg_xpupdate_kernel(long long n, T* __restrict__ x, T* __restrict__ p,
                                                          const T* __restrict__ z, const A* __restrict__ scal,
                                                          const int* __restrict__ state, int it) {
  // xp_ept<T>() contiguous elements per thread over an exact grid: the fastest of the
  // access patterns measured for this five-stream update
  constexpr int E = xp_ept<T>();
  if (state[0] && state[0] != it) return;
  const long long i0 = ((long long)blockIdx.x * blockDim.x + threadIdx.x) * E;
  if (i0 >= n) return;
  const bool pupd = state[0] == 0;
  const T lambda = (T)scal[kSlotLambda];
  const T beta = pupd ? (T)scal[kSlotBeta] : T(0);
  // x streams (non-temporal); p, reread by the next apply, stays cached, z if KEEP
  if constexpr (E == 2) {
    if (i0 + 1 < n) {  // two contiguous floats as one 8-byte access per stream
      typedef T v2 __attribute__((ext_vector_type(2)));
      const v2 pv = *reinterpret_cast<const v2*>(p + i0);
      v2* xv = reinterpret_cast<v2*>(x + i0);
      st_stream<v2>(ld_stream<v2>(xv) + lambda * pv, xv);
      if (pupd) *reinterpret_cast<v2*>(p + i0) = ld_vec<!KEEP>(reinterpret_cast<const v2*>(z + i0)) + beta * pv;
      return;
    }
  }
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const long long i = i0 + e;
    if (i < n) {
      const T pv = p[i];
      st_stream<T>(ld_stream<T>(x + i) + lambda * pv, x + i);
      if (pupd) p[i] = ld_vec<!KEEP>(z + i) + beta * pv;
    }
  }
}

// b *= d or b /= d: between r and z = W^{-1} r = dinv r at the ends of the loop
template <typename T, bool DIV>
__global__ __launch_bounds__(256) void cg_scale_kernel(long long n, T* __restrict__ b, const T* __restrict__ d) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    b[i] = DIV ? b[i] / d[i] : b[i] * d[i];
}

// The same with the check of iteration `it` in front (cg_check_kernel's), by every workgroup from
// the nparts pairs of partials: out[0..1] = (r.r, z.r), beta = z.r / *rho_old. Workgroup 0 records
// the outcome; the others may see the flag it raises, so that the flag holds the iteration.
template <typename T, typename A>
__global__ __launch_bounds__(kRedThreads) void cg_xpcheck_kernel(long long n, T* __restrict__ x, T* __restrict__ p,
                                                                 const T* __restrict__ z, const A* __restrict__ scal,
                                                                 int* state, double* __restrict__ dstate, int it,
                                                                 const A* __restrict__ partial, int nparts,
                                                                 const A* __restrict__ rho_old, A* __restrict__ out) {
  const int stopped = *(volatile int*)state;
  if (stopped && stopped != it) return;
  const long long S = (long long)gridDim.x * kRedThreads;
  T xv[kVecUnroll], pv[kVecUnroll], zv[kVecUnroll];
  auto load = [&](long long i0) {
#pragma unroll
    for (int u = 0; u < kVecUnroll; ++u) {
      const long long i = i0 + u * S;
      xv[u] = pv[u] = zv[u] = T(0);
      if (i < n) {
        xv[u] = x[i];
        pv[u] = p[i];
        zv[u] = z[i];
      }
    }
  };
  const long long first = (long long)blockIdx.x * kRedThreads + threadIdx.x;
  load(first);  // on their way while the sums are formed
  const T lambda = (T)scal[kSlotLambda];
  const A rho = *rho_old;
  A v[2];
  group_partial_sum<A, 2>(partial, nparts, v);
  const double def = sqrt((double)v[0]);
  const T beta = (T)(v[1] / rho);
  const bool pupd = !cg_stops(def, dstate);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    out[0] = v[0];
    out[1] = v[1];
    cg_record(def, it, state, dstate);
  }
  for (long long i0 = first; i0 < n;) {
#pragma unroll
    for (int u = 0; u < kVecUnroll; ++u) {
      const long long i = i0 + u * S;
      if (i < n) {
        x[i] = xv[u] + lambda * pv[u];
        if (pupd) p[i] = zv[u] + beta * pv[u];
      }
    }
    i0 += kVecUnroll * S;
    if (i0 < n) load(i0);
  }
}

// CG direction update: p = dinv r + beta p
template <typename T>
__global__ __launch_bounds__(256) void cg_pupdate_kernel(long long n, T* __restrict__ p, const T* __restrict__ r,
                                                         const T* __restrict__ dinv, T beta) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const T zi = dinv ? dinv[i] * r[i] : r[i];
    p[i] = zi + beta * p[i];
  }
}

// ---------------------------------------------------------------------------
// Device-side BiCGSTAB (dune-istl BiCGSTABSolver::apply with its half-step Iteration
// counting). Per iteration: y1 = W^{-1} p, v = J y1 with rt.v, r -= alpha v with r.r, the
// half-step check, y2 = W^{-1} r, t = J y2 with (r.t, t.t), x += alpha y1 + omega y2 and
// r -= omega t with (r.r, rt.r), the full-step check. The loop is bound by these streams, so
// point Jacobi works inside the updates, p is kept only for a preconditioner with a launch of
// its own, x is updated once and the FP64 matrix-core apply takes the dots: 24 vectors read or
// written per iteration where one kernel per statement moved 31 (96^3 Q2 convection, 191 MB per
// vector: 1130 -> 920 us per iteration; the updates run at 5.8 to 6.3 TB/s). alpha and omega are
// formed by every workgroup of the update that uses them, from up to kFoldPartials partials (two
// launches fewer: 48^3 Q2 131 -> 121 us per iteration, 64^3 Q3 546 -> 538). Single-workgroup kernels
// form the others and keep the solver's scalars in FP64:
//   bs = {rho, rho_new, alpha, omega, beta}; state = {not 0 once stopped, abort code, half steps};
//   dstate = {defect, def0, reduction}.
// Once state[0] is set every later kernel that writes x, r or the scalars returns at once, but
// for the alpha part of x when it was the half step that stopped the loop: x and r are those of
// the half step at which it stopped.
enum { BICG_RUNNING = 0, BICG_NAN = 1, BICG_RHO = 2, BICG_OMEGA = 3, BICG_H = 4 };
constexpr int kBsRho = 0, kBsRhoNew = 1, kBsAlpha = 2, kBsOmega = 3, kBsBeta = 4;
constexpr double kBicgEps = 1e-80;  // dune-istl's EPSILON of BiCGSTABSolver

// Iteration::step(half / 2, norm) on the device; true when the loop stops here.
__device__ __forceinline__ bool bicg_step(int* state, double* dstate, int half, double norm) {
  state[2] = half;
  dstate[0] = norm;
  if (!isfinite(norm)) {
    state[1] = BICG_NAN;
    state[0] = 1;
    return true;
  }
  if (norm < dstate[1] * dstate[2] || norm < 1e-30) {
    state[0] = 1;
    return true;
  }
  return false;
}

// bs at the start: rho = alpha = omega = 1, rho_new = rt.r (= r.r, rt being r), beta = 0
__global__ __launch_bounds__(64) void bicg_init_kernel(double* __restrict__ bs, double rr) {
  if (threadIdx.x == 0) {
    bs[kBsRho] = 1.0;
    bs[kBsRhoNew] = rr;
    bs[kBsAlpha] = 1.0;
    bs[kBsOmega] = 1.0;
    bs[kBsBeta] = 0.0;
  }
}

// p = r (first iteration) or p = r + beta (p - omega v); with POINT the preconditioned
// direction y = dinv p in p's place: y = dinv r or y = dinv (r - beta omega v) + beta y. One
// element per thread over an exact grid, as in cg_xpupdate_kernel. DSTREAM, here and below: dinv
// streams past the memory-side cache, for vectors that do not all fit there (cg_cache; 96^3 Q2 925 ->
// 918, 64^3 Q3 559 -> 545 us per iteration; at 48^3 Q2, where they fit, no gain: 127 and 131 us).
template <typename T, bool POINT, bool DSTREAM>
__global__ __launch_bounds__(256) void bicg_dir_kernel(long long n, T* __restrict__ p, const T* __restrict__ r,
                                                       const T* __restrict__ v, const T* __restrict__ dinv,
                                                       const double* __restrict__ bs, const int* __restrict__ state,
                                                       int first) {
  constexpr int E = xp_ept<T>();
  typedef T V __attribute__((ext_vector_type(E)));
  if (state[0]) return;
  const T beta = (T)bs[kBsBeta], omega = (T)bs[kBsOmega], bo = beta * omega;
  const long long i0 = ((long long)blockIdx.x * blockDim.x + threadIdx.x) * E;
  if (i0 >= n) return;
  if (i0 + E <= n) {
    V pn = *reinterpret_cast<const V*>(r + i0);
    V d;
    if constexpr (POINT) d = ld_vec<DSTREAM>(reinterpret_cast<const V*>(dinv + i0));
    if (!first) {
      const V po = *reinterpret_cast<const V*>(p + i0), vo = ld_stream<V>(reinterpret_cast<const V*>(v + i0));
      if constexpr (POINT) pn = d * (pn - bo * vo) + beta * po;
      else pn = beta * (po - omega * vo) + pn;
    } else if constexpr (POINT) pn = d * pn;
    *reinterpret_cast<V*>(p + i0) = pn;
    return;
  }
  for (long long i = i0; i < n; ++i) {  // an odd last float
    T pn = r[i];
    if (!first) {
      if constexpr (POINT) pn = dinv[i] * (pn - bo * v[i]) + beta * p[i];
      else pn = beta * (p[i] - omega * v[i]) + pn;
    } else if constexpr (POINT) pn = dinv[i] * pn;
    p[i] = pn;
  }
}

// y = dinv .* x (or y = x), skipped once the loop has stopped
template <typename T>
__global__ __launch_bounds__(256) void prec_stop_kernel(long long n, const T* __restrict__ dinv, const T* __restrict__ x,
                                                        T* __restrict__ y, const int* __restrict__ state) {
  if (state[0]) return;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    y[i] = dinv ? dinv[i] * x[i] : x[i];
}

// alpha of the half step from h = rt.v; false: abort, |h| < EPSILON
__device__ __forceinline__ bool bicg_alpha(double h, const double* __restrict__ bs, const double* __restrict__ dstate,
                                           double& alpha) {
  alpha = dstate[0] == 0.0 ? 0.0 : bs[kBsRhoNew] / h;
  return !(fabs(h) < kBicgEps);
}

// First half step `half`: r -= alpha v with the r.r partials; with POINT also y = dinv r. FOLD: alpha
// from the nd partials of rt.v at dots, by every workgroup (bicg_scalar_kernel's phase 0), else from
// bs. On an abort workgroup 0 raises the flag as -half, which no wave of this launch obeys: a workgroup
// that starts late may read it in some waves and not in others, and all of them have to meet at
// the barrier of the sum, whose result sends every one of them away.
template <typename T, typename A, bool POINT, bool DSTREAM, bool FOLD>
__global__ __launch_bounds__(kRedThreads) void bicg_half_kernel(long long n, T* __restrict__ r, const T* __restrict__ v,
                                                                const T* __restrict__ dinv, T* __restrict__ y,
                                                                double* bs, A* __restrict__ partial, int* state,
                                                                int half, const double* __restrict__ dstate,
                                                                const A* __restrict__ dots, int nd) {
  const int stopped = *(volatile int*)state;
  if (stopped && stopped != -half) return;
  A s[1] = {A(0)};
  constexpr long long S = (long long)kRedBlocks * kRedThreads;
  T rv[kVecUnroll], vv[kVecUnroll], dv[kVecUnroll];
  auto load = [&](long long i0) {
#pragma unroll
    for (int u = 0; u < kVecUnroll; ++u) {
      const long long i = i0 + u * S;
      rv[u] = vv[u] = dv[u] = T(0);
      if (i < n) {
        rv[u] = r[i];
        vv[u] = v[i];
        if constexpr (POINT) dv[u] = ld_vec<DSTREAM>(dinv + i);
      }
    }
  };
  const long long first = (long long)blockIdx.x * kRedThreads + threadIdx.x;
  load(first);  // on their way while alpha is formed
  T alpha;
  if constexpr (FOLD) {
    A h[1];
    double al;
    group_partial_sum<A, 1>(dots, nd, h);
    const bool go = bicg_alpha((double)h[0], bs, dstate, al);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      if (go) bs[kBsAlpha] = al;
      else {
        state[1] = BICG_H;
        state[0] = -half;
      }
    }
    if (!go) return;
    alpha = (T)al;
  } else alpha = (T)bs[kBsAlpha];
  for (long long i0 = first; i0 < n;) {
#pragma unroll
    for (int u = 0; u < kVecUnroll; ++u) {
      const long long i = i0 + u * S;
      if (i < n) {
        const T ri = rv[u] - alpha * vv[u];
        r[i] = ri;
        if constexpr (POINT) y[i] = dv[u] * ri;
        s[0] += (A)ri * (A)ri;
      }
    }
    i0 += kVecUnroll * S;
    if (i0 < n) load(i0);
  }
  block_sum<A, 1>(s);
  if (threadIdx.x == 0) partial[blockIdx.x] = s[0];
}

// Second half step `half`: x += alpha y1 + omega y2, r -= omega t with the (r.r, rt.r)
// partials; y2 null: r before its update (no preconditioner); y1 null: its part is in x already.
// If the first half step stopped the loop, only x += alpha y1. FOLD: omega from the nd pairs of
// partials of (r.t, t.t) at dots, by every workgroup (bicg_scalar_kernel's phase 2), else from bs.
template <typename T, typename A, bool FOLD>
__global__ __launch_bounds__(kRedThreads) void bicg_full_kernel(long long n, T* __restrict__ x, const T* __restrict__ y1,
                                                                const T* __restrict__ y2, T* __restrict__ r,
                                                                const T* __restrict__ t, const T* __restrict__ rt,
                                                                double* bs, A* __restrict__ partial,
                                                                const int* __restrict__ state, int half,
                                                                const double* __restrict__ dstate,
                                                                const A* __restrict__ dots, int nd) {
  const long long first = (long long)blockIdx.x * kRedThreads + threadIdx.x;
  constexpr long long S = (long long)kRedBlocks * kRedThreads;
  const T alpha = (T)bs[kBsAlpha];
  if (state[0]) {
    if (state[2] == half - 1 && y1)
      for (long long i = first; i < n; i += S) x[i] += alpha * y1[i];
    return;
  }
  A s[2] = {A(0), A(0)};
  T xv[kVecUnroll], av[kVecUnroll], bv[kVecUnroll], rv[kVecUnroll], tv[kVecUnroll], sv[kVecUnroll];
  auto load = [&](long long i0) {
#pragma unroll
    for (int u = 0; u < kVecUnroll; ++u) {
      const long long i = i0 + u * S;
      xv[u] = av[u] = bv[u] = rv[u] = tv[u] = sv[u] = T(0);
      if (i < n) {
        xv[u] = ld_stream<T>(x + i);
        if (y1) av[u] = y1[i];
        rv[u] = r[i];
        bv[u] = y2 ? ld_stream<T>(y2 + i) : rv[u];
        tv[u] = ld_stream<T>(t + i);
        sv[u] = ld_stream<T>(rt + i);
      }
    }
  };
  load(first);  // on their way while omega is formed
  T omega;
  if constexpr (FOLD) {
    A d[2];
    group_partial_sum<A, 2>(dots, nd, d);
    const double om = dstate[0] == 0.0 ? 0.0 : (double)d[0] / (double)d[1];
    if (blockIdx.x == 0 && threadIdx.x == 0) bs[kBsOmega] = om;
    omega = (T)om;
  } else omega = (T)bs[kBsOmega];
  for (long long i0 = first; i0 < n;) {
#pragma unroll
    for (int u = 0; u < kVecUnroll; ++u) {
      const long long i = i0 + u * S;
      if (i < n) {
        T xi = xv[u];
        if (y1) xi += alpha * av[u];
        st_stream<T>(xi + omega * bv[u], x + i);
        const T ri = rv[u] - omega * tv[u];
        r[i] = ri;
        s[0] += (A)ri * (A)ri;
        s[1] += (A)sv[u] * (A)ri;
      }
    }
    i0 += kVecUnroll * S;
    if (i0 < n) load(i0);
  }
  block_sum<A, 2>(s);
  if (threadIdx.x == 0) {
    partial[2 * blockIdx.x] = s[0];
    partial[2 * blockIdx.x + 1] = s[1];
  }
}

// The scalar steps, one workgroup reducing the partials first:
//   PHASE 0: h = rt.v; |h| < EPSILON aborts; alpha = rho_new / h (0 when the defect is 0)
//   PHASE 1: defect of the half step, Iteration::step
//   PHASE 2: omega = r.t / t.t (0 when the defect is 0)
//   PHASE 3: defect of the full step, rho = rho_new, rho_new = rt.r, Iteration::step; then
//            the breakdown checks at the top of dune-istl's next iteration (|rho|, |omega|
//            <= EPSILON) and beta = (rho_new / rho)(alpha / omega)
template <typename A, int PHASE>
__global__ __launch_bounds__(kFinalThreads) void bicg_scalar_kernel(const A* __restrict__ partial, int nb,
                                                                    double* __restrict__ bs, int* __restrict__ state,
                                                                    double* __restrict__ dstate, int half) {
  if (state[0]) return;
  constexpr int NR = (PHASE == 2 || PHASE == 3) ? 2 : 1;
  A v[NR];
  strided_partial_sum<A, NR>(partial, nb, v);
  if (threadIdx.x != 0) return;
  const double norm = dstate[0];
  if constexpr (PHASE == 0) {
    double alpha;
    if (!bicg_alpha((double)v[0], bs, dstate, alpha)) {
      state[1] = BICG_H;
      state[0] = 1;
      return;
    }
    bs[kBsAlpha] = alpha;
  } else if constexpr (PHASE == 1) {
    bicg_step(state, dstate, half, sqrt((double)v[0]));
  } else if constexpr (PHASE == 2) {
    bs[kBsOmega] = norm == 0.0 ? 0.0 : (double)v[0] / (double)v[1];
  } else {
    const double nrm = sqrt((double)v[0]);
    bs[kBsRho] = bs[kBsRhoNew];
    bs[kBsRhoNew] = (double)v[1];
    if (bicg_step(state, dstate, half, nrm)) return;
    if (fabs(bs[kBsRho]) <= kBicgEps) {
      state[1] = BICG_RHO;
      state[0] = 1;
      return;
    }
    if (fabs(bs[kBsOmega]) <= kBicgEps) {
      state[1] = BICG_OMEGA;
      state[0] = 1;
      return;
    }
    bs[kBsBeta] = nrm == 0.0 ? 0.0 : (bs[kBsRhoNew] / bs[kBsRho]) * (bs[kBsAlpha] / bs[kBsOmega]);
  }
}

}  // namespace pdelab_amd

#endif
