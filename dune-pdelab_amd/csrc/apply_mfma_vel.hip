// apply_mfma_vel.hip -- launches of the matrix-core apply with the velocity field's convection
// terms in the same pass (dg_mfma.hh, VEL).
#include "handle.hh"

template <int N1, int M, int KIND, int VEL>
static void launch_mode(H* h, const double* z, double* y, const MfmaTab* tab, const MfmaArgs& a, unsigned nb, bool accum,
                        const int* stop) {
  const double* fc = KIND == MFMA_WEIGHT ? h->d_fw64 : h->d_fc64;
  if (accum)
    hipLaunchKernelGGL((dg_mfma_kernel<N1, KIND, 1, VEL, M>), dim3(nb), dim3(256), 0, h->stream, z, y, fc, tab, a, nb,
                       (double*)nullptr, stop);
  else
    hipLaunchKernelGGL((dg_mfma_kernel<N1, KIND, 0, VEL, M>), dim3(nb), dim3(256), 0, h->stream, z, y, fc, tab, a, nb,
                       (double*)nullptr, stop);
}

template <int N1, int M, int VEL>
static void launch_kind(H* h, const double* z, double* y, const MfmaTab* tab, const MfmaArgs& a, unsigned nb, bool accum,
                        const int* stop) {
  if (!h->vark) launch_mode<N1, M, MFMA_CONST, VEL>(h, z, y, tab, a, nb, accum, stop);
  else if (h->a64.aniso || !h->a64.weightsOn) launch_mode<N1, M, MFMA_GENERAL, VEL>(h, z, y, tab, a, nb, accum, stop);
  else launch_mode<N1, M, MFMA_WEIGHT, VEL>(h, z, y, tab, a, nb, accum, stop);
}

template <int N1, int M>
static void launch_nm(H* h, const double* z, double* y, const MfmaTab* tab, const MfmaArgs& a, unsigned nb, bool trans,
                      bool accum, const int* stop) {
  if (trans) launch_kind<N1, M, 2>(h, z, y, tab, a, nb, accum, stop);
  else launch_kind<N1, M, 1>(h, z, y, tab, a, nb, accum, stop);
}

int launch_apply_mfma_vel(H* h, const double* z, double* y, bool trans, bool accum, const int* stop) {
  MfmaArgs a = mfma_args(h, trans);
  a.bv = h->d_bv64;
  a.bf = h->d_bf64;
  a.vt = h->d_mfma_vel;
  for (int d = 0; d < 3; ++d) {
    a.vs[d] = h->va64.vs[d];
    a.area[d] = h->va64.area[d];
  }
  const unsigned nb = (unsigned)mfma_blocks(h);
  const MfmaTab* tab = h->d_tab->mfma + (trans ? 1 : 0) + (h->vark ? 2 : 0);
  if (h->n1 == 4) launch_nm<4, 4>(h, z, y, tab, a, nb, trans, accum, stop);
  else if (h->tab.m == 3) launch_nm<3, 3>(h, z, y, tab, a, nb, trans, accum, stop);
  else launch_nm<3, 4>(h, z, y, tab, a, nb, trans, accum, stop);
  HIPCHK(h, hipGetLastError());
  return PDELAB_OK;
}

int mfma_vel_setup(H* h) {
  MfmaVelTab t;
  std::memset(&t, 0, sizeof(t));
  const Tables1D& tb = h->tab;
  const VelArgs<double>& v = h->va64;
  for (int q = 0; q < tb.m && q < 4; ++q)
    for (int i = 0; i < tb.n1; ++i) {
      const long double P = tb.P[q][i], D = lagrange_dp(tb.k, i, tb.qx[q]), w = tb.qw[q];
      t.LB[4 * q + i] = t.B[q][i] = (double)P;
      t.LD[4 * q + i] = t.D[q][i] = (double)D;
      t.WB[4 * i + q] = t.BW[q][i] = (double)(w * P);
      t.WDy[4 * i + q] = (double)(v.vs[1] * w * D);
      t.WDz[4 * i + q] = (double)(v.vs[2] * w * D);
      t.DW[q][i] = (double)(v.vs[0] * w * D);
    }
  HIPCHK(h, hipMalloc(&h->d_mfma_vel, sizeof(t)));
  HIPCHK(h, hipMemcpy(h->d_mfma_vel, &t, sizeof(t), hipMemcpyHostToDevice));
  return PDELAB_OK;
}
