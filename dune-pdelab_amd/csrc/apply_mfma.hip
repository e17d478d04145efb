// apply_mfma.hip -- launches of the matrix-core apply (dg_mfma.hh): Q2 and Q3 in FP64.
#include "handle.hh"

// f(kernel) with the instance of a degree, coefficient form and mode
template <int N1, int KIND, typename F>
static void with_mode(int mode, F f) {
  switch (mode) {
    case 1: f(dg_mfma_kernel<N1, KIND, 1>); break;
    case 2: f(dg_mfma_kernel<N1, KIND, 2>); break;
    case 3: f(dg_mfma_kernel<N1, KIND, 3>); break;
    case 4: f(dg_mfma_kernel<N1, KIND, 4>); break;
    case 5: f(dg_mfma_kernel<N1, KIND, 5>); break;
    default: f(dg_mfma_kernel<N1, KIND, 0>); break;
  }
}
template <int N1, typename F>
static void with_kind(int kind, int mode, F f) {
  switch (kind) {
    case MFMA_CONST: with_mode<N1, MFMA_CONST>(mode, f); break;
    case MFMA_CONV: with_mode<N1, MFMA_CONV>(mode, f); break;
    case MFMA_GENERAL: with_mode<N1, MFMA_GENERAL>(mode, f); break;
    case MFMA_TENSOR: with_mode<N1, MFMA_TENSOR>(mode, f); break;
    default: with_mode<N1, MFMA_WEIGHT>(mode, f); break;
  }
}
// Arguments of one launch without the field's.
MfmaArgs mfma_args(const H* h, bool trans) {
  MfmaArgs a;
  std::memset(&a, 0, sizeof(a));
  const DGArgs<double>& d = h->a64;
  a.nx = d.n[0];
  a.ny = d.n[1];
  a.nz = d.n[2];
  a.np = (unsigned)((long long)d.n[0] * d.n[1]);
  const MfmaGrid grid = mfma_grid(h);
  a.zw = grid.zw;
  a.zsegs = grid.zsegs;
  a.prow = grid.prow;
  a.prows = grid.prow ? (unsigned)(grid.wgs / grid.prow) : 0;
  a.vc = d.vc;
  for (int i = 0; i < 3; ++i) a.S[i] = d.S[i];
  a.fg = trans ? -d.theta : 1.0;
  a.fh = trans ? -1.0 : d.theta;
  a.alphak = d.alphak;
  a.weightsOn = d.weightsOn;
  for (int s = 0; s < 6; ++s) a.bc[s] = d.bc[s];
  a.x = h->mfma_x[(trans ? 1 : 0) + (h->vark ? 2 : 0)];
  if (!h->vark)
    for (int i = 0; i < h->n1; ++i) a.x.A[i][i] += a.vc;
  return a;
}

int launch_apply_mfma(H* h, const double* z, double* y, bool trans, int mode, double* dotp, const int* stop,
                      const double* w) {
  const MfmaArgs a = mfma_args(h, trans);
  const unsigned nb = (unsigned)mfma_blocks(h);
  // J and J^T, each with the whole matrices and with their convection part (cell-wise kappa)
  const MfmaTab* tab = h->d_tab->mfma + (trans ? 1 : 0) + (h->vark ? 2 : 0);
  const int kind = mfma_kind(h, false);
  const double* fc = kind == MFMA_WEIGHT || kind == MFMA_TENSOR ? h->d_fw64 : h->d_fc64;
  auto run = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(nb), dim3(256), 0, h->stream, z, y, fc, tab, a, nb, dotp, stop, w);
  };
  if (h->n1 == 3) with_kind<3>(kind, mode, run);
  else with_kind<4>(kind, mode, run);
  HIPCHK(h, hipGetLastError());
  return PDELAB_OK;
}

int mfma_weights(H* h) {
  hipLaunchKernelGGL(mfma_weight_kernel, dim3((unsigned)((h->ncells + 255) / 256)), dim3(256), 0, h->stream,
                     (const double*)h->d_fc64, h->d_fw64, h->ncells, h->a64.aniso);
  HIPCHK(h, hipGetLastError());
  return PDELAB_OK;
}

// Fills one table from the 1D matrices m (no reaction) and the tables of al; cellwise: m is the
// convection part, the x-line constants are those of cell-wise kappa.
static void fill_tab(const DGArgs<long double>& al, const LineMats<long double>& m, bool trans, bool cellwise, int n,
                     MfmaTab& t, MfmaX& x) {
  std::memset(&t, 0, sizeof(t));
  std::memset(&x, 0, sizeof(x));
  auto lane = [&](double (&dst)[16], auto f) {
    for (int i = 0; i < n; ++i)
      for (int k = 0; k < n; ++k) dst[4 * i + k] = (double)f(i, k);
  };
  const long double th = al.theta;
  const long double g = trans ? -th : 1.0L, hh = trans ? -1.0L : th;
  auto e0 = [&](int k) { return (long double)(k == 0); };
  auto e1 = [&](int k) { return (long double)(k == n - 1); };
  for (int s = 0; s < 2; ++s) {
    const int d = s + 1;
    lane(t.own[s], [&](int i, int k) { return m.A[d][i][k]; });
    lane(t.dlo[s], [&](int i, int k) { return m.Dlo[d][i][k]; });
    lane(t.dhi[s], [&](int i, int k) { return m.Dhi[d][i][k]; });
    lane(t.nlo[s], [&](int i, int k) { return m.Pl[d][i] * e1(k) + m.Ql[d][i] * al.d1[k]; });
    lane(t.nhi[s], [&](int i, int k) { return m.Pr[d][i] * e0(k) + m.Qr[d][i] * al.d0[k]; });
  }
  lane(t.M, [&](int i, int k) { return al.M[i][k]; });
  lane(t.K, [&](int i, int k) { return al.MiK[i][k]; });
  lane(t.U[0], [&](int i, int k) { return g * al.Mie0[i] * al.d0[k] - hh * al.Mid0[i] * e0(k); });
  lane(t.U[1], [&](int i, int k) { return al.Mie0[i] * e0(k); });
  lane(t.U[2], [&](int i, int k) { return al.Mie1[i] * e1(k); });
  lane(t.U[3], [&](int i, int k) { return g * al.Mie1[i] * al.d1[k] - hh * al.Mid1[i] * e1(k); });
  lane(t.X[0], [&](int i, int k) { return g * al.Mie0[i] * al.d1[k]; });
  lane(t.X[1], [&](int i, int k) { return -al.Mie0[i] * e1(k); });
  lane(t.X[2], [&](int i, int k) { return hh * al.Mid0[i] * e1(k); });
  lane(t.X[3], [&](int i, int k) { return -al.Mie1[i] * e0(k); });
  lane(t.X[4], [&](int i, int k) { return -g * al.Mie1[i] * al.d0[k]; });
  lane(t.X[5], [&](int i, int k) { return -hh * al.Mid1[i] * e0(k); });
  const long double al1 = al.alphak, al2 = 2 * al1;
  lane(t.WL, [&](int i, int k) { return g * al.Mie0[i] * al.d0[k] - hh * al.Mid0[i] * e0(k) + al2 * al.Mie0[i] * e0(k); });
  lane(t.WU, [&](int i, int k) { return al2 * al.Mie1[i] * e1(k) - g * al.Mie1[i] * al.d1[k] + hh * al.Mid1[i] * e1(k); });
  lane(t.NL, [&](int i, int k) { return g * al.Mie0[i] * al.d1[k] - al2 * al.Mie0[i] * e1(k) + hh * al.Mid0[i] * e1(k); });
  lane(t.NU, [&](int i, int k) { return -al2 * al.Mie1[i] * e0(k) - g * al.Mie1[i] * al.d0[k] - hh * al.Mid1[i] * e0(k); });
  for (int s = 0; s < 2; ++s) {
    if (al.bc[2 * (s + 1)] == BC_DIRICHLET)
      lane(t.BL[s], [&](int i, int k) { return g * al.Mie0[i] * al.d0[k] - hh * al.Mid0[i] * e0(k) + al1 * al.Mie0[i] * e0(k); });
    if (al.bc[2 * (s + 1) + 1] == BC_DIRICHLET)
      lane(t.BU[s], [&](int i, int k) { return al1 * al.Mie1[i] * e1(k) - g * al.Mie1[i] * al.d1[k] + hh * al.Mid1[i] * e1(k); });
  }
  for (int i = 0; i < n; ++i) {
    for (int j = 0; j < n; ++j) {
      t.A[i][j] = (double)m.A[0][i][j];
      t.Dlo[i][j] = (double)m.Dlo[0][i][j];
      t.Dhi[i][j] = (double)m.Dhi[0][i][j];
      x.M[i][j] = (double)al.M[i][j];
      x.A[i][j] = (double)(cellwise ? al.MiK[i][j] : m.A[0][i][j]);
    }
    t.Pl[i] = (double)m.Pl[0][i];
    t.Ql[i] = (double)m.Ql[0][i];
    t.Pr[i] = (double)m.Pr[0][i];
    t.Qr[i] = (double)m.Qr[0][i];
    x.d1[i] = (double)al.d1[i];
    x.P[i] = (double)(cellwise ? al.Mie0[i] : m.Pl[0][i]);
    x.Q[i] = (double)(cellwise ? al.Mid0[i] : m.Ql[0][i]);
  }
}

void mfma_setup(H* h, const DGArgs<long double>& al, const LineMats<long double> (&m)[2],
                const LineMats<long double> (&mconv)[2], MfmaTab (&t)[4]) {
  for (int tr = 0; tr < 2; ++tr) {
    fill_tab(al, m[tr], tr == 1, false, h->n1, t[tr], h->mfma_x[tr]);
    fill_tab(al, mconv[tr], tr == 1, true, h->n1, t[2 + tr], h->mfma_x[2 + tr]);
  }
}
