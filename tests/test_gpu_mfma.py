"""The matrix-core apply (Q2 and Q3, FP64) against the oracle where its tiling has edges: planes
that are no multiple of a wave's four cells or a workgroup's sixteen (the last group is moved
back), rows shorter than a group, one plane, walks that end inside a column, every kind of
coefficient, and vectors that are only 8-byte aligned.

Tolerance: 1e-12 relative (2-norm), the operator's; a line operator sums at most 3 x 4 products
per direction and the mass sweeps 4 each, about 60 roundings of 1.1e-16 on values of the size of
the largest term, whose cancellation in the penalty terms costs up to two digits.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
RTOL = 1e-12

GRIDS = [(4, 1, 1), (2, 2, 3), (5, 1, 2), (1, 7, 2), (3, 3, 1), (7, 5, 3), (16, 1, 4), (17, 3, 2), (13, 11, 35)]
KINDS = {
    "const": dict(),
    "react": dict(c=0.7),
    "conv": dict(b=(1.0, -0.5, 0.25), c=0.3, kappa0=0.05),
    "outflow": dict(b=(1.0, 0.0, 0.0), bctype=(0, -2, 0, -1, -3, 0)),
    "cells": dict(kappa_per_cell=1),
    "cells_neumann": dict(kappa_per_cell=1, bctype=(-1, 0, 0, -1, 0, -1), method=0),
    "cells_conv": dict(kappa_per_cell=1, b=(-0.5, 1.0, 2.0)),
    "cells_off": dict(kappa_per_cell=1, weights=1),
    "tensor": dict(kappa_per_cell=2, lx=2.0, ly=0.5),
}


@pytest.mark.parametrize("degree", [2, 3])
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: "x".join(map(str, g)))
def test_mfma_apply_edges(pkg, of, grid, kind, degree):
    print(f"[gpu] matrix-core apply {grid} Q{degree} {kind}", flush=True)
    nx, ny, nz = grid
    cfg = pkg.make_config(nx=nx, ny=ny, nz=nz, degree=degree, alpha=3.0, **KINDS[kind])
    rng = np.random.default_rng(7)
    kappa = np.exp(rng.normal(size=pkg.ncells(cfg) * (3 if cfg.kappa_per_cell == 2 else 1))) if cfg.kappa_per_cell else None
    go, o = pkg.GridOperator(cfg, kappa), of.Oracle(cfg, kappa)
    z, y0 = rng.uniform(-1, 1, go.N), rng.uniform(-1, 1, go.N)
    zd, yd = go.vector(z), go.vector(y0)
    ref = o.jacobian_apply(z)
    go.jacobian_apply(zd, yd)
    assert np.linalg.norm(yd.download() - y0 - ref) <= RTOL * (np.linalg.norm(ref) + np.linalg.norm(y0))
    go.operator_apply(zd, yd)
    assert np.linalg.norm(yd.download() - ref) <= RTOL * np.linalg.norm(ref)
    ref = o.jacobian_apply_transpose(z)
    yd.zero()
    go.jacobian_apply_transpose(zd, yd)
    assert np.linalg.norm(yd.download() - ref) <= RTOL * np.linalg.norm(ref)


@pytest.mark.parametrize("degree", [2, 3])
def test_mfma_apply_offset_vectors(pkg, degree):
    """The same result, bit for bit, from vectors that start 8 bytes after an allocation, and
    nothing written outside them."""
    cfg = pkg.make_config(nx=7, ny=5, nz=6, degree=degree, alpha=3.0)
    go = pkg.GridOperator(cfg)
    z = np.random.default_rng(8).uniform(-1, 1, go.N)
    y = go.vector()
    go.operator_apply(go.vector(z), y)
    pad = pkg.DeviceVector(go, go.N + 2).upload(np.concatenate([[1e300], z, [1e300]]))
    out = pkg.DeviceVector(go, go.N + 2).upload(np.full(go.N + 2, 3.0))
    p = lambda v: ctypes.c_void_p(v.ptr.value + 8)  # noqa: E731
    assert pkg.lib().pdelab_gpu_operator_apply(go.h, p(pad), p(out)) == 0
    got = out.download()
    assert np.array_equal(got[1:-1], y.download()) and got[0] == 3.0 and got[-1] == 3.0


def test_mfma_apply_nan_stays_local(pkg):
    """A NaN in one cell reaches that cell and its face neighbours only."""
    cfg = pkg.make_config(nx=6, ny=4, nz=5, degree=3, alpha=3.0)
    go = pkg.GridOperator(cfg)
    z = np.ones(go.N)
    c = 2 + 6 * (1 + 4 * 2)
    z[64 * c + 5] = np.nan
    y = go.vector()
    go.operator_apply(go.vector(z), y)
    bad = np.flatnonzero(np.isnan(y.download().reshape(-1, 64)).any(axis=1))
    assert set(bad) <= {c, c - 1, c + 1, c - 6, c + 6, c - 24, c + 24} and c in bad


FIELDS = {
    "const": dict(),
    "intorderadd2": dict(intorderadd=2),
    "cells": dict(kappa_per_cell=1, c=0.3),
    "cells_neumann": dict(kappa_per_cell=1, bctype=(-1, 0, -3, -1, 0, -1), method=0),
    "cells_off": dict(kappa_per_cell=1, weights=1),
    "tensor_add2": dict(kappa_per_cell=2, lx=2.0, ly=0.5, intorderadd=2),
    "outflow": dict(kappa0=0.1, bctype=(0, -2, -1, 0, 0, -2)),
}


@pytest.mark.parametrize("degree", [2, 3])
@pytest.mark.parametrize("kind", FIELDS)
@pytest.mark.parametrize("grid", [(4, 1, 1), (2, 2, 3), (5, 3, 2), (3, 3, 4), (17, 1, 2), (6, 7, 34)],
                         ids=lambda g: "x".join(map(str, g)))
def test_mfma_velocity_edges(pkg, of, grid, kind, degree):
    """The velocity field's terms in the same pass, J and J^T: random values (positive where a
    side is an outflow side), so every face point's upwind choice is its own."""
    print(f"[gpu] matrix-core apply with a velocity field {grid} Q{degree} {kind}", flush=True)
    nx, ny, nz = grid
    cfg = pkg.make_config(nx=nx, ny=ny, nz=nz, degree=degree, alpha=3.0, **FIELDS[kind])
    rng = np.random.default_rng(9)
    kappa = np.exp(rng.normal(size=pkg.ncells(cfg) * (3 if cfg.kappa_per_cell == 2 else 1))) if cfg.kappa_per_cell else None
    m = pkg.quadrature_points(cfg)
    nf = (nx + 1) * ny * nz + nx * (ny + 1) * nz + nx * ny * (nz + 1)
    bv, bf = rng.normal(size=nx * ny * nz * 3 * m ** 3), rng.normal(size=nf * m ** 2)
    if kind == "outflow":
        bf = np.abs(bf)
    go, o = pkg.GridOperator(cfg, kappa), of.Oracle(cfg, kappa)
    go.set_velocity_field(bv, bf)
    o.set_velocity_field(bv, bf)
    z, y0 = rng.uniform(-1, 1, go.N), rng.uniform(-1, 1, go.N)
    zd, yd = go.vector(z), go.vector(y0)
    ref = o.jacobian_apply(z)
    go.jacobian_apply(zd, yd)
    assert np.linalg.norm(yd.download() - y0 - ref) <= RTOL * (np.linalg.norm(ref) + np.linalg.norm(y0))
    go.operator_apply(zd, yd)
    assert np.linalg.norm(yd.download() - ref) <= RTOL * np.linalg.norm(ref)
    ref = o.jacobian_apply_transpose(z)
    yd.zero()
    go.jacobian_apply_transpose(zd, yd)
    assert np.linalg.norm(yd.download() - ref) <= RTOL * np.linalg.norm(ref)


@pytest.mark.parametrize("degree", [2, 3])
@pytest.mark.parametrize("kind", ["const", "outflow", "cells", "cells_conv", "tensor"])
@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: "x".join(map(str, g)))
def test_mfma_residual_edges(pkg, of, grid, kind, degree):
    """r += R(x): R(0) is added by the apply. Tolerance RTOL of the apply's and the load's size."""
    print(f"[gpu] matrix-core residual {grid} Q{degree} {kind}", flush=True)
    nx, ny, nz = grid
    cfg = pkg.make_config(nx=nx, ny=ny, nz=nz, degree=degree, alpha=3.0, problem=pkg.PROBLEM_CONSTANT, f0=1.0, **KINDS[kind])
    rng = np.random.default_rng(11)
    kappa = np.exp(rng.normal(size=pkg.ncells(cfg) * (3 if cfg.kappa_per_cell == 2 else 1))) if cfg.kappa_per_cell else None
    go, o = pkg.GridOperator(cfg, kappa), of.Oracle(cfg, kappa)
    x, r0 = rng.uniform(-1, 1, go.N), rng.uniform(-1, 1, go.N)
    xd, rd = go.vector(x), go.vector(r0)
    go.residual(xd, rd)
    ref = o.residual(x)
    assert np.linalg.norm(rd.download() - r0 - ref) <= RTOL * (np.linalg.norm(ref) + np.linalg.norm(r0))


@pytest.mark.parametrize("precond", [0, 1, 2], ids=["none", "point", "block"])
@pytest.mark.parametrize("degree", [1, 2, 3])
@pytest.mark.parametrize("kind", ["const", "conv", "cells_conv", "tensor"])
@pytest.mark.parametrize("grid", [(4, 1, 1), (5, 1, 2), (7, 5, 3), (13, 11, 35)], ids=lambda g: "x".join(map(str, g)))
def test_bicgstab_first_iterations(pkg, of, grid, kind, degree, precond):
    """The iterate after one and two BiCGSTAB iterations (Q1's dots are passes of their own, Q2's
    and Q3's part of the apply), and the one at which a loose reduction stops, the half step
    included. Two iterations form eight quotients of sums; each sum carries at most 1e-12 (the
    apply's bound) times its cancellation, for which 1e4 is allowed: 1e-7 in all."""
    print(f"[gpu] BiCGSTAB steps {grid} Q{degree} {kind} precond {precond}", flush=True)
    nx, ny, nz = grid
    cfg = pkg.make_config(nx=nx, ny=ny, nz=nz, degree=degree, alpha=3.0, **KINDS[kind])
    rng = np.random.default_rng(13)
    kappa = np.exp(rng.normal(size=pkg.ncells(cfg) * (3 if cfg.kappa_per_cell == 2 else 1))) if cfg.kappa_per_cell else None
    go, o = pkg.GridOperator(cfg, kappa), of.Oracle(cfg, kappa)
    b, x0 = rng.uniform(-1, 1, go.N), rng.uniform(-1, 1, go.N)
    for maxit, reduction in ((1, 1e-14), (2, 1e-14), (50, 0.7), (50, 0.3)):
        zd, rd = go.vector(x0), go.vector(b)
        res = go.solve(zd, rd, method=pkg.SOLVER_BICGSTAB, precond=precond, reduction=reduction, maxit=maxit)
        z_ref, _, ref = o.solve(b, x0, method=pkg.SOLVER_BICGSTAB, precond=precond, reduction=reduction, maxit=maxit)
        if res["iterations"] > 2:
            continue  # rounding has grown past what two iterations bound
        assert res["iterations"] == ref["iterations"]
        z, r = zd.download(), rd.download()
        assert np.linalg.norm(z - z_ref) <= 1e-7 * np.linalg.norm(z_ref)
        # the returned defect is that of the returned iterate
        assert np.linalg.norm(r - (b - o.jacobian_apply(z))) <= 1e-10 * np.linalg.norm(b - o.jacobian_apply(x0))
