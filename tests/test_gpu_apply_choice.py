"""Which kernel an FP64 Q2/Q3 apply takes: the matrix-core, the row and the general kernel against
the oracle on both sides of the lines between them, and the time of the chosen one against the
general kernel's.

Tolerance of the results: 1e-12 relative (2-norm), the operator's. The times' bounds lie between
those measured with the right and with the wrong choice.
"""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
RTOL = 1e-12

KINDS = {
    "const": dict(),
    "conv": dict(b=(1.0, 0.5, 0.25), kappa0=1e-2),
    "cells": dict(kappa_per_cell=1),
    "cells_conv": dict(kappa_per_cell=1, b=(-0.5, 1.0, 2.0), c=0.3),
    "cells_off": dict(kappa_per_cell=1, weights=1),
    "tensor": dict(kappa_per_cell=2, lx=2.0, ly=0.5),
}
# cell-wise kappa with convection or weightsOff: 255, 256 and more steps of workgroups, with whole and
# partial chunks of the row kernel; thin planes of 4, 5, 17 and 18 cells past 1024 steps; one and
# two planes of 128^2 cells, whole and partial chunks; wide planes, walked in strips of 128 cells (one
# whole strip and a rest, rows that no workgroup starts with, a plane of one row and a bit)
GENERAL = [(16, 16, 15), (16, 16, 16), (32, 16, 9), (33, 17, 8), (5, 3, 257)]
THIN = [(2, 2, 1024), (2, 2, 1025), (5, 1, 1030), (17, 1, 513), (6, 3, 515)]
FLAT = [(128, 128, 1), (129, 127, 1), (131, 127, 2), (160, 112, 2)]
WIDE = [(257, 5, 8), (300, 9, 8), (272, 3, 9), (1040, 2, 10)]
CASES = ([(g, k) for g in GENERAL for k in ("cells_conv", "cells_off")]
         + [(g, k) for g in THIN for k in ("const", "conv", "cells", "tensor")]
         + [(g, k) for g in FLAT for k in ("const", "conv", "cells", "tensor")]
         + [(g, k) for g in WIDE for k in ("const", "cells")])


def operator(pkg, grid, degree, kind, seed=21):
    nx, ny, nz = grid
    cfg = pkg.make_config(nx=nx, ny=ny, nz=nz, degree=degree, alpha=3.0, problem=pkg.PROBLEM_CONSTANT, f0=1.0, **KINDS[kind])
    n = pkg.ncells(cfg) * (3 if cfg.kappa_per_cell == 2 else 1)
    kappa = np.exp(np.random.default_rng(seed).normal(size=n)) if cfg.kappa_per_cell else None
    return cfg, kappa


def general_operator(pkg, cfg, kappa):
    """A handle whose applies run the general kernel, which every grid can take."""
    os.environ["PDELAB_GPU_APPLY"] = "general"  # read when a handle is created
    try:
        return pkg.GridOperator(cfg, kappa)
    finally:
        del os.environ["PDELAB_GPU_APPLY"]


@pytest.mark.parametrize("degree", [2, 3])
@pytest.mark.parametrize("grid,kind", CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else v)
def test_apply_choice_vs_oracle(pkg, of, grid, kind, degree):
    """y = J z and r += R(x) against the oracle, y += J^T z against the general kernel."""
    print(f"[gpu] apply choice {grid} Q{degree} {kind}", flush=True)
    cfg, kappa = operator(pkg, grid, degree, kind)
    go, o, general = pkg.GridOperator(cfg, kappa), of.Oracle(cfg, kappa), general_operator(pkg, cfg, kappa)
    rng = np.random.default_rng(22)
    z, y0 = rng.uniform(-1, 1, go.N), rng.uniform(-1, 1, go.N)
    zd, yd = go.vector(z), go.vector()
    ref = o.jacobian_apply(z)
    go.operator_apply(zd, yd)
    assert np.linalg.norm(yd.download() - ref) <= RTOL * np.linalg.norm(ref)
    zg, yg = general.vector(z), general.vector(y0)
    general.jacobian_apply_transpose(zg, yg)
    yd.upload(y0)
    go.jacobian_apply_transpose(zd, yd)
    ref = yg.download()
    assert np.linalg.norm(yd.download() - ref) <= RTOL * np.linalg.norm(ref)
    ref = o.residual(z)
    yd.upload(y0)
    go.residual(zd, yd)
    assert np.linalg.norm(yd.download() - y0 - ref) <= RTOL * (np.linalg.norm(ref) + np.linalg.norm(y0))


@pytest.mark.parametrize("grid,degree,kind", [((17, 1, 513), 2, "const"), ((32, 16, 9), 3, "cells"), ((129, 127, 1), 2, "tensor")],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_cg_over_the_choice(pkg, grid, degree, kind):
    """Three CG iterations (the apply with its fused dot) where the row and general kernels take over,
    against the same recurrences in numpy. 1e-7: six quotients of sums, each of at most 1e-12 times
    a cancellation of 1e4."""
    print(f"[gpu] CG over the choice {grid} Q{degree} {kind}", flush=True)
    cfg, kappa = operator(pkg, grid, degree, kind)
    go = pkg.GridOperator(cfg, kappa)
    rng = np.random.default_rng(23)
    b = rng.uniform(-1, 1, go.N)
    zd, yd = go.vector(), go.vector()

    def apply(v):
        zd.upload(v)
        go.operator_apply(zd, yd)
        return yd.download()

    x, r = np.zeros(go.N), b.copy()
    p, rho = r.copy(), b @ b
    for _ in range(3):
        q = apply(p)
        lam = rho / (p @ q)
        x += lam * p
        r -= lam * q
        rho, old = r @ r, rho
        p = r + rho / old * p
    xd, rd = go.vector(), go.vector(b)
    assert go.solve(xd, rd, method=pkg.SOLVER_CG, precond=0, reduction=1e-14, maxit=3)["iterations"] == 3
    assert np.linalg.norm(xd.download() - x) <= 1e-7 * np.linalg.norm(x)
    assert np.linalg.norm(rd.download() - r) <= 1e-7 * np.linalg.norm(b)


# 1.1 where the general kernel is the right choice or close to it; less where the row kernel (0.87 of
# the general kernel's time on the plane of more than 4 GiB, 0.80 on the single plane) is, or the
# matrix-core kernel walking a wide plane in strips (0.67; row after row 1.03)
TIMES = [((64, 64, 64), 2, "cells_off", 1.1), ((64, 64, 64), 2, "cells_conv", 1.1), ((48, 48, 48), 3, "cells_off", 1.1),
         ((2, 2, 8192), 2, "const", 1.1), ((5, 1, 8192), 3, "cells", 1.1), ((17, 1, 8192), 2, "const", 1.1),
         ((512, 512, 1), 2, "const", 0.95), ((4096, 2056, 1), 3, "conv", 0.95), ((2048, 64, 32), 3, "const", 0.85)]


@pytest.mark.parametrize("grid,degree,kind,most", TIMES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_apply_choice_is_not_the_slower_one(pkg, grid, degree, kind, most):
    """The chosen kernel takes at most so much of the general one's time."""
    print(f"[gpu] apply choice, times {grid} Q{degree} {kind}", flush=True)
    cfg, kappa = operator(pkg, grid, degree, kind)
    go, general = pkg.GridOperator(cfg, kappa), general_operator(pkg, cfg, kappa)
    pairs = [(h, h.vector(), h.vector()) for h in (go, general)]
    best = [np.inf, np.inf]
    for _ in range(5):
        for i, (h, z, y) in enumerate(pairs):
            best[i] = min(best[i], h.time_apply(z, y, warmup=3, reps=20))
    print(f"[gpu] chosen {1e3 * best[0]:.1f} us, general {1e3 * best[1]:.1f} us", flush=True)
    assert best[0] <= most * best[1]
