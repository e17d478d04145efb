"""The device CG loop against the same recurrences in numpy, with the operator and the
preconditioner of the library's own (elsewhere tested) entry points: the iterate and the defect
after a few iterations and at a loose reduction. The sizes are those where the loop's kernels
change: vectors shorter than a workgroup, sums finished by the vector kernels or by launches of
their own (2048 partials, 2^23 elements), block Jacobi applied again instead of stored.

Tolerance: three iterations form six quotients of sums; each sum carries at most 1e-12 (the
apply's bound) times its cancellation, for which 1e4 is allowed: 1e-7 in all.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [((1, 1, 1), 1), ((1, 1, 3), 2), ((5, 3, 2), 3), ((13, 11, 9), 2), ((33, 35, 31), 1), ((68, 69, 67), 2),
         ((53, 52, 51), 3), ((103, 102, 101), 1)]


def reference(apply, prec, b, x0, maxit, reduction):
    x, r = x0.copy(), b - apply(x0)
    def0 = np.linalg.norm(r)
    p = prec(r)
    rho = p @ r
    for it in range(1, maxit + 1):
        q = apply(p)
        lam = rho / (p @ q)
        x += lam * p
        r -= lam * q
        if np.linalg.norm(r) < reduction * def0:
            break
        z = prec(r)
        rho, old = z @ r, rho
        p = z + rho / old * p
    return x, r, it


@pytest.mark.parametrize("precond", [0, 1, 2], ids=["none", "point", "block"])
@pytest.mark.parametrize("kind", ["const", "cells"])
@pytest.mark.parametrize("grid,degree", CASES, ids=lambda g: "x".join(map(str, g)) if isinstance(g, tuple) else f"Q{g}")
def test_cg_first_iterations(pkg, grid, degree, kind, precond):
    print(f"[gpu] CG steps {grid} Q{degree} {kind} precond {precond}", flush=True)
    nx, ny, nz = grid
    cells = kind == "cells"
    if cells and nx * ny * nz > 1_000_000:
        pytest.skip("the constant operator covers this size")
    cfg = pkg.make_config(nx=nx, ny=ny, nz=nz, degree=degree, alpha=3.0, kappa_per_cell=cells)
    rng = np.random.default_rng(17)
    kappa = np.exp(0.5 * rng.normal(size=pkg.ncells(cfg))) if cells else None
    go = pkg.GridOperator(cfg, kappa)
    zd, yd = go.vector(), go.vector()

    def through(call):
        def f(v):
            zd.upload(v)
            yd.zero()
            call(zd, yd)
            return yd.download()
        return f

    apply = through(go.operator_apply)
    prec = [lambda v: v.copy(), None, through(go.block_jacobi_apply)][precond]
    if precond == 1:
        go.point_diagonal(yd)
        d = yd.download()
        prec = lambda v: v / d  # noqa: E731
    b, x0 = rng.uniform(-1, 1, go.N), rng.uniform(-1, 1, go.N)
    for maxit, reduction in ((1, 1e-14), (3, 1e-14), (3, 0.9)):
        xd, rd = go.vector(x0), go.vector(b)
        res = go.solve(xd, rd, method=pkg.SOLVER_CG, precond=precond, reduction=reduction, maxit=maxit)
        x, r, it = reference(apply, prec, b, x0, maxit, reduction)
        if np.linalg.norm(r) < 1e-7 * np.linalg.norm(b):
            continue  # exact after fewer steps than asked: nothing but rounding is left
        assert res["iterations"] == it
        assert np.linalg.norm(xd.download() - x) <= 1e-7 * np.linalg.norm(x)
        assert np.linalg.norm(rd.download() - r) <= 1e-7 * np.linalg.norm(b - apply(x0))
