"""The device Krylov loops against the same recurrences in numpy, with the operator and the
preconditioner of the library's own (elsewhere tested) entry points: where each run stops, half steps
included, and the kernels that only long vectors or many partials reach.

Tolerance: a few iterations form up to eight quotients of sums; each sum carries at most 1e-12 (the
apply's bound) times its cancellation, for which 1e4 is allowed: 1e-7 in all.
"""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
RTOL = 1e-7

KINDS = {
    "const": dict(),
    "conv": dict(b=(1.0, 0.5, 0.25), kappa0=1e-2),
    "cells_conv": dict(kappa_per_cell=1, b=(-0.5, 1.0, 2.0)),
}


def setup(pkg, grid, degree, kind, precond):
    """The handle, z -> J z and z -> W^{-1} z as functions of numpy arrays."""
    nx, ny, nz = grid
    cfg = pkg.make_config(nx=nx, ny=ny, nz=nz, degree=degree, alpha=3.0, **KINDS[kind])
    kappa = np.exp(0.5 * np.random.default_rng(41).normal(size=pkg.ncells(cfg))) if cfg.kappa_per_cell else None
    go = pkg.GridOperator(cfg, kappa)
    zd, yd = go.vector(), go.vector()

    def through(call):
        def f(v):
            zd.upload(v)
            yd.zero()
            call(zd, yd)
            return yd.download()
        return f

    prec = [lambda v: v.copy(), None, through(go.block_jacobi_apply)][precond]
    if precond == 1:
        go.point_diagonal(yd)
        d = yd.download()
        prec = lambda v: v / d  # noqa: E731
    return go, through(go.operator_apply), prec


def bicgstab(apply, prec, b, x0, halves):
    """x, r and the defect after each of so many half steps (dune-istl's BiCGSTABSolver::apply)."""
    x, r = x0.copy(), b - apply(x0)
    rt, out = r.copy(), []
    rho = alpha = omega = 1.0
    p = v = None
    for half in range(1, halves + 1):
        if half % 2:
            rho_new = rt @ r
            p = r.copy() if p is None else r + (rho_new / rho) * (alpha / omega) * (p - omega * v)
            y = prec(p)
            v = apply(y)
            alpha = rho_new / (rt @ v)
            x += alpha * y
            r -= alpha * v
            rho = rho_new
        else:
            y = prec(r)
            t = apply(y)
            omega = (t @ r) / (t @ t)
            x += omega * y
            r -= omega * t
        out.append((x.copy(), r.copy(), np.linalg.norm(r)))
    return out


def check(go, pkg, apply, b, x0, want, **solve):
    xd, rd = go.vector(x0), go.vector(b)
    res = go.solve(xd, rd, method=pkg.SOLVER_BICGSTAB, **solve)
    x, r, _ = want
    assert np.linalg.norm(xd.download() - x) <= RTOL * np.linalg.norm(x)
    assert np.linalg.norm(rd.download() - r) <= RTOL * np.linalg.norm(b - apply(x0))
    xd.free()
    rd.free()
    return res


@pytest.mark.parametrize("precond", [0, 1, 2], ids=["none", "point", "block"])
@pytest.mark.parametrize("degree", [1, 2, 3])
def test_bicgstab_stops_at_each_half_step(pkg, degree, precond):
    """A reduction between two defects of the recurrence stops the loop at that very half step (it may
    not run on), with x and r of that half step. From a random right-hand side the second half steps
    bring the defect down, from one close to an eigenvector of J W^{-1} (a power iteration) the first."""
    met = set()
    for kind in ("conv", "cells_conv"):
        print(f"[gpu] BiCGSTAB half steps Q{degree} {kind} precond {precond}", flush=True)
        go, apply, prec = setup(pkg, (13, 11, 9), degree, kind, precond)
        rng = np.random.default_rng(42)
        v = rng.uniform(-1, 1, go.N)
        for _ in range(40):
            v = apply(prec(v))
            v /= np.linalg.norm(v)
        for b, x0 in ((rng.uniform(-1, 1, go.N), rng.uniform(-1, 1, go.N)), (v, np.zeros(go.N))):
            lowest = def0 = np.linalg.norm(b - apply(x0))
            for k, want in enumerate(bicgstab(apply, prec, b, x0, 4), 1):
                if want[2] < 0.95 * lowest:
                    res = check(go, pkg, apply, b, x0, want, precond=precond, reduction=np.sqrt(want[2] * lowest) / def0, maxit=50)
                    assert res["converged"] and res["iterations"] == (k + 1) // 2
                    met.add(k % 2)
                lowest = min(lowest, want[2])
    assert met == {0, 1}


@pytest.mark.parametrize("grid,degree,kind,precond", [
    ((200, 200, 1), 2, "conv", 0), ((200, 200, 1), 2, "conv", 1),  # 2500 partials of the apply's dots
    ((61, 61, 60), 2, "conv", 1), ((61, 61, 60), 2, "conv", 0),    # five vectors do not fit the memory-side cache
    ((46, 46, 45), 3, "cells_conv", 1)],
    ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_bicgstab_sizes(pkg, grid, degree, kind, precond):
    """Two iterations where alpha and omega come from launches of their own, and of long vectors."""
    print(f"[gpu] BiCGSTAB sizes {grid} Q{degree} {kind} precond {precond}", flush=True)
    go, apply, prec = setup(pkg, grid, degree, kind, precond)
    rng = np.random.default_rng(43)
    b, x0 = rng.uniform(-1, 1, go.N), rng.uniform(-1, 1, go.N)
    want = bicgstab(apply, prec, b, x0, 4)[-1]
    assert check(go, pkg, apply, b, x0, want, precond=precond, reduction=1e-14, maxit=2)["iterations"] == 2


@pytest.mark.parametrize("precond", [0, 1], ids=["none", "point"])
def test_cg_beyond_the_cache(pkg, precond):
    """Three CG iterations of 10 million unknowns, of which not even three vectors fit the memory-side cache."""
    print(f"[gpu] CG beyond the cache precond {precond}", flush=True)
    go, apply, prec = setup(pkg, (72, 72, 72), 2, "const", precond)
    rng = np.random.default_rng(44)
    b = rng.uniform(-1, 1, go.N)
    x, r = np.zeros(go.N), b.copy()
    p = prec(r)
    rho = p @ r
    for _ in range(3):
        q = apply(p)
        lam = rho / (p @ q)
        x += lam * p
        r -= lam * q
        z = prec(r)
        rho, old = z @ r, rho
        p = z + rho / old * p
    xd, rd = go.vector(), go.vector(b)
    assert go.solve(xd, rd, method=pkg.SOLVER_CG, precond=precond, reduction=1e-14, maxit=3)["iterations"] == 3
    assert np.linalg.norm(xd.download() - x) <= RTOL * np.linalg.norm(x)
    assert np.linalg.norm(rd.download() - r) <= RTOL * np.linalg.norm(b)


def mixed_block_jacobi(pkg, n, degree):
    """The handle, the solution of the mixed-precision CG with block Jacobi to 1e-8 and its result."""
    go = pkg.GridOperator(pkg.make_config(n=n, degree=degree, alpha=3.0, problem=pkg.PROBLEM_CONSTANT, f0=1.0))
    x = go.vector()
    return go, x, go.solve_mixed(x, method=pkg.SOLVER_CG, precond=2, outer_reduction=1e-8)


def test_mixed_block_jacobi_of_long_vectors(pkg):
    """Mixed-precision CG with the block Jacobi of a constant Q3 operator above 2^23 unknowns, where the FP32
    p update applies W^{-1} to r again: the FP64 defect of the solution is at the reduction asked, and the
    iterations are those of the grid just below, which stores W^{-1} r, times the ratio of the sizes
    (CG's count grows with n) within a tenth."""
    print("[gpu] mixed CG, block Jacobi, 52^3 Q3", flush=True)
    go, x, res = mixed_block_jacobi(pkg, 52, 3)
    assert go.N > 1 << 23
    r = go.vector()
    go.residual(x, r)
    x.zero()
    def0 = go.vector()
    go.residual(x, def0)
    assert res["converged"] and go.norm(r) <= 1.0001e-8 * go.norm(def0)
    below, _, ref = mixed_block_jacobi(pkg, 50, 3)
    assert below.N < 1 << 23
    assert abs(res["inner_iterations"] / (52 / 50 * ref["inner_iterations"]) - 1) <= 0.1


def test_block_jacobi_time_of_long_vectors(pkg):
    """Q2 above 2^23 unknowns: W^{-1} r of a constant operator is stored, not formed twice. Time per
    mixed-precision iteration against that of the same operator as cell-wise kappa = 1, whose blocks
    are read from memory: 0.76 where it is stored, 0.84 where it is formed twice; 0.81 is the line."""
    print("[gpu] block Jacobi times, 96^3 Q2", flush=True)
    times = []
    for kw in (dict(), dict(kappa=np.ones(96 ** 3))):
        cfg = pkg.make_config(n=96, degree=2, alpha=3.0, problem=pkg.PROBLEM_CONSTANT, f0=1.0, kappa_per_cell=bool(kw))
        go = pkg.GridOperator(cfg, **kw)
        x, best = go.vector(), np.inf
        for _ in range(4):
            x.zero()
            go.synchronize()
            t = time.perf_counter()
            res = go.solve_mixed(x, method=pkg.SOLVER_CG, precond=2, outer_reduction=1e-13, inner_maxit=200)
            best = min(best, (time.perf_counter() - t) / res["inner_iterations"])
        times.append(best)
        x.free()
        go.close()
    print(f"[gpu] constant {1e6 * times[0]:.0f} us, cell-wise {1e6 * times[1]:.0f} us", flush=True)
    assert times[0] <= 0.81 * times[1]
