"""The device Krylov loops where their kernels change with the length of the vectors."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


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
