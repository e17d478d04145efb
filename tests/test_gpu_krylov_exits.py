"""What the device Krylov loops leave behind when they end early."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid,degree", [((2, 1, 1), 1), ((13, 11, 9), 2), ((40, 40, 40), 2), ((200, 200, 1), 2)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else f"Q{v}")
def test_bicgstab_abort_leaves_x_and_r(pkg, grid, degree):
    """rt.v below dune-istl's EPSILON (1e-80) ends the first half step before anything is updated:
    x keeps its bits and r is the defect of x, from one workgroup to all 1024 of the update, with
    alpha formed by every workgroup (up to 2048 partials of rt.v) and by a launch of its own
    (200x200x1: 2500). kappa = 1e-60: rt.v = r.Jr is about 1e-60 r.r, whose 1e-40 to 1e-35 is no breakdown."""
    print(f"[gpu] BiCGSTAB abort {grid} Q{degree}", flush=True)
    nx, ny, nz = grid
    cfg = pkg.make_config(nx=nx, ny=ny, nz=nz, degree=degree, alpha=3.0, kappa0=1e-60, b=(1e-60, 0.0, 0.0))
    go = pkg.GridOperator(cfg)
    b = 1e-20 * np.random.default_rng(31).uniform(0.5, 1.0, go.N)
    xd, rd = go.vector(), go.vector()
    for _ in range(5):
        xd.zero()
        rd.upload(b)
        with pytest.raises(pkg.PdelabError, match="EPSILON"):
            go.solve(xd, rd, method=pkg.SOLVER_BICGSTAB, precond=0, reduction=1e-10, maxit=3)
        assert np.array_equal(rd.download(), b)
        assert not xd.download().any()
