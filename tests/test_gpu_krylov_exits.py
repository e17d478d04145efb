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


@pytest.mark.parametrize("precond", [0, 1, 2], ids=["none", "point", "block"])
def test_refused_cg_leaves_the_defect(pkg, precond):
    """CG is refused with a velocity field: x keeps its bits and r is the defect of x, in which
    dune-istl's solvers take and leave it."""
    print(f"[gpu] refused CG precond {precond}", flush=True)
    cfg = pkg.make_config(nx=5, ny=4, nz=3, degree=2, alpha=3.0)
    go = pkg.GridOperator(cfg)
    rng = np.random.default_rng(32)
    m = pkg.quadrature_points(cfg)
    go.set_velocity_field(rng.normal(size=60 * 3 * m ** 3), rng.normal(size=(6 * 12 + 5 * 15 + 20 * 4) * m ** 2))
    b, x0 = rng.uniform(-1, 1, go.N), rng.uniform(-1, 1, go.N)
    xd, rd, jx = go.vector(x0), go.vector(b), go.vector()
    go.operator_apply(xd, jx)
    with pytest.raises(pkg.PdelabError, match="CG"):
        go.solve(xd, rd, method=pkg.SOLVER_CG, precond=precond, reduction=1e-10, maxit=5)
    assert np.array_equal(xd.download(), x0)
    # one multiply-add per entry, fused or not: two roundings of |b| + |Jx|
    assert np.all(np.abs(rd.download() - (b - jx.download())) <= 2.3e-16 * (np.abs(b) + np.abs(jx.download())))
