"""Right-hand sides of every magnitude: the solvers are linear, so a right-hand
side multiplied by a power of two has the solution multiplied by it, down to
where the coarsest solve's own stopping rule (||r||^2 < FLT_MIN, Eigen's) ends
it early. Small ones are what a liquid nearly at rest or a good starting guess
give, and the second visits of a deep W-cycle hand on far smaller ones."""
import numpy as np
import pytest

import oracle as O
import uaamg_amd as U

pytestmark = pytest.mark.gpu

FLT_MIN_ROOT = float(np.sqrt(np.finfo(np.float32).tiny))


def _rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(np.asarray(b, np.float64)))


def _check_coarsest(solve, ndof, matvec, lowest):
    """solve(2^k b) for ||b||_inf = 1. Equal to 2^k solve(b) bit for bit where the stopping rule is the
    relative one (||b|| FLT_EPSILON above FLT_MIN's root); below, the residual is at most the larger of
    the unscaled solve's share and FLT_MIN's root, beside the rounding of r in ten steps (1e-6 ||b||)."""
    b = np.random.default_rng(5).uniform(-1, 1, ndof).astype(np.float32)
    unit = solve(b)
    norm = float(np.linalg.norm(b.astype(np.float64)))
    share = float(np.linalg.norm(b - matvec(unit.astype(np.float64)))) / norm
    assert np.isfinite(unit).all() and share < 1
    for k in [45, 20, *range(0, lowest, -4)]:
        s = 2.0 ** k
        x = solve((b * np.float32(s)).astype(np.float32))
        assert np.isfinite(x).all(), f"2^{k}"
        if s * norm * np.finfo(np.float32).eps > 2 * FLT_MIN_ROOT:
            assert np.array_equal(x, unit * np.float32(s)), f"2^{k}"
        else:
            left = float(np.linalg.norm(s * b.astype(np.float64) - matvec(x.astype(np.float64))))
            assert left <= max(1.01 * share * s * norm, FLT_MIN_ROOT) + 1e-6 * s * norm, f"2^{k}"


# one level; three levels; a coarsest system of more than 2048 rows; an early-stopping one of few rows
@pytest.mark.parametrize("config,n", [(3, 16), (0, 48), (0, 72), (0, 6)])
def test_coarsest_solve(hip_available, config, n):
    s = U.Scene(config, n, seed=0)
    lap = U.LaplacianWithLevel(s.phi, s.weights, dt=1.0, dx=s.dx)
    last = lap.nlevels - 1
    ndof = lap.level_ndof(last)
    print(f"[case] config {config}, {n}^3: {ndof} rows", flush=True)
    i, j, v = lap.getTriplets(last)

    def matvec(x):
        return np.bincount(i, weights=v.astype(np.float64) * x[j], minlength=ndof)
    _check_coarsest(lap.coarsest_solve, ndof, matvec, -72)


# D^-1 of about 1, 1e-4 and 1e-6; coarsest systems of two, four and eight rows per thread
@pytest.mark.parametrize("n,mu", [(33, 1.0), (33, 1e5), (23, 1e7), (28, 1e5)])
def test_viscosity_coarsest_solve(hip_available, n, mu):
    s = U.ViscScene(0, n, seed=n, mu=mu)
    lw = U.L_with_level(s.viscosity, s.liquid, s.solid, s.dt, s.rho, s.dx)
    last = lw.nlevels - 1
    ndof = lw.level_ndof(last)
    print(f"[case] viscosity {n}^3, mu {mu:g}: {ndof} rows", flush=True)
    ptr, col, val = lw.level_matrix(last)
    row = np.repeat(np.arange(ndof), np.diff(ptr))

    def matvec(x):
        return np.bincount(row, weights=val.astype(np.float64) * x[col], minlength=ndof)
    _check_coarsest(lw.solve_exact, ndof, matvec, -72)


def _poisson(config, n, precision=0):
    s = U.Scene(config, n, seed=n)
    lap = U.LaplacianWithLevel(s.phi, s.weights, dt=1.0, dx=s.dx, precision=precision)
    b = lap.createPressurePoissonRightHandSide(s.weights, s.vx, s.vy, s.vz)
    return s, lap, b / np.abs(b).max()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,powers", [(48, (20, 30, 37)), (128, (20, 27, 33)), (256, (17, 27))])
def test_poisson_solve(hip_available, n, powers, precision):
    s, lap, b = _poisson(0, n, precision)
    solver = U.PoissonSolver(lap)

    def solve(b):
        x = lap.getZeroVectorGrid()
        return solver.solveMultigridPCG(x, b), solver.mIterationTaken, x
    st, it, unit = solve(b)
    z = solver.precondition(b)
    orc = O.OraclePoisson(s.phi, s.weights, 1.0, s.dx) if n == 48 and precision == 0 else None
    print(f"[case] {n}^3, precision {precision}, {lap.nlevels} levels: {it} iterations", flush=True)
    assert st == U.SUCCESS
    for k in powers:
        bs = (b * np.float32(2.0 ** -k)).astype(np.float32)
        st, its, x = solve(bs)
        print(f"  2^-{k}: status {st}, {its} iterations", flush=True)
        assert np.isfinite(x).all() and st == U.SUCCESS and abs(its - it) <= 1, f"2^-{k}"
        assert _rel(x * 2.0 ** k, unit) <= 1e-5, f"2^-{k}"
        assert _rel(solver.precondition(bs) * 2.0 ** k, z) <= 1e-5, f"2^-{k}"
        if orc is not None:
            st_o, it_o, xo = orc.solve_pcg(bs)
            assert st_o == 0 and abs(its - it_o) <= 1 and _rel(x, xo) <= 1e-5, f"2^-{k}"


@pytest.mark.parametrize("precision", [0, 1])
def test_poisson_batch(hip_available, precision):
    """Problems of unlike magnitude in one batch, each as it is alone."""
    import torch
    parts = [(48, 0), (48, 30), (96, 27), (33, 37)]
    print(f"[case] batch, precision {precision}", flush=True)
    problems, bs, alone = [], [], []
    for n, k in parts:
        s, lap, b = _poisson(0, n, precision)
        b = torch.from_numpy((b * np.float32(2.0 ** -k)).astype(np.float32)).to("cuda:0")
        x = torch.zeros_like(b)
        alone.append((*lap.solve_pcg_device(x.data_ptr(), b.data_ptr()), x))
        problems.append((s.phi, s.weights, 1.0, s.dx))
        bs.append(b)
    xs = [torch.zeros_like(b) for b in bs]
    st, it = U.PoissonBatch(problems, precision=precision).solve_device([x.data_ptr() for x in xs],
                                                                        [b.data_ptr() for b in bs])
    torch.cuda.synchronize()
    for i, (st1, it1, x1) in enumerate(alone):
        assert st[i] == st1 == U.SUCCESS and it[i] == it1, f"problem {i}"
        assert bool(torch.isfinite(xs[i]).all()) and torch.equal(xs[i], x1), f"problem {i}"


@pytest.mark.parametrize("rows", ["1", "0"])
@pytest.mark.parametrize("precision", [0, 1])
def test_viscosity_cycle(hip_available, monkeypatch, precision, rows):
    """D^-1 of about 1e-4: W-cycles of scaled right-hand sides, with the coarsest solve inside the level
    above it and as its own launch; finite where the coarsest solve ends early."""
    monkeypatch.setenv("UAAMG_VROWS", rows)
    s = U.ViscScene(0, 33, seed=33, mu=1e5)
    lw = U.L_with_level(s.viscosity, s.liquid, s.solid, s.dt, s.rho, s.dx, precision=precision)
    solver = U.simd_viscosity3d(lw, s.velocity)
    b = solver.m_rhs.data / np.abs(solver.m_rhs.data).max()
    unit = solver.precondition(b)
    print(f"[case] viscosity W-cycle, precision {precision}, rows {rows}", flush=True)
    for k in (20, 30, 40):
        z = solver.precondition((b * np.float32(2.0 ** -k)).astype(np.float32))
        assert np.isfinite(z).all() and _rel(z * 2.0 ** k, unit) <= 1e-5, f"2^-{k}"
    for k in range(50, 66, 3):
        assert np.isfinite(solver.precondition((b * np.float32(2.0 ** -k)).astype(np.float32))).all(), f"2^-{k}"
