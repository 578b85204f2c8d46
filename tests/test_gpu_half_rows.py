"""The half-row kernels of level 0 (two wavefronts a leaf, two leaves a
workgroup; four a reduction block) where the last workgroup is not full: W-cycle
and PCG against the CPU oracle, the maximum of its rounding as in the tests of
the whole path (1e-5 relative L2), at leaf counts of every remainder by 4."""
import numpy as np
import pytest

import oracle as O
import uaamg_amd as U

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.linalg.norm(a.astype(np.float64) - b) / max(np.linalg.norm(b.astype(np.float64)), 1e-300))


@pytest.mark.parametrize("config,n,left", [(0, 24, 3), (0, 33, 2), (3, 47, 0), (3, 36, 1)])
def test_half_rows_at_remainders(hip_available, monkeypatch, config, n, left):
    monkeypatch.setenv("UAAMG_BLOCK0_LEAVES", "0")
    s = U.Scene(config, n, seed=n)
    lap = U.LaplacianWithLevel(s.phi, s.weights, dt=1.0, dx=s.dx)
    leaves = lap.level_info(0)["nleaf_dof"]
    print(f"[case] config {config}, {n}^3: {leaves} leaves", flush=True)
    assert leaves % 4 == left
    orc = O.OraclePoisson(s.phi, s.weights, 1.0, s.dx)
    b = orc.build_rhs(s.weights, s.vx, s.vy, s.vz)
    solver = U.PoissonSolver(lap)
    assert _rel(solver.precondition(b), orc.precondition(b, solver.mSmoother)) <= 1e-5
    x = lap.getZeroVectorGrid()
    st = solver.solveMultigridPCG(x, b)
    st_o, it_o, xo = orc.solve_pcg(b, smoother=solver.mSmoother)
    assert (st, abs(solver.mIterationTaken - it_o) <= 1) == (U.SUCCESS, True) and st_o == 0
    assert _rel(x, xo) <= 1e-5
