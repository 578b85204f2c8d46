"""Level 0's W-cycle visit as block-visit launches (small problems) equals the
per-sweep kernels bit for bit: W-cycle, solution, status and iterations, from a
two-level hierarchy (the coarsest solve inside level 0's post-visit) to the
largest level 0 that takes it, with edges that are no multiple of the leaf."""
import numpy as np
import pytest

import uaamg_amd as U

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("config,n", [(0, 24), (0, 33), (3, 47), (1, 64), (0, 75)])
@pytest.mark.parametrize("smoother", [0, 1])
def test_block_visits_on_level_0(hip_available, monkeypatch, config, n, smoother):
    s = U.Scene(config, n, seed=n)
    print(f"[case] config {config}, {n}^3, smoother {smoother}", flush=True)
    out = {}
    for most in ("600", "0"):
        monkeypatch.setenv("UAAMG_BLOCK0_LEAVES", most)
        lap = U.LaplacianWithLevel(s.phi, s.weights, dt=1.0, dx=s.dx, smoother=smoother)
        assert lap.kernel_map()[0]["block"] == (lap.level_info(0)["nleaf_dof"] <= int(most))
        b = lap.createPressurePoissonRightHandSide(s.weights, s.vx, s.vy, s.vz)
        solver = U.PoissonSolver(lap)
        solver.mSmoother = smoother
        z = solver.precondition(b)
        x = lap.getZeroVectorGrid()
        out[most] = (z, x, solver.solveMultigridPCG(x, b), solver.mIterationTaken)
    (z, x, st, it), (z0, x0, st0, it0) = out["600"], out["0"]
    assert np.array_equal(z, z0) and np.array_equal(x, x0) and (st, it) == (st0, it0)
