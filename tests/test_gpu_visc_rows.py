"""The viscosity level above the coarsest as rows: its visits in one launch
(with the coarsest solve inside) equal the per-pass launches bit for bit, since
every value is formed by the same terms in the same order. The sizes cover a
two-level hierarchy (the whole W-cycle in one launch), coarsest systems of two,
four and eight rows per thread, levels from a few thousand rows to near the most
the kernel takes, BF16 level vectors, and edges that are no multiple of the leaf.
"""
import numpy as np
import pytest

import uaamg_amd as U

pytestmark = pytest.mark.gpu

def _say(*a):
    print(*a, flush=True)


def _run(s, precision):
    lw = U.L_with_level(s.viscosity, s.liquid, s.solid, s.dt, s.rho, s.dx, precision=precision)
    solver = U.simd_viscosity3d(lw, s.velocity)
    z = solver.precondition(solver.m_rhs.data)
    x = lw.get_zero_vec()
    solver.pcg_solve(x, 1e-6)
    return lw, z, x.data, solver.m_iteration


@pytest.mark.parametrize("config,n,precision", [(0, 17, 0), (0, 20, 0), (0, 23, 0), (0, 28, 0), (0, 23, 1), (0, 33, 0),
                                                (0, 33, 1), (3, 41, 0), (0, 47, 0), (3, 57, 1), (0, 60, 0)])
def test_row_visits_equal_pass_launches(hip_available, monkeypatch, config, n, precision):
    s = U.ViscScene(config, n, seed=n, mu=3.0)
    _say(f"[case] config {config}, {n}^3, precision {precision}")
    out = {}
    for rows in ("1", "0"):
        monkeypatch.setenv("UAAMG_VROWS", rows)
        out[rows] = _run(s, precision)
    lw, z, x, it = out["1"]
    _, z0, x0, it0 = out["0"]
    levels = [lw.level_ndof(l) for l in range(lw.nlevels)]
    _say(f"  levels {levels}, iterations {it}")
    assert np.array_equal(z, z0)
    assert it == it0 and np.array_equal(x, x0)
    assert np.isfinite(x).all()
