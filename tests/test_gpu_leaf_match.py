"""Leaf matching on the device (right-hand side, pressure gradient) against the
tables matched on the host: leaves in any order with some missing, on both
sides of the origin, and grids of one leaf or none; and the grids that are refused
(an origin that is no multiple of 8, one that comes twice), whichever comes
first, with nothing written."""
import numpy as np
import pytest

import uaamg_amd as U

pytestmark = pytest.mark.gpu


def _shift(g, by):
    return U.Grid(g.origins + np.int32(by), g.values, g.active, g.background)


def _some(g, seed, keep):
    p = np.random.default_rng(seed).permutation(g.origins.shape[0])[:keep]
    return U.Grid(g.origins[p].copy(), g.values[p].copy(), None, (0.25, 0.25, 0.25))


@pytest.mark.parametrize("by", [0, -24])
@pytest.mark.parametrize("keep", [0, 1, 17, 10**6])
def test_matches_as_on_the_host(hip_available, by, keep):
    import torch
    s = U.Scene(0, 33, seed=2)
    print(f"[case] shift {by}, {keep} leaves kept", flush=True)
    phi, w = _shift(s.phi, by), _shift(s.weights, by)
    v = [_some(_shift(g, by), 5 + c, keep) for c, g in enumerate((s.vx, s.vy, s.vz))]
    lap = U.LaplacianWithLevel(phi, w, dt=1.0, dx=s.dx)
    out = torch.full((lap.mNumDof,), float("nan"), device="cuda:0")
    lap.createPressurePoissonRightHandSide_device(out.data_ptr(), w, *v)
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy(), lap.createPressurePoissonRightHandSide(w, *v))


@pytest.mark.parametrize("grid", [0, 1, 3])
@pytest.mark.parametrize("kind", ["misaligned", "duplicate"])
def test_refused_origins(hip_available, grid, kind):
    import torch
    s = U.Scene(0, 33, seed=2)
    print(f"[case] grid {grid} {kind}", flush=True)
    lap = U.LaplacianWithLevel(s.phi, s.weights, dt=1.0, dx=s.dx)
    g = [s.weights, s.vx, s.vy, s.vz]
    org = g[grid].origins.copy()
    org[-1] = org[0] if kind == "duplicate" else org[-1] + 1
    bad = U.Grid(org, g[grid].values, g[grid].active, g[grid].background)
    text = "duplicate" if kind == "duplicate" else "multiple of 8"
    out = torch.full((lap.mNumDof,), 7.0, device="cuda:0")
    with pytest.raises(Exception, match=text):
        lap.createPressurePoissonRightHandSide_device(out.data_ptr(), *(g[:grid] + [bad] + g[grid + 1:]))
    torch.cuda.synchronize()
    assert bool((out == 7.0).all())
    p = torch.zeros(lap.mNumDof, device="cuda:0")
    vel = g[1:]
    w = g[0]
    if grid:
        vel = vel[:grid - 1] + [bad] + vel[grid:]
    else:
        w = bad
    with pytest.raises(Exception, match=text):
        lap.apply_pressure_gradient_device(p.data_ptr(), s.phi, w, None, vel, dt=0.1, friction=0.0)
    # the handle works on
    lap.createPressurePoissonRightHandSide_device(out.data_ptr(), *g)
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy(), lap.createPressurePoissonRightHandSide(*g))
