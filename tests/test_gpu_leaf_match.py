"""Leaf matching on the device: the right-hand side against the tables matched
on the host, the pressure gradient against the oracle, with leaves in any order
and some missing, on both sides of the origin, grids of one leaf or none, and
grids that share their leaves or their order of them; and the grids that are
refused (an origin that is no multiple of 8, one that comes twice), whichever
comes first, with nothing written."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
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


def _part(g, p, bg=None):
    """leaves p of a grid, in that order"""
    act = None if g.active is None else np.ascontiguousarray(g.active[p])
    return U.Grid(np.ascontiguousarray(g.origins[p]), np.ascontiguousarray(g.values[p]), act,
                  g.background if bg is None else bg)


def _inputs(s, by, order, keep):
    """phi, weights, a solid velocity and three velocities of a scene moved by `by`, `keep` leaves of each:
    every grid in an order of its own, or all in one"""
    rng = np.random.default_rng(11)
    solid = U.Grid(s.weights.origins.copy(), rng.uniform(-1, 1, s.weights.values.shape).astype(np.float32), None,
                   (0.5, -0.25, 0.125))
    out, p = [], None
    for k, g in enumerate((s.phi, s.weights, solid, s.vx, s.vy, s.vz)):
        if p is None or order == "own":
            p = rng.permutation(g.origins.shape[0])[:keep]
        out.append(_part(_shift(g, by), p, (0.75, 0.5, 0.25) if k == 1 else None))
    return out


@pytest.mark.parametrize("on_dev", [False, True])
@pytest.mark.parametrize("by", [0, -24])
@pytest.mark.parametrize("order,keep", [("own", 10**6), ("own", 60), ("one", 60), ("own", 1)])
def test_gradient_equals_oracle(hip_available, order, keep, by, on_dev):
    import torch
    s = U.Scene(0, 33, seed=2)
    print(f"[case] gradient, {order} order, {keep} leaves kept, shift {by}, values on device {on_dev}", flush=True)
    assert len({g.origins.shape[0] for g in (s.phi, s.weights, s.vx, s.vy, s.vz)}) == 1
    lap = U.LaplacianWithLevel(_shift(s.phi, by), _shift(s.weights, by), dt=1.0, dx=s.dx)
    orc = O.OraclePoisson(_shift(s.phi, by), _shift(s.weights, by), 1.0, s.dx)
    phi, w, solid, *vel = _inputs(s, by, order, keep)
    p = np.random.default_rng(4).uniform(-1, 1, lap.mNumDof).astype(np.float32)
    full = [np.full((g.origins.shape[0], 8), ~np.uint64(0), np.uint64) if g.active is None else g.active for g in vel]
    ref = orc.apply_pressure_gradient(p, phi, w, solid, [(g.origins, a, g.values) for g, a in zip(vel, full)],
                                      dt=0.04, friction=0.35)
    pd = torch.from_numpy(p).to("cuda:0")
    got = lap.apply_pressure_gradient_device(pd.data_ptr(), phi, w, solid, vel, dt=0.04, friction=0.35,
                                             values_on_device=on_dev)
    updated = 0
    for c in range(3):
        for name, a, b in zip(("active", "values", "update", "reflected"), got[c], ref[c]):
            assert np.array_equal(a, b.reshape(a.shape)), f"channel {c}: {name}"
        updated += int(np.unpackbits(got[c][0].view(np.uint8)).sum())
    assert updated > 0 or keep == 1


@pytest.mark.parametrize("on_dev", [0, 1])
@pytest.mark.parametrize("grid", range(6))
@pytest.mark.parametrize("kind", ["misaligned", "duplicate"])
def test_refused_gradient_writes_nothing(hip_available, kind, grid, on_dev):
    import torch
    s = U.Scene(0, 33, seed=2)
    print(f"[case] refused gradient, grid {grid} {kind}, values on device {on_dev}", flush=True)
    lap = U.LaplacianWithLevel(s.phi, s.weights, dt=1.0, dx=s.dx)
    g = _inputs(s, 0, "one", 10**6)
    org = g[grid].origins
    org[-1] = org[0] if kind == "duplicate" else org[-1] + 1
    keep = []

    def place(a):
        keep.append(torch.from_numpy(a).to("cuda:0") if on_dev else a)
        return keep[-1].data_ptr() if on_dev else a.ctypes.data
    st = [x._struct(place(np.ascontiguousarray(x.values, dtype=np.float32))) for x in g[:3]]
    p = torch.ones(lap.mNumDof, device="cuda:0")
    ch = (U._FaceChannel * 3)()
    act = [np.full((x.origins.shape[0], 8), 0x1234567 + c, np.uint64) for c, x in enumerate(g[3:])]
    n = len(keep)
    for c, x in enumerate(g[3:]):
        ch[c].nleaf, ch[c].origins, ch[c].active = x.origins.shape[0], x.origins.ctypes.data, act[c].ctypes.data
        for k, field in enumerate(("values", "update", "reflected")):
            setattr(ch[c], field, place(np.full((x.origins.shape[0], 512), 1.0 + c + 10 * k, np.float32)))
    rc = U.lib().uaamg_poisson_apply_pressure_gradient_device(
        lap._h, C.c_void_p(p.data_ptr()), C.byref(st[0]), C.byref(st[1]), C.byref(st[2]), ch, 0.1, 0.0, on_dev)
    text = U.lib().uaamg_last_error()
    torch.cuda.synchronize()
    assert rc < 0 and (b"duplicate" if kind == "duplicate" else b"multiple of 8") in text
    name = [b"liquid_phi", b"face_weights", b"solid_velocity", b"velocity channel"][min(grid, 3)]
    assert text.startswith(name)
    for c in range(3):
        assert (act[c] == np.uint64(0x1234567 + c)).all(), f"channel {c}: active"
        for k in range(3):
            a = keep[n + 3 * c + k]
            assert bool((a == 1.0 + c + 10 * k).all()), f"channel {c}: output {k}"
