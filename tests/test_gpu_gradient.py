"""GPU parity of the device pressure-gradient update
(uaamg_poisson_apply_pressure_gradient_device, FLIP_vdb.cpp:2571-2667): active
masks, updated velocities, update and reflected grids bit-identical to the
oracle's restatement, for the pressure of an actual solve, with and without a
solid velocity, friction, host- and device-resident values.
"""
import ctypes as C

import numpy as np
import pytest

import oracle as O
import uaamg_amd as U

pytestmark = pytest.mark.gpu


def _say(*a):
    print(*a, flush=True)


def _solid(grid: U.Grid, seed: int) -> U.Grid:
    rng = np.random.default_rng(seed)
    vals = rng.uniform(-1.0, 1.0, size=(grid.origins.shape[0], 512, 3)).astype(np.float32)
    return U.Grid(grid.origins.copy(), vals, None, (0.5, -0.25, 0.125))


@pytest.mark.parametrize("cfg,n,seed", [(0, 32, 0), (1, 48, 1)])
def test_gradient_equals_oracle(hip_available, cfg, n, seed):
    import torch
    dev = torch.device("cuda:0")
    _say(f"[setup] gradient cfg={cfg} n={n} seed={seed}")
    s = U.Scene(cfg, n, seed=seed)
    lap = U.LaplacianWithLevel(s.phi, s.weights, dt=1.0, dx=s.dx)
    orc = O.OraclePoisson(s.phi, s.weights, 1.0, s.dx)
    b = lap.createPressurePoissonRightHandSide(s.weights, s.vx, s.vy, s.vz)
    x = torch.zeros(lap.mNumDof, dtype=torch.float32, device=dev)
    lap.solve_pcg_device(x.data_ptr(), torch.from_numpy(b).to(dev).data_ptr())
    torch.cuda.synchronize()
    p = x.cpu().numpy()
    vel = [s.vx, s.vy, s.vz]
    velo = [(g.origins, g.active, g.values) for g in vel]
    for solid, friction in ((None, 0.0), (_solid(s.weights, seed + 5), 0.35)):
        ref = orc.apply_pressure_gradient(p, s.phi, s.weights, solid, velo, dt=0.04, friction=friction)
        for on_dev in (False, True):
            got = lap.apply_pressure_gradient_device(x.data_ptr(), s.phi, s.weights, solid, vel, dt=0.04,
                                                     friction=friction, values_on_device=on_dev)
            for c in range(3):
                ra, rv, ru, rr = ref[c]
                ga, gv, gu, gr = got[c]
                tag = f"solid={solid is not None} device={on_dev} channel {c}"
                assert np.array_equal(ga, ra), tag + ": active"
                assert np.array_equal(gv, rv.reshape(gv.shape)), tag + ": values"
                assert np.array_equal(gu, ru.reshape(gu.shape)), tag + ": update"
                assert np.array_equal(gr, rr.reshape(gr.shape)), tag + ": reflected"
            on = sum(int(np.unpackbits(ga.view(np.uint8)).sum()) for ga, _, _, _ in got)
            _say(f"  solid={solid is not None} device={on_dev}: {on} faces updated")


def _channels(arrays):
    """[(origins, active, values)] as the C struct; values: a numpy array or a device tensor"""
    ch = (U._FaceChannel * 3)()
    for c, a in enumerate(arrays):
        if a is None:
            continue
        org, act, val = a
        ch[c].nleaf = org.shape[0]
        ch[c].origins = org.ctypes.data
        ch[c].active = act.ctypes.data
        ch[c].values = val.ctypes.data if isinstance(val, np.ndarray) else val.data_ptr()
    return ch


@pytest.mark.parametrize("on_dev", [0, 1])
@pytest.mark.parametrize("shift", [0, 2])
def test_channels_that_share_masks(hip_available, on_dev, shift):
    """One active array for several channels (or arrays that overlap by all but `shift` leaves): each
    channel finds the masks that the one before it left, as in calls of one channel at a time."""
    import torch
    s = U.Scene(1, 48, seed=1)
    lap = U.LaplacianWithLevel(s.phi, s.weights, dt=1.0, dx=s.dx)
    p = torch.linspace(-1, 1, lap.mNumDof, device="cuda:0")
    _say(f"[case] shared masks, values on device {on_dev}, shift {shift}")
    n = s.vx.origins.shape[0] - 2 * shift
    org = [np.ascontiguousarray(g.origins[:n]) for g in (s.vx, s.vy, s.vz)]
    val = [np.ascontiguousarray(g.values[:n], dtype=np.float32) for g in (s.vx, s.vy, s.vz)]
    phi, w = s.phi, s.weights
    keep = [torch.from_numpy(np.ascontiguousarray(g.values, dtype=np.float32)).to("cuda:0") for g in (phi, w)]

    def run(calls, act, val):
        g = [grid._struct(t.data_ptr() if on_dev else None) for grid, t in zip((phi, w), keep)]
        for call in calls:
            ch = _channels([(org[c], act[c * shift:], val[c]) if c in call else None for c in range(3)])
            assert U.lib().uaamg_poisson_apply_pressure_gradient_device(
                lap._h, C.c_void_p(p.data_ptr()), C.byref(g[0]), C.byref(g[1]), None, ch, 0.04, 0.0, on_dev) == 0
        torch.cuda.synchronize()
    out = []
    for calls in ([(0, 1, 2)], [(0,), (1,), (2,)]):
        act = np.full((n + 2 * shift, 8), ~np.uint64(0), np.uint64)
        v = [torch.from_numpy(a).to("cuda:0") if on_dev else a.copy() for a in val]
        run(calls, act, v)
        out.append((act, [a.cpu().numpy() if on_dev else a for a in v]))
    (act, v), (act1, v1) = out
    assert np.array_equal(act, act1)
    for c in range(3):
        assert np.array_equal(v[c], v1[c]), f"channel {c}"
