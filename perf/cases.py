"""The calls a fluid simulation makes of this package, as timed cases.

Every case works on a liquid in a closed unit box on an n^3 grid: a pool with a
waving surface, spheres above it and, where said, a solid sphere cut out by fractional face
weights (the viscosity cases take the library's own scene of a pool and a
sphere). The grids are made on the GPU from the seed and handed over as the
flattened 8^3 leaves (tree order) that the entry points take; velocities stay
in device memory.

kinds
  poisson  one pressure solve to 1e-7 with the vectors in device memory
  batch    many pressure problems of uneven size solved together
  substep  what a simulation does per time step: build the hierarchy, build the
           right-hand side, solve, apply the pressure gradient
  faces    the two steps either side of a solve, all values in device memory
  visc     one variational viscosity solve to 1e-6
  viscstep build the viscosity hierarchy and right-hand side, solve
  vbatch   many viscosity problems solved together
"""
import ctypes
import math

import numpy as np
import torch

import uaamg_amd as U

DEV = "cuda"
BAND = 3.0  # voxels of signed distance kept outside the liquid
VISC_DT, VISC_RHO = 1.0 / 24.0, 1000.0


def listed():
    return [
        # the smallest solve: two levels, nothing but launches and latency
        {"name": "poisson_32", "kind": "poisson", "n": 32, "spheres": 1, "pool": 0.4, "solid": False,
         "precision": 0, "smoother": 0, "warm": False},
        # an ordinary interactive resolution, pool and one drop
        {"name": "poisson_128", "kind": "poisson", "n": 128, "spheres": 1, "pool": 0.4, "solid": False,
         "precision": 0, "smoother": 0, "warm": False},
        # the headline size, plain FP32
        {"name": "poisson_256", "kind": "poisson", "n": 256, "spheres": 8, "pool": 0.3, "solid": True,
         "precision": 0, "smoother": 0, "warm": False},
        # the headline size with the W-cycle's vectors stored in BF16
        {"name": "poisson_256_mixed", "kind": "poisson", "n": 256, "spheres": 8, "pool": 0.3, "solid": True,
         "precision": 1, "smoother": 0, "warm": False},
        # the largest grid: every level-0 vector is far beyond the caches
        {"name": "poisson_512", "kind": "poisson", "n": 512, "spheres": 8, "pool": 0.3, "solid": True,
         "precision": 0, "smoother": 0, "warm": False},
        # a production batch of independent problems of uneven size
        {"name": "batch_64", "kind": "batch", "count": 64, "lo": 32, "hi": 128, "precision": 0},
        # a whole pressure step: the hierarchy is rebuilt in every time step
        {"name": "substep_128", "kind": "substep", "n": 128, "spheres": 4, "pool": 0.35, "solid": True},
        # right-hand side and pressure gradient at the headline size
        {"name": "faces_256", "kind": "faces", "n": 256, "spheres": 8, "pool": 0.3, "solid": True},
        # a small viscous liquid
        {"name": "visc_64", "kind": "visc", "n": 64, "mu": 1.0, "precision": 0},
        # the ordinary viscosity resolution
        {"name": "visc_128", "kind": "visc", "n": 128, "mu": 1.0, "precision": 0},
        # a whole viscosity step with its hierarchy build
        {"name": "viscstep_64", "kind": "viscstep", "n": 64, "mu": 1.0},
        # a batch of viscosity problems of uneven size
        {"name": "vbatch_16", "kind": "vbatch", "count": 16, "lo": 32, "hi": 96, "mu": 1.0},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(lo * math.exp(rng.random() * math.log(hi / lo))))


def draw(rng):
    kind = rng.choice(["poisson", "poisson", "poisson", "poisson", "batch", "substep", "faces", "visc", "visc",
                       "viscstep", "vbatch"])
    scene = {"spheres": rng.randint(1, 8), "pool": round(rng.uniform(0.1, 0.5), 3), "solid": rng.random() < 0.5}
    if kind == "poisson":
        # scheduled Jacobi is the default smoother; the red-black one is the other a simulation picks
        return {"kind": kind, "n": _log_uniform(rng, 32, 384), **scene,
                "precision": int(rng.random() < 0.35), "smoother": rng.choice([0, 0, 0, 0, 2]),
                "warm": rng.random() < 0.3}
    if kind == "batch":
        lo = rng.randint(24, 48)
        return {"kind": kind, "count": rng.randint(5, 64), "lo": lo, "hi": rng.randint(lo + 20, 128),
                "precision": int(rng.random() < 0.5)}
    if kind == "substep":
        return {"kind": kind, "n": _log_uniform(rng, 32, 160), **scene}
    if kind == "faces":
        return {"kind": kind, "n": _log_uniform(rng, 32, 256), **scene}
    mu = round(math.exp(rng.uniform(math.log(0.1), math.log(20.0))), 3)
    if kind == "visc":
        return {"kind": kind, "n": _log_uniform(rng, 32, 144), "mu": mu, "precision": int(rng.random() < 0.25)}
    if kind == "viscstep":
        return {"kind": kind, "n": _log_uniform(rng, 32, 96), "mu": mu}
    return {"kind": kind, "count": rng.randint(3, 16), "lo": rng.randint(24, 40), "hi": rng.randint(48, 96), "mu": mu}


# ------------------------------------------------------------------ scenes

def _spheres(count):
    """Centres and radii"""
    g = torch.Generator().manual_seed(977)
    s = torch.rand((max(count, 1), 4), generator=g, dtype=torch.float64)[:count]
    s[:, 1] = 0.35 + 0.6 * s[:, 1]
    s[:, 3] = 0.05 + 0.1 * s[:, 3]
    return s


def _liquid(case, x, y, z):
    wave = 0.012 * (torch.cos(9.0 * x + 0.4) + torch.cos(7.0 * z + 2.1))
    d = y - (case["pool"] + wave)
    for s in _spheres(case["spheres"]).tolist():
        d = torch.minimum(d, torch.sqrt((x - s[0]) ** 2 + (y - s[1]) ** 2 + (z - s[2]) ** 2) - s[3])
    return d


def _solid(x, y, z):
    return torch.sqrt((x - 0.5) ** 2 + (y - 0.5) ** 2 + (z - 0.5) ** 2) - 0.2


def _dof_estimate(case):
    """DOFs of the case's liquid, by sampling."""
    m = 64
    c = (torch.arange(m, dtype=torch.float64) + 0.5) / m
    x, y, z = torch.meshgrid(c, c, c, indexing="ij")
    inside = _liquid(case, x, y, z) < 0
    if case["solid"]:
        inside &= _solid(x, y, z) > 0
    return case["n"] ** 3 * float(inside.double().mean())


def _leaves(a):
    """dense [m, m, m, ...] to leaves [(m/8)^3, 512, ...]"""
    k = a.shape[0] // 8
    tail = tuple(range(6, 3 + a.dim()))
    return a.reshape(k, 8, k, 8, k, 8, *a.shape[3:]).permute(0, 2, 4, 1, 3, 5, *tail).reshape(
        k ** 3, 512, *a.shape[3:])


class Scene:
    """The case's grids for one seed: dense FP32 fields on the GPU padded to whole
    leaves, and the kept leaves in tree order. The case says which voxels are
    liquid; the seed gives the velocities and how far off each voxel's surface
    is (the coefficients of every cut cell)."""

    def __init__(self, case, seed):
        n = case["n"]
        k = (n + 7) // 8
        m = 8 * k
        g = torch.Generator(device=DEV).manual_seed(int(seed))
        rnd = torch.Generator().manual_seed(int(seed))
        self.n, self.m, self.dx, self.dt = n, m, 1.0 / n, 1.0
        i = torch.arange(m, device=DEV, dtype=torch.float32) / n
        x, y, z = i.view(m, 1, 1), i.view(1, m, 1), i.view(1, 1, m)
        one = torch.arange(m, device=DEV) < n
        inside = one.view(m, 1, 1) & one.view(1, m, 1) & one.view(1, 1, m)
        band = BAND / n
        phi = _liquid(case, x, y, z)
        phi = torch.where(inside, phi, torch.full_like(phi, band))
        keep = _leaves(phi).amin(1) < band
        phi = torch.where(inside, phi * (1 + 0.1 * torch.rand((m, m, m), device=DEV, generator=g)), phi)
        # faces between v - e_c and v: closed on the box, partly covered by the solid
        w = torch.empty((m, m, m, 3), device=DEV)
        h = 0.5 / n
        for c in range(3):
            at = [x, y, z]
            at[c] = at[c] - h
            open_ = inside.float()
            if case["solid"]:
                open_ = open_ * (0.5 + _solid(*at) * n).clamp(0.0, 1.0)
                open_[open_ < 0.01] = 0.0
            open_.narrow(c, 0, 1).zero_()
            w[..., c] = open_
        # a few long waves under 10% noise
        self.vel = []
        for c in range(3):
            amp = torch.rand(3, generator=rnd).tolist()
            off = (6.28 * torch.rand(3, generator=rnd)).tolist()
            v = 0.1 * torch.randn((m, m, m), device=DEV, generator=g)
            for a, o, f in zip(amp, off, (3.0, 6.0, 11.0)):
                v += a * torch.sin(f * x + o) * torch.cos(f * y - o) * torch.sin(f * z + 2 * o)
            self.vel.append(v)
        o = 8 * torch.arange(k, device=DEV)
        org = torch.stack(torch.meshgrid(o, o, o, indexing="ij"), -1).reshape(-1, 3)[keep]
        upper = ((org[:, 0] >> 7) << 10) | ((org[:, 1] >> 7) << 5) | (org[:, 2] >> 7)
        lower = (((org[:, 0] & 127) >> 3) << 8) | (((org[:, 1] & 127) >> 3) << 4) | ((org[:, 2] & 127) >> 3)
        order = torch.argsort((upper << 12) | lower)
        self.pick = torch.nonzero(keep).flatten()[order]
        self.origins = org[order].to(torch.int32).cpu().numpy()
        self.phi, self.w, self.inside = phi, w, inside

    def on_leaves(self, a):
        return _leaves(a)[self.pick].contiguous()

    def active(self):
        bits = self.on_leaves(self.inside).to(torch.uint8).cpu().numpy()
        return np.packbits(bits, axis=1, bitorder="little").view(np.uint64).reshape(-1, 8)

    def grids(self):
        act = self.active()
        phi = U.Grid(self.origins, self.on_leaves(self.phi).cpu().numpy(), act, (BAND / self.n,) * 3)
        w = U.Grid(self.origins, self.on_leaves(self.w).cpu().numpy(), act)
        return phi, w

    def velocity_grid(self, act):
        """A face-velocity grid whose values are only in device memory."""
        return U.Grid(self.origins, np.zeros((0, 512), np.float32), act)

    # ---- the discretisation, written out on dense fields in 64 bits
    def system(self):
        """(DOF numbering [m,m,m], DOF voxels, diag, [6 couplings], [6 neighbour DOFs]) with DOFs in leaf
        order. The coefficients are the operator's own 32-bit numbers (the rounding of an interior row's
        diagonal alone shifts the solution by up to 1e-4); everything done with them is in 64 bits."""
        dx = np.float32(self.dx)
        t = float(np.float32(self.dt) / (dx * dx))
        phi, w = self.phi, self.w
        wet = (self.phi < 0) & self.inside
        diag = torch.zeros_like(phi)
        coef = []
        for c in range(3):
            for s in (1, -1):
                face = _shift(w[..., c], c, 1) if s > 0 else w[..., c]
                other = _shift(phi, c, s, fill=BAND / self.n)
                term = face * t
                theta = torch.where(other < 0, torch.ones_like(phi), (phi / (phi - other)).clamp(min=0.02))
                diag += torch.where(wet, term / theta, torch.zeros_like(phi))
                coef.append(torch.where(other < 0, -term, torch.zeros_like(phi)))
        dof = wet & (diag != 0)
        # a leaf whose rows all agree with the open interior's holds one number, 6 t, for them
        off = _leaves(torch.where(dof, (diag - 6 * t).abs(), torch.zeros_like(diag)))
        plain = (off.amax(1, keepdim=True) <= 6e-5 * t).expand(-1, 512)
        k = self.m // 8
        plain = plain.reshape(k, k, k, 8, 8, 8).permute(0, 3, 1, 4, 2, 5).reshape(self.m, self.m, self.m)
        diag = torch.where(plain & dof, torch.full_like(diag, float(np.float32(6) * np.float32(t))), diag)
        flat = self.on_leaves(dof).flatten()
        number = torch.where(flat, torch.cumsum(flat.long(), 0) - 1, torch.full_like(flat, -1, dtype=torch.long))
        at = self.on_leaves(torch.arange(self.m ** 3, device=DEV).view(self.m, self.m, self.m)).flatten()[flat]
        idx = torch.full((self.m ** 3,), -1, device=DEV, dtype=torch.long)
        idx[at] = number[flat]
        idx = idx.view(self.m, self.m, self.m)
        nb, k = [], 0
        for c in range(3):
            for s in (1, -1):
                j = _shift(idx, c, s, fill=-1).flatten()[at]
                a = coef[k].flatten()[at].double()
                coef[k] = torch.where(j >= 0, a, torch.zeros_like(a))
                nb.append(j.clamp(min=0))
                k += 1
        return idx, at, diag.flatten()[at].double(), coef, nb

    def dofs(self):
        """Voxels (dense index) of the DOFs in DOF order, without building the system."""
        wet = (self.phi < 0) & self.inside
        open_ = torch.zeros_like(wet)
        for c in range(3):
            open_ |= (self.w[..., c] > 0) | (_shift(self.w[..., c], c, 1) > 0)
        flat = self.on_leaves(wet & open_).flatten()
        return self.on_leaves(torch.arange(self.m ** 3, device=DEV).view(self.m, self.m, self.m)).flatten()[flat]

    def divergence(self, dtype=torch.float64):
        """The right-hand side on the dense grid: -div(w u) with still solids."""
        r = torch.zeros((self.m,) * 3, device=DEV, dtype=dtype)
        for c in range(3):
            f = self.w[..., c].to(dtype) * self.vel[c].to(dtype)
            r += f - _shift(f, c, 1)
        return r * self.n


def _shift(a, axis, s, fill=0):
    """a at v + s e_axis, `fill` outside"""
    out = torch.full_like(a, fill)
    m = a.shape[axis]
    if s > 0:
        out.narrow(axis, 0, m - 1).copy_(a.narrow(axis, 1, m - 1))
    else:
        out.narrow(axis, 1, m - 1).copy_(a.narrow(axis, 0, m - 1))
    return out


def _cg(apply, diag, b, tol, x=None, most=6000):
    """Jacobi-preconditioned conjugate gradients in 64 bits"""
    x = torch.zeros_like(b) if x is None else x.clone()
    r = b - apply(x)
    stop = tol * b.abs().max().item()
    z = r / diag
    p = z.clone()
    rz = torch.dot(r, z)
    for k in range(most):
        q = apply(p)
        a = rz / torch.dot(p, q)
        x += a * p
        r -= a * q
        if k % 16 == 15 and r.abs().max().item() <= stop:
            break
        z = r / diag
        new = torch.dot(r, z)
        p = z + (new / rz) * p
        rz = new
    return x


def _solve64(scene, b):
    _, _, diag, coef, nb = scene.system()
    nb = torch.stack(nb).int()
    coef = torch.stack(coef)

    def apply(v):
        y = diag * v
        for k in range(6):
            y += coef[k] * v[nb[k]]
        return y
    return _cg(apply, diag, b.double(), 1e-11)


# ------------------------------------------------------------------ cases

def _batch_scenes(case):
    """Edges spread over [lo, hi]'s logarithm, each problem with its own shape."""
    out = []
    for i in range(case["count"]):
        f = (i + 0.5) / case["count"]
        out.append({"n": int(round(case["lo"] * math.exp(f * math.log(case["hi"] / case["lo"])))),
                    "spheres": 1 + i % 6, "pool": 0.1 + 0.4 * ((7 * i) % 11) / 10, "solid": i % 2 == 1})
    return out


def _vbatch_sizes(case):
    return [int(round(case["lo"] * math.exp((i + 0.5) / case["count"] * math.log(case["hi"] / case["lo"]))))
            for i in range(case["count"])]


def _noisy(b0, seed):
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    return b0 * (1 + 0.05 * torch.randn(b0.shape, device=DEV, generator=g))


def _rhs(scene):
    return scene.divergence().flatten()[scene.dofs()].float()


def _warm(b, seed):
    """A starting pressure of about the right size: the last step's solution in a simulation"""
    g = torch.Generator(device=DEV).manual_seed(int(seed) + 1)
    return 1e-6 * b.abs().mean() * torch.randn(b.shape, device=DEV, generator=g)


class _Vectors:
    """Many DOF vectors in one allocation, each at a 256-byte boundary."""

    def __init__(self, parts):
        at, self.views, self.sizes = 0, [], [p.numel() for p in parts]
        self.flat = torch.zeros(sum((s + 63) // 64 * 64 for s in self.sizes), device=DEV)
        for p in parts:
            v = self.flat[at:at + p.numel()]
            v.copy_(p)
            self.views.append(v)
            at += (p.numel() + 63) // 64 * 64
        self.ptrs = [v.data_ptr() for v in self.views]


class _Faces:
    """A simulation's face velocities in device memory with the arrays the pressure gradient writes."""

    def __init__(self, scene, phi, w):
        self.phi, self.w = phi, w
        self.phi_dev = scene.on_leaves(scene.phi)
        self.w_dev = scene.on_leaves(scene.w)
        self.vel = torch.stack([scene.on_leaves(v) for v in scene.vel])
        self.vgrid = [scene.velocity_grid(phi.active) for _ in range(3)]
        self.out = torch.empty_like(self.vel)
        self.upd, self.refl = torch.empty_like(self.vel), torch.empty_like(self.vel)
        self.act = np.stack([phi.active] * 3)

    def rhs(self, lap, b):
        lap.createPressurePoissonRightHandSide_device(
            b.data_ptr(), self.w, *self.vgrid,
            values_ptrs=[self.w_dev.data_ptr()] + [self.vel[c].data_ptr() for c in range(3)])

    def gradient(self, lap, p, dt):
        self.out.copy_(self.vel)
        gp, gw = self.phi._struct(self.phi_dev.data_ptr()), self.w._struct(self.w_dev.data_ptr())
        act = self.act.copy()
        org = np.ascontiguousarray(self.phi.origins)
        ch = (U._FaceChannel * 3)()
        for c in range(3):
            ch[c].nleaf = org.shape[0]
            ch[c].origins = org.ctypes.data
            ch[c].active = act[c].ctypes.data
            ch[c].values = self.out[c].data_ptr()
            ch[c].update = self.upd[c].data_ptr()
            ch[c].reflected = self.refl[c].data_ptr()
        rc = U.lib().uaamg_poisson_apply_pressure_gradient_device(
            lap._h, ctypes.c_void_p(p.data_ptr()), ctypes.byref(gp), ctypes.byref(gw), None, ch, float(dt), 0.0, 1)
        if rc != 0:
            raise RuntimeError("pressure gradient returned %d" % rc)
        return act.view(np.int64)


def _visc_scene(case, seed):
    return U.ViscScene(0, case["n"], seed=int(seed), mu=case["mu"], dt=VISC_DT, rho=VISC_RHO)


def _visc_handle(sc, precision=0):
    return U.L_with_level(sc.viscosity, sc.liquid, sc.solid, sc.dt, sc.rho, sc.dx, device=0, precision=precision)


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "poisson":
        sc = Scene(case, seed)
        phi, w = sc.grids()
        s["lap"] = U.LaplacianWithLevel(phi, w, dt=sc.dt, dx=sc.dx, device=0, precision=case["precision"],
                                        smoother=case["smoother"])
        s["b"] = _rhs(sc)
        if s["b"].numel() != s["lap"].mNumDof:
            raise RuntimeError("the scene has %d DOFs, the handle %d" % (s["b"].numel(), s["lap"].mNumDof))
        s["x0"] = _warm(s["b"], seed) if case["warm"] else torch.zeros_like(s["b"])
        s["x"] = torch.empty_like(s["b"])
    elif kind == "batch":
        scenes = [Scene(c, int(seed) + 31 * i) for i, c in enumerate(_batch_scenes(case))]
        grids = [sc.grids() for sc in scenes]
        s["batch"] = U.PoissonBatch([(g[0], g[1], sc.dt, sc.dx) for g, sc in zip(grids, scenes)],
                                    precision=case["precision"])
        b = [_rhs(sc) for sc in scenes]
        s["b"], s["x"] = _Vectors(b), _Vectors([torch.zeros_like(v) for v in b])
    elif kind == "substep":
        sc = Scene(case, seed)
        phi, w = sc.grids()
        s["sc"] = (sc.dt, sc.dx)
        s["faces"] = _Faces(sc, phi, w)
    elif kind == "faces":
        sc = Scene(case, seed)
        phi, w = sc.grids()
        s["sc"] = (sc.dt, sc.dx)
        s["lap"] = U.LaplacianWithLevel(phi, w, dt=sc.dt, dx=sc.dx, device=0)
        s["faces"] = _Faces(sc, phi, w)
        s["b"] = torch.empty(s["lap"].mNumDof, device=DEV)
        s["p"] = _pressure(sc, seed)
    elif kind in ("visc", "viscstep"):
        sc = _visc_scene(case, seed)
        if kind == "viscstep":
            s["sc"] = sc
        else:
            lw = _visc_handle(sc, case["precision"])
            s["solver"] = U.simd_viscosity3d(lw, sc.velocity)
            s["b"] = torch.from_numpy(s["solver"].m_rhs.data).to(DEV)
            s["x"] = torch.empty_like(s["b"])
    else:
        problems, b = [], []
        for i, n in enumerate(_vbatch_sizes(case)):
            sc = U.ViscScene(3, n, seed=i, mu=case["mu"], dt=VISC_DT, rho=VISC_RHO)
            lw = U.L_with_level(sc.viscosity, sc.liquid, sc.solid, sc.dt, sc.rho, sc.dx, device=-1)
            b.append(_noisy(torch.from_numpy(lw.build_rhs(sc.velocity).data).to(DEV), int(seed) + 31 * i))
            problems.append((sc.viscosity, sc.liquid, sc.solid, sc.dt, sc.rho, sc.dx))
        s["batch"] = U.ViscBatch(problems)
        s["b"], s["x"] = _Vectors(b), _Vectors([torch.zeros_like(v) for v in b])
    return s


def _pressure(sc, seed):
    """A smooth pressure with a little noise, in DOF order"""
    at = sc.dofs()
    g = torch.Generator(device=DEV).manual_seed(int(seed) + 5)
    x, y, z = (at // (sc.m * sc.m)).float(), ((at // sc.m) % sc.m).float(), (at % sc.m).float()
    f = 6.0 / sc.n
    return sc.dx * (torch.sin(f * x) * torch.cos(f * y) + torch.sin(f * z) +
                    0.01 * torch.randn(at.shape, device=DEV, generator=g))


def run(state):
    # A solve's status and iteration count are not among the outputs: at the edge of the stopping
    # rule they hang on the last bits, while the solution differs by no more than the tolerance.
    case, kind = state["case"], state["case"]["kind"]
    if kind == "poisson":
        x = state["x"]
        x.copy_(state["x0"])
        state["lap"].solve_pcg_device(x.data_ptr(), state["b"].data_ptr())
        return {"x": x}
    if kind == "batch":
        state["x"].flat.zero_()
        state["batch"].solve_device(state["x"].ptrs, state["b"].ptrs)
        return {"x": state["x"].flat}
    if kind == "substep":
        f, (dt, dx) = state["faces"], state["sc"]
        lap = U.LaplacianWithLevel(f.phi, f.w, dt=dt, dx=dx, device=0)
        b = torch.empty(lap.mNumDof, device=DEV)
        f.rhs(lap, b)
        p = torch.zeros_like(b)
        lap.solve_pcg_device(p.data_ptr(), b.data_ptr())
        act = f.gradient(lap, p, dt)
        return {"p": p, "u": f.out, "active": act}
    if kind == "faces":
        f = state["faces"]
        f.rhs(state["lap"], state["b"])
        act = f.gradient(state["lap"], state["p"], state["sc"][0])
        return {"b": state["b"], "u": f.out, "update": f.upd, "reflected": f.refl, "active": act}
    if kind == "visc":
        x = state["x"]
        x.zero_()
        state["solver"].solve_pcg_device(1e-6, x.data_ptr(), state["b"].data_ptr())
        return {"x": x}
    if kind == "viscstep":
        sc = state["sc"]
        solver = U.simd_viscosity3d(_visc_handle(sc), sc.velocity)
        b = torch.from_numpy(solver.m_rhs.data).to(DEV)
        x = torch.zeros_like(b)
        solver.solve_pcg_device(1e-6, x.data_ptr(), b.data_ptr())
        return {"x": x, "b": b}
    state["x"].flat.zero_()
    state["batch"].solve_device(1e-6, state["x"].ptrs, state["b"].ptrs)
    return {"x": state["x"].flat}


# ------------------------------------------------------------------ what a pass needs, and how exact it is

#: arithmetic of one preconditioned iteration per level-0 DOF (operator, smoothing on all levels, vector updates)
POISSON_FLOPS, VISC_FLOPS = 220.0, 700.0


def work(case):
    kind = case["kind"]
    if kind in ("poisson", "batch"):
        n = sum(_dof_estimate(c) for c in _batch_scenes(case)) if kind == "batch" else _dof_estimate(case)
        # right-hand side and start in, solution out; the four coefficients of the cut cells are a small share
        return {"bytes": 12.0 * n, "flops": 8 * POISSON_FLOPS * n}
    if kind in ("substep", "faces"):
        n = _dof_estimate(case)
        leaf = 1.15 * n  # voxels of the kept leaves
        faces = (1 + 3 + 3 + 3 + 3 + 3) * 4.0 * leaf  # phi, weights, velocity in; velocity, update, reflected out
        if kind == "faces":
            return {"bytes": faces + 8.0 * n, "flops": 60.0 * n}
        return {"bytes": faces + 20.0 * n, "flops": (60 + 8 * POISSON_FLOPS) * n}
    # three staggered channels; about 0.43 of the box is liquid
    edges = _vbatch_sizes(case) if kind == "vbatch" else [case["n"]]
    n = sum(3 * 0.43 * e ** 3 for e in edges)
    return {"bytes": (12.0 if kind != "viscstep" else 40.0) * n, "flops": 5 * VISC_FLOPS * n}


def tolerance(case):
    # four times the distance from the 64-bit result, or from a solve stopped one iteration apart
    kind = case["kind"]
    if kind == "faces":
        return {"rel": 4e-7, "differ": 0.0}   # a handful of 32-bit roundings per face
    if kind in ("visc", "viscstep", "vbatch"):
        return {"rel": 4e-6}                  # stopped at 1e-6 of the residual
    if kind in ("poisson", "batch"):
        return {"rel": 6e-6}                  # stopped at 1e-7 of the residual, times the grid's condition
    return {"rel": 1.2e-5, "differ": 0.0}     # the same, and the differences of its pressure


def _visc64(lw, b):
    """The 64-bit solution of the handle's explicit level-0 matrix"""
    ptr, col, val = lw.level_matrix(0)
    a = torch.sparse_csr_tensor(torch.from_numpy(ptr).to(DEV), torch.from_numpy(col.astype(np.int64)).to(DEV),
                                torch.from_numpy(val.astype(np.float64)).to(DEV), size=(b.numel(), b.numel()))
    row = torch.repeat_interleave(torch.arange(b.numel(), device=DEV), a.crow_indices().diff())
    diag = torch.zeros(b.numel(), device=DEV, dtype=torch.float64)
    on = row == a.col_indices()
    diag[row[on]] = a.values()[on]
    return _cg(lambda v: a @ v, diag, b.double(), 1e-11)


def exact(case, seed):
    kind = case["kind"]
    if kind == "poisson":
        if _dof_estimate(case) > 1.5e7:
            return None  # minutes of unpreconditioned iterations
        sc = Scene(case, seed)
        return {"x": _solve64(sc, _rhs(sc))}
    if kind == "batch":
        parts = []
        for i, c in enumerate(_batch_scenes(case)):
            sc = Scene(c, int(seed) + 31 * i)
            x = _solve64(sc, _rhs(sc))
            parts.append(torch.nn.functional.pad(x, (0, -x.numel() % 64)))
        return {"x": torch.cat(parts)}
    if kind in ("substep", "faces"):
        sc = Scene(case, seed)
        idx, at, diag, coef, nb = sc.system()
        b = sc.divergence().flatten()[at]
        if kind == "faces":
            p = _pressure(sc, seed).double()
        else:
            p = _solve64(sc, b.float())
        dense = torch.zeros(sc.m ** 3, device=DEV, dtype=torch.float64)
        dense[at] = p
        dense, has = dense.view(sc.m, sc.m, sc.m), idx >= 0
        phi = sc.phi.double()
        out, upd, refl = [], [], []
        for c in range(3):
            u = sc.vel[c].double()
            below = _shift(phi, c, -1, fill=BAND / sc.n)
            cut = (phi >= 0) | (below >= 0)
            wet = torch.where(phi < 0, phi / (phi - below), below / (below - phi))
            theta = torch.where(cut, torch.where((phi < 0) ^ (below < 0), wet, torch.zeros_like(wet)).clamp(min=0.02),
                                torch.ones_like(wet))
            du = -sc.dt * (dense - _shift(dense, c, -1)) / np.float64(np.float32(sc.dx)) / theta
            on = sc.inside & (sc.w[..., c] > 0) & (has | _shift(has, c, -1, fill=False))
            out.append(sc.on_leaves(torch.where(on, u + du, u)))
            upd.append(sc.on_leaves(torch.where(on, du, u)))
            refl.append(sc.on_leaves(torch.where(on, u + 2 * du, u)))
        if kind == "faces":
            return {"b": b, "u": torch.stack(out), "update": torch.stack(upd), "reflected": torch.stack(refl),
                    "active": None}
        return {"p": p, "u": torch.stack(out), "active": None}
    # the viscosity operator's definition fills a file of its own: the matrix that the handle reports is taken as given
    if kind in ("visc", "viscstep"):
        sc = _visc_scene(case, seed)
        lw = U.L_with_level(sc.viscosity, sc.liquid, sc.solid, sc.dt, sc.rho, sc.dx, device=-1)
        b = torch.from_numpy(lw.build_rhs(sc.velocity).data).to(DEV)
        x = _visc64(lw, b)
        return {"x": x} if kind == "visc" else {"x": x, "b": None}
    parts = []
    for i, n in enumerate(_vbatch_sizes(case)):
        sc = U.ViscScene(3, n, seed=i, mu=case["mu"], dt=VISC_DT, rho=VISC_RHO)
        lw = U.L_with_level(sc.viscosity, sc.liquid, sc.solid, sc.dt, sc.rho, sc.dx, device=-1)
        x = _visc64(lw, _noisy(torch.from_numpy(lw.build_rhs(sc.velocity).data).to(DEV), int(seed) + 31 * i))
        parts.append(torch.nn.functional.pad(x, (0, -x.numel() % 64)))
    return {"x": torch.cat(parts)}
