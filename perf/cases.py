"""The work that programs built on this package have it do, as measurable cases.

Every case is one call sequence of such a program, through the package's public classes, on sizes
from the package's own solver cases, tests and benchmark:

* ``flow``     a run of steps of the lattice-Boltzmann solver, then the macroscopic fields on the
               device (and the FP64 diagnostics where the command-line solver prints them);
* ``adjoint``  one objective with its gradients: the pressure drop through ``lbm_objective`` and
               ``backward()``, the drag (from an impulsive start) through the solver's own call;
* ``coupled``  time steps of the flow with the resident thermal, free-surface and particle modules,
               one flow step per call, then the Q-criterion;
* ``voxelize`` a triangle surface on host memory to its solid mask on host memory.

``exact`` restates each of them in 64 bits in plain torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch
from torch.utils.checkpoint import checkpoint

import cfd_solvers_amd as cfd
from cfd_solvers_amd import geometry
from cfd_solvers_amd.autograd import LbmAdjointProblem, lbm_objective

TAU = {"periodic": 0.6, "cavity": 0.55, "channel": 0.8, "duct": 0.52}
BYTES = {"fp32": 4, "fp32s": 4, "fp16s": 2, "fp64": 8}
Q = {"d2q9": 9, "d3q19": 19, "d3q27": 27}
LID, INLET_PEAK, FORCE = 0.1, 0.04, 1.0e-5


def _flow(name, lattice, nx, ny, nz, storage, scene, steps, report=False):
    return {"name": name, "kind": "flow", "lattice": lattice, "nx": nx, "ny": ny, "nz": nz, "storage": storage,
            "scene": scene, "steps": steps, "report": report}


def listed():
    return [
        # The command-line solver's 2-D case: a small periodic lattice, a run, its printed diagnostics.
        _flow("d2q9 256 periodic", "d2q9", 256, 256, 1, "fp32", "periodic", 200, True),
        # The command-line solver's two 3-D cases, which fit the caches.
        _flow("d3q19 64 periodic", "d3q19", 64, 64, 64, "fp32", "periodic", 100, True),
        _flow("d3q27 56 periodic", "d3q27", 56, 56, 56, "fp32", "periodic", 100, True),
        # A 2-D lid-driven cavity at production resolution.
        _flow("d2q9 4096 cavity", "d2q9", 4096, 4096, 1, "fp32", "cavity", 20),
        # The benchmark's lid-driven cavity in full and in compressed storage.
        _flow("d3q19 256 cavity", "d3q19", 256, 256, 256, "fp32", "cavity", 20),
        _flow("d3q19 256 cavity fp16s", "d3q19", 256, 256, 256, "fp16s", "cavity", 20),
        # A body-force driven channel with a sphere pack, on extents that divide no tile.
        _flow("d3q19 porous channel", "d3q19", 301, 150, 141, "fp32s", "channel", 20),
        # Flow past a sphere cluster with a porous halo, inlet and outlet: the largest lattice.
        _flow("d3q19 512 cluster fp16s", "d3q19", 512, 512, 512, "fp16s", "duct", 10),
        # A design gradient of the porous duct with snapshots every 100 steps.
        {"name": "adjoint 128 duct", "kind": "adjoint", "n": 128, "storage": "fp32", "objective": "pressure_drop",
         "steps": 200, "window": 20, "every": 100, "snapshots": 0},
        # A drag gradient where few states fit: binomial checkpoints, compressed storage.
        {"name": "adjoint 192 drag fp16s", "kind": "adjoint", "n": 192, "storage": "fp16s", "objective": "drag",
         "steps": 60, "window": 60, "every": 0, "snapshots": 4},
        # Thermal two-phase flow with particles: every module once per flow step.
        {"name": "coupled 192", "kind": "coupled", "nx": 192, "ny": 192, "nz": 192, "storage": "fp32",
         "particles": 131072, "two_way": True, "steps": 10},
        # A surface mesh voxelised for a solid mask on the host.
        {"name": "voxelize 384", "kind": "voxelize", "nx": 384, "ny": 384, "nz": 384, "bands": 64},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["flow2d", "flow3d", "flow3d", "flow3d", "channel", "duct", "adjoint", "coupled", "voxelize"])
    if kind == "flow2d":
        nx, ny = _log(rng, 64, 4096), _log(rng, 64, 4096)
        steps = max(20, min(200, 20 * 4096 * 4096 // (nx * ny)))
        return {k: v for k, v in _flow("", "d2q9", nx, ny, 1, rng.choice(["fp32", "fp32", "fp16s", "fp32s"]),
                                       rng.choice(["periodic", "cavity"]), steps, nx * ny < 1 << 18).items()
                if k != "name"}
    if kind == "flow3d":
        nx, ny, nz = (_log(rng, 40, 300) for _ in range(3))
        steps = max(20, min(100, 20 * 256 ** 3 // (nx * ny * nz)))
        return {k: v for k, v in _flow("", rng.choice(["d3q19", "d3q19", "d3q19", "d3q27"]), nx, ny, nz,
                                       rng.choice(["fp32", "fp32", "fp16s", "fp16s", "fp32s", "fp64"]),
                                       rng.choice(["periodic", "cavity"]), steps, nx * ny * nz < 1 << 19).items()
                if k != "name"}
    if kind == "channel":
        return {k: v for k, v in _flow("", "d3q19", _log(rng, 96, 400), _log(rng, 64, 200), _log(rng, 64, 200),
                                       rng.choice(["fp32", "fp16s", "fp32s"]), "channel", 20).items() if k != "name"}
    if kind == "duct":
        n = _log(rng, 128, 400)
        return {k: v for k, v in _flow("", "d3q19", n, n, n, rng.choice(["fp16s", "fp32"]), "duct", 10).items()
                if k != "name"}
    if kind == "adjoint":
        drag = rng.random() < 0.5
        return {"kind": "adjoint", "n": _log(rng, 96, 192) if drag else _log(rng, 48, 128),
                "storage": rng.choice(["fp16s", "fp32"]),
                "objective": "drag" if drag else "pressure_drop", "steps": rng.randint(30, 60) if drag else
                rng.randint(60, 200), "window": rng.randint(5, 30), "every": 0 if drag else rng.randint(20, 100),
                "snapshots": rng.randint(3, 8) if drag else 0}
    if kind == "coupled":
        return {"kind": "coupled", "nx": _log(rng, 64, 224), "ny": _log(rng, 64, 224), "nz": _log(rng, 64, 192),
                "storage": rng.choice(["fp32", "fp16s"]), "particles": _log(rng, 4096, 131072),
                "two_way": rng.random() < 0.5, "steps": 10}
    return {"kind": "voxelize", "nx": _log(rng, 64, 400), "ny": _log(rng, 64, 400), "nz": _log(rng, 64, 384),
            "bands": _log(rng, 8, 96)}


# ------------------------------------------------------------------ inputs
def _modes(seed, shape, count, device="cuda"):
    """`count` smooth fields of about unit size: a few seeded Fourier modes and a little white noise."""
    g = np.random.default_rng(seed)
    nz, ny, nx = shape
    x, y, z = (torch.arange(n, device=device, dtype=torch.float64).add(0.5).div(n).mul(2 * math.pi)
               for n in (nx, ny, nz))
    noise = torch.Generator(device=device)
    noise.manual_seed(int(g.integers(1 << 62)))
    out = []
    for _ in range(count):
        f = torch.zeros(shape, device=device, dtype=torch.float32)
        for _ in range(3):
            k = g.integers(1, 4, 3)
            p = g.uniform(0, 2 * math.pi, 3)
            term = (torch.cos(k[0] * x + p[0])[None, None, :] * torch.cos(k[1] * y + p[1])[None, :, None])
            term = term * (torch.cos(k[2] * z + p[2])[:, None, None] if nz > 1 else 1.0)
            f += (g.uniform(0.3, 0.6) * term).to(torch.float32)
        f += 0.01 * torch.randn(shape, device=device, generator=noise)
        out.append(f)
    return out


def _initial_fields(case, seed):
    """Seeded density and velocity of the closed and periodic flows (float32, shape (nz, ny, nx))."""
    shape = (case["nz"], case["ny"], case["nx"])
    r, u, v, w = _modes(seed, shape, 4)
    return 1.0 + 0.002 * r, 0.03 * u, 0.03 * v, (0.03 * w if case["nz"] > 1 else torch.zeros_like(w))


def _cavity_flags(nx, ny, nz):
    f = np.zeros((nz, ny, nx), np.uint8)
    f[:, -1, :] = 0x81  # the lid, wall velocity 1
    f[:, :, 0] = f[:, :, -1] = 0x80
    f[:, 0, :] = 0x80
    if nz > 1:
        f[0, :, :] = f[-1, :, :] = 0x80
    return f


def _cluster(n, seed):
    """A duct past a seeded cluster of spheres: flags, body and porous halo, shape (n, n, n)."""
    if n >= 384:
        count, r_min, r_max = 64, 10, 30
    else:
        count, r_min, r_max = 16, n / 48, n / 20
    flags, body, halo = geometry.sphere_cluster_duct(n, seed, count, r_min, r_max)
    return (a.reshape(n, n, n) for a in (flags, body, halo))


def _flow_setup(case, seed):
    """(flags or None, gamma or None, acceleration, inlet peak) of a flow case."""
    nx, ny, nz, scene = case["nx"], case["ny"], case["nz"], case["scene"]
    if scene == "cavity":
        return _cavity_flags(nx, ny, nz), None, (0.0, 0.0, 0.0), 0.0
    if scene == "channel":
        flags = geometry.channel_flags(nx, ny, nz)
        r = min(ny, nz) / 10
        centres, radii = geometry.random_spheres((nz, ny, nx), 0.4 * r, r, seed=seed, porosity=0.85)
        flags[geometry.rasterize((nz, ny, nx), centres, radii)] = geometry.WALL
        return flags, None, (FORCE, 0.0, 0.0), 0.0
    if scene == "duct":
        flags, _, halo = _cluster(nx, seed)
        return flags, halo, (0.0, 0.0, 0.0), INLET_PEAK * (1 + 0.1 * np.random.default_rng(seed).random())
    return None, None, (0.0, 0.0, 0.0), 0.0


def _adjoint_setup(case, seed):
    n = case["n"]
    g = np.random.default_rng(seed)
    if case["objective"] == "drag":
        flags, body, halo = _cluster(n, seed)
        return flags, body, halo, INLET_PEAK
    flags = geometry.channel_flags(n, n, n, inlet_outlet=True)
    blend = np.where(flags == 0, 0.01 * g.uniform(0.3, 0.7, flags.shape), 0.0).astype(np.float32)
    return flags, None, blend, 0.05


def _coupled_fields(case, seed):
    shape = (case["nz"], case["ny"], case["nx"])
    t, phi = _modes(seed + 1, shape, 2)
    g = np.random.default_rng(seed + 2)
    count = case["particles"]
    parts = np.column_stack([g.uniform(0, 1, (count, 3)) * [case["nx"], case["ny"], case["nz"]],
                             g.normal(0, 0.01, (count, 3)), g.uniform(0.5, 1.5, count) * 1e-4, np.full(count, 5.0)])
    return 300.0 + t, (0.5 + 0.3 * phi).clamp(0, 1), parts.astype(np.float32).astype(np.float64)


# ------------------------------------------------------------------ the calls
class _DeviceField:
    def __init__(self, pointer, shape, dtype):
        self.__cuda_array_interface__ = {"data": (pointer, False), "shape": shape, "typestr": dtype, "version": 3}


class _Views:
    """Torch tensors over the package's device fields, made once per address as a program does.  A view
    keeps the objects alive whose memory it shows, so it may outlive the state it came from."""

    def __init__(self, owners, shape, dtype="<f4"):
        self.owners, self.shape, self.dtype, self.made = owners, shape, dtype, {}

    def __call__(self, pointers):
        for p in pointers:
            if p not in self.made:
                field = _DeviceField(p, self.shape, self.dtype)
                field.owners = self.owners
                view = torch.as_tensor(field, device="cuda")
                view.owners = self.owners
                self.made[p] = view
        return [self.made[p] for p in pointers]


def _host(fields):
    return [f.cpu().numpy() for f in fields]


def prepare(case, seed):
    if case["kind"] == "flow":
        flags, gamma, force, peak = _flow_setup(case, seed)
        s = cfd.EsotericPullHipSolver(case["lattice"], case["nx"], case["ny"], case["nz"], TAU[case["scene"]], force,
                                      storage=case["storage"])
        if flags is not None:
            s.set_flags(flags)
        if case["scene"] == "cavity":
            s.set_wall_velocity(1, (LID, 0.0, 0.0))
        if case["scene"] == "duct":
            s.set_porosity(gamma)
            s.set_inlet_outlet(peak, 1.0)
            s.initialize_uniform(1.0, INLET_PEAK, 0.0, 0.0)
        else:
            s.initialize_fields(*_host(_initial_fields(case, seed)))
        s.wait()
        dtype = "<f8" if case["storage"] == "fp64" else "<f4"
        return {"case": case, "flow": s, "views": _Views([s], (case["nz"], case["ny"], case["nx"]), dtype)}
    if case["kind"] == "adjoint":
        flags, body, gamma, peak = _adjoint_setup(case, seed)
        n = case["n"]
        if case["objective"] == "drag":
            s = cfd.EsotericPullHipSolver("d3q19", n, n, n, 0.6, storage=case["storage"])
            s.set_flags(flags)
            s.set_drag_body(body)
            s.set_porosity(gamma)
            s.set_inlet_outlet(peak, 1.0)
            s.wait()
            return {"case": case, "flow": s,
                    "grad": torch.zeros((n, n, n), dtype=torch.float64, device="cuda")}
        problem = LbmAdjointProblem(flags=flags, shape=(n, n, n), storage=case["storage"], tau=0.6,
                                    steps=case["steps"], window=case["window"], checkpoint_every=case["every"],
                                    snapshots=case["snapshots"], objective=case["objective"])
        problem.solver().wait()
        return {"case": case, "problem": problem,
                "gamma": torch.from_numpy(gamma).cuda().requires_grad_(True),
                "peak": torch.tensor(peak, dtype=torch.float32, device="cuda", requires_grad=True)}
    if case["kind"] == "coupled":
        flow = cfd.EsotericPullHipSolver("d3q19", case["nx"], case["ny"], case["nz"], TAU["periodic"],
                                         storage=case["storage"])
        flow.initialize_fields(*_host(_initial_fields(case, seed)))
        heat, fill, parts = _coupled_fields(case, seed)
        thermal, surface = cfd.ResidentThermalD3Q7(flow, 0.02), cfd.ResidentFreeSurface(flow)
        thermal.initialize_fields(heat.cpu().numpy())
        surface.upload_fill(fill.cpu().numpy())
        particles = cfd.ResidentParticles(flow, case["particles"])
        particles.upload(parts)
        diag = cfd.ResidentFlowDiagnostics(flow)
        flow.device_local_acceleration(clear=True)
        flow.wait()
        views = _Views([diag, particles, surface, thermal, flow], (case["nz"], case["ny"], case["nx"]))
        return {"case": case, "flow": flow, "thermal": thermal, "surface": surface, "particles": particles,
                "diag": diag, "views": views}
    g = np.random.default_rng(seed)
    mesh = geometry.sphere_surface(g.uniform(0.45, 0.55, 3), g.uniform(0.3, 0.42), case["bands"], 2 * case["bands"])
    return {"case": case, "mesh": mesh}


def run(state):
    case = state["case"]
    if case["kind"] == "flow":
        flow = state["flow"]
        flow.step(case["steps"])
        out = state["views"](flow.refresh_device_macroscopic())
        return out + [list(flow.diagnostics())] if case["report"] else out
    if case["kind"] == "adjoint" and case["objective"] == "drag":
        flow, grad = state["flow"], state["grad"]
        flow.initialize_uniform(1.0, INLET_PEAK, 0.0, 0.0)
        J, dpeak, _ = flow.adjoint_run_binomial_device(case["steps"], case["window"], grad.data_ptr(),
                                                       case["snapshots"], "drag")
        # The gradients of 32-bit design values, as an optimiser takes them.
        return [J, grad.to(torch.float32), np.float32(dpeak)]
    if case["kind"] == "adjoint":
        gamma, peak = state["gamma"], state["peak"]
        gamma.grad = peak.grad = None
        J = lbm_objective(gamma, peak, state["problem"])
        J.backward()
        return [J.detach(), gamma.grad, peak.grad]
    if case["kind"] == "coupled":
        flow, thermal, surface, particles = (state[k] for k in ("flow", "thermal", "surface", "particles"))
        for _ in range(case["steps"]):
            macro = flow.refresh_device_macroscopic()
            force = flow.device_local_acceleration(clear=True)
            thermal.step(macro, 1)
            thermal.add_boussinesq_acceleration(force, 300.0, 1e-5, (0.0, -1.0, 0.0))
            surface.advect(macro, 0.5)
            surface.add_surface_tension_acceleration(force, 1e-4, 1.0)
            particles.advance(macro, force, 1.0, case["two_way"], (0.0, -1e-5, 0.0))
            flow.step(1)
        macro = flow.refresh_device_macroscopic()
        vortices = state["diag"].q_criterion(macro)
        geometry_fields = surface.refresh_geometry()
        # The particle rows come back as doubles of the module's 32-bit state.
        return state["views"]([*macro, vortices, thermal.refresh_device_scalar(), surface.fill_device(),
                               *geometry_fields]) + [particles.download().astype(np.float32)]
    return cfd.voxelize_surface(state["mesh"], (case["nx"], case["ny"], case["nz"]))


def work(case):
    if case["kind"] == "flow":
        cells, q, e = case["nx"] * case["ny"] * case["nz"], Q[case["lattice"]], BYTES[case["storage"]]
        fixed = {"periodic": 0, "cavity": 1, "channel": 1, "duct": 5}[case["scene"]]  # flags, porosity
        return {"bytes": cells * (2 * q * e + 4 * max(e, 4) + fixed), "flops": cells * case["steps"] * 14 * q}
    if case["kind"] == "adjoint":
        cells, e = case["n"] ** 3, BYTES[case["storage"]]
        # The start state, the design field, the gradient; a forward and a transposed step per step.
        return {"bytes": cells * (19 * e + 4 + 4 + 1), "flops": cells * case["steps"] * (14 + 26) * 19}
    if case["kind"] == "coupled":
        cells, e = case["nx"] * case["ny"] * case["nz"], BYTES[case["storage"]]
        state = 2 * 19 * e + 2 * 7 * 4 + 2 * 4  # flow, temperature and fill in and out
        return {"bytes": cells * (state + 10 * 4) + 112 * case["particles"],
                "flops": case["steps"] * (cells * (14 * 19 + 60 + 100 + 40) + 150 * case["particles"])}
    cells, mesh = case["nx"] * case["ny"] * case["nz"], 4 * case["bands"] * (case["bands"] - 1)
    return {"bytes": cells + 72 * mesh, "flops": 20 * cells}


# ------------------------------------------------------------------ the same in 64 bits, in plain torch
def _lattice(name):
    if name == "d2q9":
        c = [(0, 0, 0), (1, 0, 0), (0, 1, 0), (1, 1, 0), (1, -1, 0)]
    else:
        c = [(0, 0, 0)] + [(x, y, z) for x in (1, 0, -1) for y in (1, 0, -1) for z in (1, 0, -1)
                           if (x, y, z) > (0, 0, 0) and (name == "d3q27" or abs(x) + abs(y) + abs(z) < 3)]
    c = c[:1] + [s for v in c[1:] for s in (v, tuple(-a for a in v))]
    by_length = {"d2q9": (4 / 9, 1 / 9, 1 / 36), "d3q19": (1 / 3, 1 / 18, 1 / 36),
                 "d3q27": (8 / 27, 2 / 27, 1 / 54, 1 / 216)}[name]
    return c, [by_length[sum(map(abs, v))] for v in c], [0] + [i + 1 if i % 2 else i - 1 for i in range(1, len(c))]


def _dot(c, u):
    s = 0.0
    for a, b in zip(c, u):
        if a:
            s = s + a * b
    return s


def _roll(f, c):
    """f(x - c): what arrives from the upstream cell on the periodic lattice."""
    if not any(c):
        return f
    return torch.roll(f, (c[2], c[1], c[0]), (0, 1, 2))


class _Exact:
    """Stream and collide on arriving populations, one tensor per direction, shape (nz, ny, nx)."""

    def __init__(self, lattice, tau, flags=None, gamma=None, force=(0.0, 0.0, 0.0), peak=0.0, lid=None):
        self.c, self.w, self.opp = _lattice(lattice)
        self.tau, self.force, self.peak, self.gamma, self.lid = tau, force, peak, gamma, lid
        self.flags = None if flags is None else torch.from_numpy(flags).cuda()
        if flags is not None:
            self.wall = self.flags >= 0x80
            self.inlet, self.outlet = self.flags == 1, self.flags == 2
            self.from_wall = [_roll(self.wall, c) for c in self.c]
            self.to_lid = [_roll(self.flags == 0x81, tuple(-a for a in c)) for c in self.c] if lid else None
            self.openings = bool(self.inlet.any() or self.outlet.any())

    def equilibrium(self, rho, u):
        uu = 1.5 * (u[0] * u[0] + u[1] * u[1] + u[2] * u[2])
        for c, w in zip(self.c, self.w):
            cu = 3 * _dot(c, u)
            yield w * rho * (1 + cu + 0.5 * cu * cu - uu)

    def start(self, rho, u):
        rho, u = rho.double(), [v.double() for v in u]
        if self.flags is not None:
            u = [torch.where(self.wall, 0.0, v) for v in u]
            self.wall_rho = rho
        return list(self.equilibrium(rho, u))

    def profile(self, shape):
        nz, ny, _ = shape
        e = (torch.arange(ny, device="cuda", dtype=torch.float64) - 0.5) / (ny - 2)
        p = (4 * e * (1 - e))[None, :, None]
        if nz > 1:
            t = (torch.arange(nz, device="cuda", dtype=torch.float64) - 0.5) / (nz - 2)
            p = p * (4 * t * (1 - t))[:, None, None]
        return self.peak * p

    def moments(self, f, local=None):
        rho = f[0].clone()
        for v in f[1:]:
            rho = rho + v
        a = [self.force[k] + (0.0 if local is None else local[k]) for k in range(3)]
        u = []
        for k in range(3):
            m = 0.0
            for c, v in zip(self.c, f):
                if c[k]:
                    m = m + c[k] * v
            u.append((m / rho if isinstance(m, torch.Tensor) else torch.zeros_like(rho)) + 0.5 * a[k])
        if self.flags is not None and self.openings:
            side = {k: sum(v for c, v in zip(self.c, f) if c[0] == k) for k in (-1, 0, 1)}
            p = self.profile(rho.shape)
            rho = torch.where(self.inlet, (side[0] + 2 * side[-1]) / (1 - p), rho)
            rho = torch.where(self.outlet, 1.0, rho)
            ux = torch.where(self.inlet, p, u[0])
            ux = torch.where(self.outlet, -1 + side[0] + 2 * side[1], ux)
            opening = self.inlet | self.outlet
            u = [ux] + [torch.where(opening, 0.0, v) for v in u[1:]]
        return rho, u, a

    def step(self, f, local=None):
        rho, u, a = self.moments(f, local)
        omega = 1 / self.tau
        forced = local is not None or any(self.force)
        uf = sum(rho * a[k] * u[k] for k in range(3)) if forced else None
        out = []
        opening = self.flags is not None and self.openings
        for d, feq in enumerate(self.equilibrium(rho, u)):
            v = f[d] - omega * (f[d] - feq)
            if forced:
                cf, cu = rho * _dot(self.c[d], a), _dot(self.c[d], u)
                v = v + self.w[d] * (1 - 0.5 * omega) * (3 * (cf - uf) + 9 * cu * cf)
            if self.gamma is not None:
                v = (1 - self.gamma) * v + self.gamma * f[self.opp[d]]
            out.append(torch.where(self.inlet | self.outlet, feq, v) if opening else v)
        if self.flags is None:
            return [_roll(v, c) for v, c in zip(out, self.c)]
        if self.lid:
            for d, c in enumerate(self.c):
                cu = _dot(c, self.lid)
                if cu:
                    out[d] = out[d] - torch.where(self.to_lid[d], 6 * self.w[d] * rho * cu, 0.0)
        # Arrivals: from the upstream cell, or this cell's own reflected population at a wall.  What a
        # lid reflects was corrected above and reaches no other fluid cell.
        return [torch.where(wall, out[self.opp[d]], _roll(out[d], self.c[d])) if d else out[0]
                for d, wall in enumerate(self.from_wall)]

    def fields(self, f, local=None):
        rho, u, _ = self.moments(f, local)
        if self.flags is not None:
            rho = torch.where(self.wall, self.wall_rho, rho)
            u = [torch.where(self.wall, 0.0, v) for v in u]
        return [rho, *u]


def _f32(v):
    return float(np.float32(v))


def _exact_flow(case, seed):
    flags, gamma, force, peak = _flow_setup(case, seed)
    lid = (_f32(LID), 0.0, 0.0) if case["scene"] == "cavity" else None
    x = _Exact(case["lattice"], _f32(TAU[case["scene"]]), flags, None if gamma is None else
               torch.from_numpy(gamma).cuda().double(), tuple(map(_f32, force)), _f32(peak), lid)
    if case["scene"] == "duct":
        one = torch.ones((case["nz"], case["ny"], case["nx"]), device="cuda", dtype=torch.float64)
        f = x.start(one, [_f32(INLET_PEAK) * one, 0 * one, 0 * one])
    else:
        rho, *u = _initial_fields(case, seed)
        f = x.start(rho, u)
    for _ in range(case["steps"]):
        f = x.step(f)
    out = x.fields(f)
    if not case["report"]:
        return out
    # Mass counts the walls' frozen density; energy and speed leave the walls out (u = 0 there).
    speed2 = out[1] ** 2 + out[2] ** 2 + out[3] ** 2
    return out + [[float(out[0].sum()), float(0.5 * (out[0] * speed2).sum()), float(speed2.max().sqrt())]]


def _exact_adjoint(case, seed):
    flags, body, blend, peak_value = _adjoint_setup(case, seed)
    gamma = torch.from_numpy(blend).cuda().double().requires_grad_(True)
    peak = torch.tensor(_f32(peak_value), device="cuda", dtype=torch.float64, requires_grad=True)
    x = _Exact("d3q19", _f32(0.6), flags, gamma, peak=peak)
    one = torch.ones(flags.shape, device="cuda", dtype=torch.float64)
    f = x.start(one, [(0.0 if body is None else _f32(INLET_PEAK)) * one, 0 * one, 0 * one])
    fluid = x.flags == 0
    if body is not None:
        b = torch.from_numpy(body).cuda()
        links = [_roll(b, c) & fluid if c[0] else None for c in x.c]
    planes = [(k, fluid[:, :, k]) for k in (1, case["n"] - 2)]

    def measure(f):
        if body is not None:
            return sum(-2 * c[0] * v[m].sum() for c, v, m in zip(x.c, f, links) if c[0])
        means = [sum(v[:, :, k] for v in f)[m].mean() / 3 for k, m in planes]
        return means[0] - means[1]

    J = 0.0
    for t in range(case["steps"]):
        f = list(checkpoint(lambda *a: tuple(x.step(list(a))), *f, use_reentrant=False))
        if t + 1 > case["steps"] - case["window"]:
            J = J + measure(f) / case["window"]
    J.backward()
    grad = torch.where(fluid, gamma.grad, 0.0)
    return [J.detach(), grad, torch.zeros_like(peak) if peak.grad is None else peak.grad]


def _shift(f, dx, dy, dz):
    """The neighbour's value f(x + d)."""
    return torch.roll(f, (-dz, -dy, -dx), (0, 1, 2))


def _exact_coupled(case, seed):
    x = _Exact("d3q19", _f32(TAU["periodic"]))
    rho0, *u0 = _initial_fields(case, seed)
    f = x.start(rho0, u0)
    heat, fill, parts = _coupled_fields(case, seed)
    phi = fill.double()
    c7 = [(0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1)]
    w7 = [0.25] + [0.125] * 6
    g7 = [w * heat.double() for w in w7]
    om7 = 1 / (0.5 + 4 * _f32(0.02))
    P = torch.from_numpy(parts).cuda().double()
    pos, vel, mass, resp = P[:, :3].clone(), P[:, 3:6].clone(), P[:, 6:7], P[:, 7:8]
    size = torch.tensor([case["nx"], case["ny"], case["nz"]], device="cuda")
    gravity = torch.tensor([0.0, _f32(-1e-5), 0.0], device="cuda", dtype=torch.float64)
    axes = ((1, 0, 0), (0, 1, 0), (0, 0, 1))
    grad = lambda s: [0.5 * (_shift(s, *e) - _shift(s, *(-a for a in e))) for e in axes]  # noqa: E731

    def interface(phi):
        g = grad(phi)
        mag = (g[0] ** 2 + g[1] ** 2 + g[2] ** 2).sqrt()
        n = [torch.where(mag > 1e-12, v / mag, 0.0) for v in g]
        kappa = sum(-0.5 * (_shift(v, *e) - _shift(v, *(-a for a in e))) for v, e in zip(n, axes))
        return g, n, kappa

    local = [torch.zeros_like(phi) for _ in range(3)]
    for _ in range(case["steps"]):
        _, u, _ = x.moments(f, local)
        local = [torch.zeros_like(phi) for _ in range(3)]
        g7 = [_roll(v, c) for v, c in zip(g7, c7)]
        T = sum(g7)
        g7 = [v - om7 * (v - w * T * (1 + 4 * _dot(c, u))) for v, w, c in zip(g7, w7, c7)]
        local[1] = local[1] + _f32(1e-5) * (sum(g7) - 300.0)
        flux = 0.0
        for k, e in enumerate(axes):
            face = 0.5 * (u[k] + _shift(u[k], *e))  # between the cell and its + neighbour
            through = torch.where(face >= 0, face * phi, face * _shift(phi, *e))
            flux = flux + through - _shift(through, *(-a for a in e))
        phi = (phi - 0.5 * flux).clamp(0, 1)
        g, n, kappa = interface(phi)
        local = [a + _f32(1e-4) * kappa * v for a, v in zip(local, g)]
        base = pos.floor().long()
        frac = pos - base
        V = torch.zeros_like(vel)
        corners = []
        for dx in (0, 1):
            for dy in (0, 1):
                for dz in (0, 1):
                    d = torch.tensor([dx, dy, dz], device="cuda")
                    at = (base + d) % size
                    w = torch.where(d.bool(), frac, 1 - frac).prod(1, keepdim=True)
                    cell = (at[:, 2] * case["ny"] + at[:, 1]) * case["nx"] + at[:, 0]
                    corners.append((cell, w))
                    V += w * torch.stack([c.reshape(-1)[cell] for c in u], 1)
        drag = mass * (V - vel) / resp
        if case["two_way"]:
            for cell, w in corners:
                for k in range(3):
                    local[k] = local[k].reshape(-1).index_add(0, cell, -(w * drag)[:, k]).reshape(phi.shape)
        vel = vel + drag / mass + gravity
        pos = (pos + vel) % size
        f = x.step(f, local)
    rho, *u = x.fields(f, local)
    du = [grad(v) for v in u]
    s2 = sum((0.5 * (du[i][j] + du[j][i])) ** 2 for i in range(3) for j in range(3))
    o2 = sum((0.5 * (du[i][j] - du[j][i])) ** 2 for i in range(3) for j in range(3))
    _, n, kappa = interface(phi)
    return [rho, *u, 0.5 * (o2 - s2), sum(g7), phi, *n, kappa, torch.cat([pos, vel, mass, resp], 1)]


def exact(case, seed):
    if case["kind"] == "flow":
        with torch.no_grad():
            return _exact_flow(case, seed)
    if case["kind"] == "adjoint":
        return _exact_adjoint(case, seed)
    if case["kind"] == "coupled":
        with torch.no_grad():
            return _exact_coupled(case, seed)
    return None  # a mask of whole numbers
