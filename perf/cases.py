"""The engine's working range as a set of timed cases.

``listed()`` names the cases, ``draw(rng)`` gives more of the same ranges, ``prepare`` builds
what a program has in hand before the call (the lattice with its fields uploaded, or the
surface and the face codes), ``run`` is one pass through the public entry points, ``work`` the
bytes and operations a pass cannot do without, and ``exact`` the outputs in 64 bits from a
plain torch restatement of the step (no code of the engine but the builders of its inputs).

A pass of a flow case is one output interval of the reference's time loop (ns.cpp:509-603):
so many steps, then the fields and sums the host reads at an output step.  Every flow starts
from a seeded, divergence-free disturbance on its base flow.

Kinds, and what each stands for in use:
  cavity      lid-driven cavity (testCases/cavityFlow), the validation flow: small lattices,
              where launches and latency count; FP32, FP64 (the accuracy reference), 2-D or 3-D
  wake        flow past a cylinder, interpolated bounce-back, the drag and lift history read
              every few steps (lbffs_reduce) and the velocity at the end
  backstep    the benchmark's workload, Smagorinsky LES over a backward-facing step, on half
              its length: the production size, launch shape autotuned as the benchmark does
  bluff       D3Q27 cumulant + WALE around a procedural body with FP64 q-distances
  ensemble    many small lattices advanced together (a parameter sweep)
  rotor       moving walls: immersed-boundary markers turning in a forced channel
  checkpoint  a short interval followed by everything an output step reads: density and
              velocity recomputed from the populations, tauSGS and the populations themselves
  geometry    the preprocessing of an LES case: solid flags, their neighbours and the signed
              wall distance from the walls' triangles
"""
from __future__ import annotations

import itertools
import math

import numpy as np
import torch

import lbffs_amd as lb
from lbffs_amd import cases, geometry

STORAGE = {"f32": lb.STORE_F32, "f16": lb.STORE_F16DEV, "bf16": lb.STORE_BF16DEV, "f64": lb.STORE_F64}
WIDTH = {"f32": 4, "f16": 2, "bf16": 2, "f64": 8}


def listed():
    return [
        # the smallest run: 32^3 cells, a kernel of a few microseconds per step
        dict(name="cavity_32_f32", kind="cavity", n=32, nz=32, storage="f32", steps=100),
        # the 64^3 validation cavity in the FP64 form that accuracy is measured against
        dict(name="cavity_64_f64", kind="cavity", n=64, nz=64, storage="f64", steps=100),
        # Re 100 cylinder wake at its stated size: force history every 20 steps
        dict(name="wake_f32", kind="wake", nx=400, ny=160, nz=16, storage="f32", every=20, samples=10),
        # the same in 16-bit storage on odd sizes (no row is a whole number of waves)
        dict(name="wake_odd_f16", kind="wake", nx=421, ny=167, nz=21, storage="f16", every=20, samples=10),
        # the benchmark's workload, half its length, both storage forms
        dict(name="backstep_f32", kind="backstep", nx=768, ny=192, nz=128, storage="f32", steps=300),
        dict(name="backstep_f16", kind="backstep", nx=768, ny=192, nz=128, storage="f16", steps=300),
        # D3Q27 wind tunnel: 16-bit at production proportions, FP32 on odd sizes
        dict(name="bluff_bf16", kind="bluff", nx=448, ny=168, nz=140, storage="bf16", every=50, samples=3),
        dict(name="bluff_odd_f32", kind="bluff", nx=257, ny=97, nz=81, storage="f32", every=50, samples=3),
        # a sweep of cavities and cylinder channels of edge 24 to 96
        dict(name="ensemble_f16", kind="ensemble", count=60, lo=24, hi=96, storage="f16", steps=100),
        # a turning ring of 6400 markers
        dict(name="rotor_f32", kind="rotor", nx=192, ny=96, nz=64, markers=6400, storage="f32", steps=200),
        # output step after a short interval
        dict(name="checkpoint_f32", kind="checkpoint", nx=160, ny=128, nz=128, storage="f32", steps=50),
        # LES preprocessing of a body of 31 840 triangles
        dict(name="geometry", kind="geometry", nx=320, ny=192, nz=160, n_lat=100, n_lon=160),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cavity", "cavity", "wake", "wake", "backstep", "backstep", "bluff", "bluff", "ensemble",
                       "rotor", "checkpoint", "geometry"])
    if kind == "cavity":
        if rng.random() < 0.4:
            return dict(kind=kind, n=_log(rng, 48, 600), nz=1, storage=rng.choice(["f32", "f64"]),
                        steps=rng.randint(40, 160))
        n = _log(rng, 24, 160)
        return dict(kind=kind, n=n, nz=n, storage=rng.choice(["f32", "f32", "f16", "f64"]),
                    steps=rng.randint(40, 120))
    if kind == "wake":
        nx = _log(rng, 120, 640)
        return dict(kind=kind, nx=nx, ny=max(48, int(nx * rng.uniform(0.3, 0.5))), nz=_log(rng, 6, 40),
                    storage=rng.choice(["f32", "f16", "f64"]), every=rng.randint(8, 30), samples=rng.randint(4, 12))
    if kind == "backstep":
        ny = _log(rng, 48, 170)
        return dict(kind=kind, nx=int(ny * rng.uniform(3.0, 5.0)), ny=ny, nz=int(ny * rng.uniform(0.4, 0.8)),
                    storage=rng.choice(["f32", "f16", "bf16"]), steps=rng.randint(60, 200))
    if kind == "bluff":
        nx = _log(rng, 120, 330)
        return dict(kind=kind, nx=nx, ny=int(nx * rng.uniform(0.35, 0.45)), nz=int(nx * rng.uniform(0.3, 0.4)),
                    storage=rng.choice(["f32", "bf16", "f16"]), every=rng.randint(15, 50), samples=rng.randint(1, 3))
    if kind == "ensemble":
        lo = rng.randint(20, 40)
        return dict(kind=kind, count=_log(rng, 8, 60), lo=lo, hi=rng.randint(lo + 10, 96),
                    storage=rng.choice(["f16", "f32"]), steps=rng.randint(40, 100))
    if kind == "rotor":
        ny = _log(rng, 48, 128)
        return dict(kind=kind, nx=int(ny * rng.uniform(1.5, 2.2)), ny=ny, nz=int(ny * rng.uniform(0.3, 0.8)),
                    markers=_log(rng, 400, 12000), storage=rng.choice(["f32", "f64"]), steps=rng.randint(50, 200))
    if kind == "checkpoint":
        return dict(kind=kind, nx=_log(rng, 64, 180), ny=_log(rng, 64, 150), nz=_log(rng, 32, 140),
                    storage=rng.choice(["f32", "f16"]), steps=rng.randint(10, 60))
    nx = _log(rng, 120, 330)
    n_lat = _log(rng, 24, 100)
    return dict(kind="geometry", nx=nx, ny=int(nx * rng.uniform(0.45, 0.62)), nz=int(nx * rng.uniform(0.4, 0.52)),
                n_lat=n_lat, n_lon=int(1.6 * n_lat))


# ---- inputs ----

C19 = ([0, 1, -1, 0, 0, 0, 0, 1, -1, 1, -1, 1, -1, 1, -1, 0, 0, 0, 0],
       [0, 0, 0, 1, -1, 0, 0, 1, -1, -1, 1, 0, 0, 0, 0, 1, -1, 1, -1],
       [0, 0, 0, 0, 0, 1, -1, 0, 0, 0, 0, 1, -1, -1, 1, 1, -1, -1, 1])
C27 = (C19[0] + [1, -1, -1, 1, 1, -1, 1, -1], C19[1] + [1, -1, 1, -1, -1, 1, 1, -1],
       C19[2] + [1, -1, 1, -1, 1, -1, -1, 1])


def _lattice(q):
    c = list(zip(*(C27 if q == 27 else C19)))
    by_speed = [8 / 27, 2 / 27, 1 / 54, 1 / 216] if q == 27 else [1 / 3, 1 / 18, 1 / 36]
    return c, [by_speed[sum(map(abs, d))] for d in c]


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _disturb(c, rng, base, amp):
    """Populations of the base flow (u, v, w) with four divergence-free Fourier modes of amplitude amp."""
    dev = _device()
    x, y, z = (torch.arange(n, device=dev, dtype=torch.float32) for n in (c.nx, c.ny, c.nz))
    vel = [torch.full((c.nz, c.ny, c.nx), float(b), device=dev) for b in base]
    rho = torch.ones_like(vel[0])
    for m in range(4):
        k = [2 * math.pi * rng.integers(1, 4) / n if n > 1 else 0.0 for n in (c.nx, c.ny, c.nz)]
        d = np.cross(k, rng.standard_normal(3))
        d /= np.linalg.norm(d)
        if c.nz == 1:
            d = np.array([k[1], -k[0], 0.0]) / math.hypot(k[0], k[1])
        ph = (k[0] * x)[None, None, :] + (k[1] * y)[None, :, None] + (k[2] * z)[:, None, None]
        ph += rng.uniform(0, 2 * math.pi)
        wave = torch.sin(ph)
        for a in range(3):
            vel[a] += float(amp * d[a]) * wave
        rho += 5e-4 * torch.cos(ph)
    fluid = torch.from_numpy(c.arrays["solid"].reshape(c.nz, c.ny, c.nx)).to(dev) == 0
    vel = [v * fluid for v in vel]
    dirs, w = _lattice(c.q)
    u2 = 1.5 * (vel[0] ** 2 + vel[1] ** 2 + vel[2] ** 2)
    f = torch.empty((c.q, c.N), device=dev)
    for q, (cx, cy, cz) in enumerate(dirs):
        cu = cx * vel[0] + cy * vel[1] + cz * vel[2]
        f[q] = (w[q] * (rho + 3 * cu + 4.5 * cu * cu - u2)).reshape(-1)
    c.arrays["f"] = f.reshape(-1).cpu().numpy()


def _base_case(case, seed):
    """The lattice and its fields, as the builders of lbffs_amd.cases make them."""
    kind, rng = case["kind"], np.random.default_rng(seed)
    if kind == "cavity":
        c = cases.cavity(case["n"], nz=case["nz"], Re=float(rng.uniform(100, 400)))
        _disturb(c, rng, (0, 0, 0), 0.01)
    elif kind == "wake":
        nx, ny = case["nx"], case["ny"]
        c = cases.cylinder_channel(nx, ny, case["nz"], D=ny // 4, cx=nx // 4, cy=ny // 2, seed=seed, ibb=True)
        _disturb(c, rng, (0.05, 0, 0), 0.005)
    elif kind == "backstep":
        c = cases.backward_step(case["nx"], case["ny"], case["nz"], H=case["ny"] // 3, spz_cells=max(8, case["nx"] // 24),
                                seed=seed)
        _disturb(c, rng, (0.05, 0, 0), 0.005)
    elif kind == "bluff":
        D = case["nx"] * 80.0 / 1024.0
        n_lat = max(16, int(250 * D / 80.0))
        c = cases.bluff_body(case["nx"], case["ny"], case["nz"], D=D, spz_cells=max(6, case["nx"] // 16), seed=seed,
                             n_lat=n_lat, n_lon=int(1.6 * n_lat))
        _disturb(c, rng, (0.04, 0, 0), 0.004)
    elif kind in ("rotor", "checkpoint"):
        c = cases.channel(case["nx"], case["ny"], case["nz"], tau=0.6, force=1e-6, sgs=lb.SGS_WALE)
        _disturb(c, rng, (0.02, 0, 0), 0.01)
    return c


def _ensemble_specs(case, seed):
    # kinds and edges belong to the case, the Reynolds numbers to the seed
    rng = np.random.default_rng(seed)
    specs = cases.ensemble_specs(case["count"], edges=(case["lo"], case["hi"]))
    return [(kind, edge, float(rng.uniform(50.0, 400.0))) for kind, edge, _ in specs]


def _ring(case, seed):
    """Markers of a closed cylinder turning about the channel's middle, and its motion."""
    rng = np.random.default_rng(seed + 1)
    R = 0.25 * case["ny"]
    layers = max(2, int(math.sqrt(case["markers"] * 0.3 * case["nz"] / (2 * math.pi * R))))
    per = max(2, case["markers"] // layers)
    centre = (case["nx"] / 2 + rng.uniform(-1, 1), case["ny"] / 2 + rng.uniform(-1, 1), 0.0)
    t = 2 * math.pi * np.arange(per) / per + rng.uniform(0, 1)
    zs = 0.35 * case["nz"] + 0.3 * case["nz"] * np.arange(layers) / layers
    T, Z = np.meshgrid(t, zs, indexing="ij")
    xyz = np.stack([centre[0] + R * np.cos(T), centre[1] + R * np.sin(T), Z], axis=-1).reshape(-1, 3)
    return xyz.astype(np.float32), dict(trans=(1e-3, 0.0, 0.0), center=centre, axis=(0.0, 0.0, 1.0), omega=0.02 / R)


def _surface(case, seed):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    rng = np.random.default_rng(seed)
    at = [n / 2 + rng.uniform(-2, 2) for n in (nx * 0.7, ny, nz)]
    return geometry.procedural_body(at, 0.25 * min(ny, nz), n_lat=case["n_lat"], n_lon=case["n_lon"], seed=seed)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "geometry":
        codes = {f: ("Cyclic", "Cyclic", "Cyclic") for f in cases.FACES}
        codes["nyMin"] = codes["nyMax"] = ("Cyclic", "BounceBack", "Cyclic")
        cin, un = cases.units(case["nx"], case["ny"], case["nz"], 1.0, 1.0, 0.05, 1e-4, face_codes=codes)
        return dict(case=case, surface=_surface(case, seed), codes=cases.build_faces(cin, un)[0][1:])
    if kind == "ensemble":
        specs = _ensemble_specs(case, seed)
        built = [cases.ensemble_case(s, d, seed) for d, s in enumerate(specs)]
        for d, c in enumerate(built):
            _disturb(c, np.random.default_rng([seed, d]), (0, 0, 0), 0.01)
        batch = lb.Batch([(c.nx, c.ny, c.nz, c.omega0) for c in built], storage=STORAGE[case["storage"]])
        for c, lat in zip(built, batch.lattice):
            c.upload_to(lat)
        return dict(case=case, batch=batch, params=[c.params for c in built])
    c = _base_case(case, seed)
    lat = lb.Lattice(c.nx, c.ny, c.nz, q=c.q, storage=STORAGE[case["storage"]], sgs=c.sgs, collision=c.coll,
                     omega0=c.omega0)
    c.upload_to(lat)
    if kind == "rotor":
        xyz, motion = _ring(case, seed)
        lat.ibm_set_markers(xyz)
        lat.ibm_set_motion(**motion)
    if kind == "backstep":
        lat.autotune(10, **c.params)  # long runs choose their launch shape once
    return dict(case=case, lat=lat, params=c.params)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "geometry":
        return geometry.preprocess(state["surface"], 19, case["nx"], case["ny"], case["nz"], True, *state["codes"])
    if kind == "ensemble":
        b = state["batch"]
        b.step(case["steps"], state["params"])
        return dict(sums=np.stack([lat.reduce() for lat in b.lattice]), u=[lat.download("u") for lat in b.lattice])
    lat, p = state["lat"], state["params"]
    if kind in ("wake", "bluff"):
        sums = []
        for _ in range(case["samples"]):
            lat.step(case["every"], **p)
            sums.append(lat.reduce())
        return dict(sums=np.stack(sums), **{k: lat.download(k) for k in "uvw"})
    lat.step(case["steps"], **p)
    if kind == "checkpoint":
        return dict(lat.output_macros(p["dpdx"]), tauSGS=lat.download("tauSGS"), f=lat.download("f"))
    out = {k: lat.download(k) for k in ("rho", "u", "v", "w") if k != "w" or lat.nz > 1}  # (2-D: w is zero)
    if kind == "rotor":
        out.update(positions=lat.ibm_download(lb.IBM_POSITIONS), forcing=lat.ibm_download(lb.IBM_FORCING))
    return out


def work(case):
    """Bytes: each step reads and writes every population once and, with WALE, the velocity its
    gradient needs; the outputs are read on the device and written on the host once.
    Operations: about 400 (D3Q19) or 1000 (D3Q27) per cell update."""
    kind = case["kind"]
    if kind == "geometry":
        n = case["nx"] * case["ny"] * case["nz"]
        tris = 2 * case["n_lon"] * (case["n_lat"] - 1)
        # flags, neighbours and distances out; each triangle's vertices, centroid and normal in
        return dict(bytes=6.0 * n + 60.0 * tris, flops=100.0 * tris)
    s, q = WIDTH[case["storage"]], 27 if kind == "bluff" else 19
    real = 8 if case["storage"] == "f64" else 4
    if kind == "ensemble":
        n = sum(edge ** 3 for _, edge, _ in _ensemble_specs(case, 0))
    elif kind == "cavity":
        n = case["n"] ** 2 * case["nz"]
    else:
        n = case["nx"] * case["ny"] * case["nz"]
    sampled = kind in ("wake", "bluff")
    steps = case["every"] * case["samples"] if sampled else case["steps"]
    per_cell = 2 * q * s + (0 if kind == "backstep" else 6 * real)
    out = {"ensemble": 1, "checkpoint": 5 + q}.get(kind, 3 if sampled else 4) * real
    sums = (case["samples"] if sampled else 1 if kind == "ensemble" else 0) * (q * s + 3 * real)
    return dict(bytes=float(n) * (steps * per_cell + 2 * out + sums),
                flops=float(n) * steps * (1000.0 if q == 27 else 400.0))


# ---- the outputs in 64 bits ----

def exact(case, seed):
    """The step restated in plain torch at 64 bits: previous-step neighbour reads of the
    moments (the engine's rule), every other formula as the reference's kernels write it.
    None where it takes over about 20 seconds (the large lattices and ensembles), and for the
    geometry, whose flags are whole numbers and whose distances are sums over all triangles
    near a cell."""
    kind = case["kind"]
    if kind == "geometry":
        return None
    sampled = kind in ("wake", "bluff")
    steps = case["every"] * case["samples"] if sampled else case["steps"]
    n = work(case)["bytes"] / steps / 100.0  # cells, near enough
    if kind == "ensemble":
        if case["count"] * steps > 2500:
            return None
        fields = []
        for d, spec in enumerate(_ensemble_specs(case, seed)):
            c = cases.ensemble_case(spec, d, seed)
            _disturb(c, np.random.default_rng([seed, d]), (0, 0, 0), 0.01)
            e = _Exact(c)
            e.steps(steps)
            fields.append((e.sums(), e.vel[0].reshape(-1)))
        return dict(sums=torch.stack([a for a, _ in fields]), u=[u for _, u in fields])
    if n * steps > 1.5e9:
        return None
    c = _base_case(case, seed)
    if kind == "bluff":  # the body's q-distances are an input: cast once, as prepare does
        with lb.Lattice(c.nx, c.ny, c.nz, q=27, collision=c.coll, omega0=c.omega0) as lat:
            c.upload_to(lat)
            c.arrays["qlink"] = lat.download("qlink")
    e = _Exact(c)
    if kind == "rotor":
        e.markers(*_ring(case, seed))
    if sampled:
        sums = []
        for _ in range(case["samples"]):
            e.steps(case["every"])
            sums.append(e.sums())
        return dict(sums=torch.stack(sums), **{k: a.reshape(-1) for k, a in zip("uvw", e.vel)})
    e.steps(steps)
    if kind == "checkpoint":
        rho = e.f.sum(0)
        vel = [torch.einsum("q,qn->n", e.c[:, a], e.f) / rho for a in range(3)]
        vel[0] = vel[0] + 0.5 * e.p["dpdx"] / rho
        return dict(rho=rho, u=vel[0], v=vel[1], w=vel[2], tauSGS=e.tau_sgs.reshape(-1), f=e.f.reshape(-1))
    out = dict(rho=e.rho.reshape(-1), **{k: a.reshape(-1) for k, a in zip("uvw" if c.nz > 1 else "uv", e.vel)})
    if kind == "rotor":
        out.update(positions=e.xyz.reshape(-1), forcing=e.forcing.T.reshape(-1))
    return out


class _Exact:
    """One lattice in float64.  Arrays are (nz, ny, nx), populations (q, cells)."""

    def __init__(self, c):
        self.q, self.sgs, self.p = c.q, c.sgs, c.params
        self.shape = (c.nz, c.ny, c.nx)
        self.dev = _device()
        self.dirs, weights = _lattice(c.q)
        self.w = self.put(weights)
        self.c = self.put(self.dirs)
        self.opp = [self.dirs.index(tuple(-x for x in d)) for d in self.dirs]
        a = c.arrays
        self.f = self.put(a["f"]).reshape(c.q, -1)
        grid = lambda k, t=torch.float64: torch.as_tensor(a[k], device=self.dev).to(t).reshape(self.shape)  # noqa: E731
        self.solid = grid("solid", torch.int32) != 0
        self.omega, self.sdf = grid("omega"), grid("sdf")
        self.wall_vel = [grid(k) for k in ("u0", "v0", "w0")]
        self.code = [grid(k, torch.int32) for k in ("boundary1", "boundary2", "boundary3")]
        pos = torch.meshgrid(*(torch.arange(n, device=self.dev) for n in self.shape), indexing="ij")
        self.pos, self.n = pos[::-1], self.shape[::-1]  # by axis x, y, z
        edge = [(p == 0) | (p == n - 1) for p, n in zip(self.pos, self.n)]
        xy = edge[0] & edge[1]
        flat = (self.code[2] == 0) | (self.n[2] == 1)
        self.corner = torch.where(flat, xy, xy | (edge[0] & edge[2]) | (edge[1] & edge[2]))
        self.stopped = [[self.wall(ax) & (self.pos[ax] == e) for e in (0, self.n[ax] - 1)] for ax in range(3)]
        nei = (grid("neiSolid", torch.int32) == 1) & ~self.solid
        self.nei = nei.reshape(-1).nonzero()[:, 0]
        self.qlink = self.put(a["qlink"]).reshape(c.q, -1)[:, self.nei] if self.p.get("ibb") else None
        self.rho, self.tau_sgs, *vel = (torch.zeros(self.shape, dtype=torch.float64, device=self.dev) for _ in range(5))
        self.vel = vel
        self.force = [torch.zeros_like(self.rho) for _ in range(3)]
        self.sponge = []
        for ax in range(3):
            for hi in (0, 1):
                mid = [n // 2 for n in self.n]
                mid[ax] = (self.n[ax] - 1) * hi
                if int(self.code[ax][mid[2], mid[1], mid[0]]) in (3, 6):
                    self.sponge.append((ax, hi))
        # the moments x^a y^b z^c that determine the populations: D3Q19 has no direction along all three axes
        self.powers = [t for t in itertools.product(range(3), repeat=3) if c.q == 27 or 0 in t]
        self.moment = torch.stack([torch.prod(self.c ** self.put(t), dim=1) for t in self.powers])
        self.back = torch.linalg.inv(self.moment)
        self.xyz = None

    def put(self, a):
        return torch.as_tensor(np.asarray(a, np.float64), device=self.dev)

    def wall(self, ax):
        code = self.code[ax]
        return (code == 1) | (code >= 4)

    def at(self, ax, i):
        s = [slice(None)] * 3
        s[2 - ax] = i
        return tuple(s)

    def cells(self, f):
        return f.reshape((self.q,) + self.shape)

    def steps(self, n):
        for _ in range(n):
            self.step()

    def mirrored(self, q):
        """Per cell the direction a wall turns q into: reversed, or across a Symmetry face only its normal component."""
        part = torch.full(self.shape, self.opp[q], device=self.dev)
        for ax in range(3):
            d = list(self.dirs[q])
            if d[ax]:
                d[ax] = -d[ax]
                part[self.code[ax] == 4] = self.dirs.index(tuple(d))
            else:
                part[self.code[ax] == 4] = self.opp[q]
        return part

    def stream(self):
        old = self.cells(self.f)
        new = torch.empty_like(old)
        for q, d in enumerate(self.dirs):
            new[q] = torch.roll(old[q], d[::-1], (0, 1, 2))
            if q == 0:
                continue
            hit = torch.zeros_like(self.solid)
            for ax in range(3):
                if d[ax] and not (ax == 2 and self.n[2] == 1):
                    hit |= self.stopped[ax][0 if d[ax] > 0 else 1]
            ic = hit.reshape(-1).nonzero()[:, 0]
            if len(ic):
                if bool((self.code[1] == 4).any() | (self.code[2] == 4).any()):
                    back = self.f[self.mirrored(q).reshape(-1)[ic], ic]
                else:
                    back = self.f[self.opp[q], ic]
                new[q].view(-1)[ic] = back
        return new

    def faces(self, f):
        """Fixed-velocity faces (moving-wall bounce-back with the Zou-He density), then convective outlets."""
        old = self.cells(self.f)
        for ax in range(3):
            for hi in (0, 1):
                at = self.at(ax, -1 if hi else 0)
                fixed = (self.code[ax][at] == 5) & ~self.corner[at]
                if not bool(fixed.any()):
                    continue
                out = 1 if hi else -1
                face = f[(slice(None),) + at]
                un = self.wall_vel[ax][at]
                along = sum(face[q] for q, d in enumerate(self.dirs) if d[ax] == 0)
                leave = sum(face[q] for q, d in enumerate(self.dirs) if d[ax] == out)
                rho = (along + 2 * leave) / (1 + out * un)
                inner = self.at(ax, (-1 if ax == 0 else -2) if hi else 1)
                rho = torch.where(un * out > 0, self.rho[inner], rho)
                for q, d in enumerate(self.dirs):
                    if d[ax] == -out:
                        cu = sum(x * v[at] for x, v in zip(d, self.wall_vel))
                        face[q] = torch.where(fixed, face[q] + 6 * self.w[q] * rho * cu, face[q])
        for ax in range(3):
            for hi in (0, 1):
                at, inner = self.at(ax, -1 if hi else 0), self.at(ax, -2 if hi else 1)
                open_ = self.code[ax][at] == 3
                if not bool(open_.any()):
                    continue
                rate = 1 / math.sqrt(3) - self.vel[ax][at]
                for q, d in enumerate(self.dirs):
                    if d[ax] == (-1 if hi else 1):
                        g = (slice(None),)
                        v = rate * old[q][inner] + (1 - rate) * old[q][at]
                        f[(q,) + at] = torch.where(open_, v, f[(q,) + at])
        return f

    def links(self, f):
        """Bounce-back on the links to solid cells (interpolated where q-distances are given) and its momentum."""
        f = f.reshape(self.q, -1)
        ic = self.nei
        F = torch.zeros((3, len(ic)), dtype=torch.float64, device=self.dev)
        x, y, z = (p.reshape(-1)[ic] for p in self.pos)

        def cell(d, s):
            nx, ny, nz = self.n
            return (x + s * d[0]) % nx + nx * ((y + s * d[1]) % ny + ny * ((z + s * d[2]) % nz))

        flat = [v.reshape(-1) for v in self.vel]
        solid = self.solid.reshape(-1)
        om = 1 / (1 / self.omega.reshape(-1)[ic] + self.tau_sgs.reshape(-1)[ic])
        rho, vel = self.rho.reshape(-1)[ic], [v[ic] for v in flat]
        u2 = sum(v * v for v in vel)
        for q, d in enumerate(self.dirs[1:], 1):
            hit = solid[cell(d, -1)]
            fb = self.f[self.opp[q], ic]
            new = fb
            if self.qlink is not None:
                ql, nb = self.qlink[q], cell(d, 1)
                uc = -sum(v * s for v, s in zip(vel, d))
                near = -sum(v[nb] * s for v, s in zip(flat, d))
                slip = torch.where(ql <= 0.5, near, (1 - 1 / ql) * uc)
                feq = self.w[q] * (rho + 3 * slip + 4.5 * uc * uc - 1.5 * u2)
                chi = om * (2 * ql - 1) / torch.where(ql <= 0.5, 1 - 2 * om, torch.ones_like(om))
                new = (1 - chi) * fb + chi * feq
            f[q, ic] = torch.where(hit, new, f[q, ic])
            for a in range(3):
                F[a] -= torch.where(hit, (fb + new) * d[a], torch.zeros_like(fb))
        self.force = []
        for a in range(3):
            g = torch.zeros(f.shape[1], dtype=torch.float64, device=self.dev)
            g[ic] = F[a]
            self.force.append(g)
        return f

    def gradient(self, old, new, ax):
        """Central differences of the previous step inside, one-sided with the cell's new value on a face (0 at k = 0)."""
        n = self.n[ax]
        g = torch.zeros_like(old)
        if n == 1:
            return g
        if n > 2:
            g[self.at(ax, slice(1, -1))] = 0.5 * (old[self.at(ax, slice(2, None))] - old[self.at(ax, slice(0, -2))])
        if ax < 2:
            g[self.at(ax, 0)] = old[self.at(ax, 1)] - new[self.at(ax, 0)]
        g[self.at(ax, -1)] = new[self.at(ax, -1)] - old[self.at(ax, -2)]
        return g

    def wale(self, new):
        G = [[self.gradient(self.vel[a], new[a], b) for b in range(3)] for a in range(3)]  # du_a / dx_b
        S = [[0.5 * (G[a][b] + G[b][a]) for b in range(3)] for a in range(3)]
        SS = sum(S[a][b] ** 2 for a in range(3) for b in range(3))
        G2 = [[sum(G[a][c] * G[c][b] for c in range(3)) for b in range(3)] for a in range(3)]
        third = (G2[0][0] + G2[1][1] + G2[2][2]) / 3
        D = 0
        for a in range(3):
            for b in range(3):
                d = 0.5 * (G2[a][b] + G2[b][a]) - (third if a == b else 0)
                D = D + d * d
        on = (SS > 1e-24) & (D > 1e-24)
        SS, D = (torch.where(on, t, torch.ones_like(t)) for t in (SS, D))
        return torch.where(on, 9 * 0.325 ** 2 * D ** 1.5 / (SS ** 2.5 + D ** 1.25), torch.zeros_like(SS))

    def smagorinsky(self, rho, vel, second, tau):
        P2 = 0
        for a in range(3):
            for b in range(3):
                P = second[a][b] - (rho / 3 if a == b else 0) - vel[a] * vel[b]
                P2 = P2 + P * P
        Cs = float(np.float32(self.p["Cs"]))
        t = 0.5 * self.p["LES"] * (torch.sqrt(tau * tau + 18 * math.sqrt(2) * Cs * Cs * torch.sqrt(P2) / rho) - tau)
        damp = torch.clamp(0.41 * self.sdf / Cs, max=1.0) ** 2
        return torch.where((self.sdf != 10000) & (self.sdf > 0), t * damp, t)

    def step(self):
        f = self.links(self.faces(self.stream()))
        dpdx = float(np.float32(self.p["dpdx"]))
        M = dict(zip(self.powers, (self.moment @ f).reshape((-1,) + self.shape)))
        rho = M[0, 0, 0]
        half = 0.5 * dpdx / rho
        vel = [M[1, 0, 0] / rho + half, M[0, 1, 0] / rho, M[0, 0, 1] / rho]
        fluid = ~self.solid
        tau = 1 / self.omega
        if self.sgs == lb.SGS_WALE:
            sgs = self.wale([torch.where(fluid, v, torch.zeros_like(v)) for v in vel])
        elif self.sgs == lb.SGS_SMAGORINSKY:
            e = [(1, 0, 0), (0, 1, 0), (0, 0, 1)]
            second = [[M[tuple(x + y for x, y in zip(a, b))] for b in e] for a in e]
            sgs = self.smagorinsky(rho, vel, second, tau)
        else:
            sgs = torch.zeros_like(rho)
        spz = float(np.float32(self.p["spzWidth"]))
        for ax, hi in self.sponge:
            pos, n = self.pos[ax].double(), self.n[ax]
            frac = ((n - pos) if hi else pos) / (n * spz)
            inside = pos > n * (1 - spz) if hi else pos < n * spz
            tau = torch.where(inside, (1 - frac) * (1 - sgs) + frac * tau, tau)
        om = 1 / (tau + sgs)
        if self.q == 19:
            out = self.regularized(M, rho, vel, half, om, dpdx)
        else:
            out = self.cumulant(M, rho, vel, om)
        self.f = torch.where(self.solid.reshape(-1), self.f, out)
        keep = lambda a: torch.where(fluid, a, torch.zeros_like(a))  # noqa: E731
        self.rho, self.vel, self.tau_sgs = keep(rho), [keep(v) for v in vel], keep(sgs)
        if self.xyz is not None:
            self.turn()

    def regularized(self, M, rho, vel, half, om, dpdx):
        """Second-order moments relaxed (trace at omegaB), third and fourth order rebuilt recursively from them."""
        ob = float(np.float32(self.p["omegaB"]))
        u = [vel[0] - half, vel[1], vel[2]]
        unit = [(1, 0, 0), (0, 1, 0), (0, 0, 1)]
        add = lambda *t: tuple(map(sum, zip(*t)))  # noqa: E731
        N, R = {}, {}
        for a in range(3):
            for b in range(a, 3):
                k = add(unit[a], unit[b])
                R[k] = M[k] / rho - (1 / 3 if a == b else 0)
                N[k] = R[k] - u[a] * u[b]
        trace = sum(N[add(e, e)] for e in unit) * (ob - om) / 3
        T = {(0, 0, 0): torch.ones_like(rho)}
        for a in range(3):
            T[unit[a]] = u[a]
            for b in range(a, 3):
                k = add(unit[a], unit[b])
                T[k] = R[k] - om * N[k] - (trace if a == b else 0)
        H = dict(T)
        for a in range(3):
            H[add(unit[a], unit[a])] = T[add(unit[a], unit[a])] + 1 / 3
            for b in range(3):
                if a == b:
                    continue
                aa, ab, bb = add(unit[a], unit[a]), add(unit[a], unit[b]), add(unit[b], unit[b])
                H[add(aa, unit[b])] = u[a] * u[a] * u[b] + (1 - om) * (u[b] * N[aa] + 2 * u[a] * N[ab]) + u[b] / 3
                H[add(aa, bb)] = (u[a] ** 2 * u[b] ** 2 + (1 - om) * (u[b] ** 2 * N[aa] + u[a] ** 2 * N[bb]
                                  + 4 * u[a] * u[b] * N[ab]) + (T[aa] + T[bb]) / 3 + 1 / 9)
        out = self.back @ torch.stack([H[t].reshape(-1) for t in self.powers])
        return rho.reshape(-1) * (out + 3 * dpdx * (self.w * self.c[:, 0])[:, None])

    def cumulant(self, M, rho, vel, o1):
        """Parametrized cumulants (Geier et al. 2017) about the shifted velocity, as the reference's D3Q27 kernel."""
        o2, clim = (float(np.float32(self.p[k])) for k in ("omegaB", "clim"))
        K = torch.stack([M[t] for t in itertools.product(range(3), repeat=3)]).reshape((3, 3, 3) + self.shape)
        for ax in range(3):
            m0, m1, m2 = K.movedim(ax, 0)
            v = vel[ax]
            K = torch.stack([m0, m1 - v * m0, m2 - 2 * v * m1 + v * v * m0]).movedim(0, ax)
        inv = 1 / rho

        def products(A):
            """rho times the difference between the fourth-order central moments and cumulants."""
            two = (A[2, 0, 0], A[0, 2, 0], A[0, 0, 2])
            n = {}
            for a, b, c in ((0, 1, 2), (1, 0, 2), (2, 0, 1)):
                key = lambda i, j, k: tuple({a: i, b: j, c: k}[x] for x in range(3))  # noqa: E731
                n[key(2, 1, 1)] = two[a] * A[key(0, 1, 1)] + 2 * A[key(1, 1, 0)] * A[key(1, 0, 1)]
                n[key(0, 2, 2)] = two[b] * two[c] + 2 * A[key(0, 1, 1)] ** 2
            return n, two

        n, two = products(K)
        C = {t: K[t] for t in itertools.product(range(3), repeat=3)}
        for t, v in n.items():
            C[t] = K[t] - v * inv
        # relaxation rates
        o3 = 8 * (o1 - 2) * (o2 * (3 * o1 - 1) - 5 * o1) / (8 * (5 - 2 * o1) * o1 + o2 * (8 + o1 * (9 * o1 - 26)))
        o4 = 8 * (o1 - 2) * (o1 + o2 * (3 * o1 - 7)) / (o2 * (56 - 42 * o1 + 9 * o1 * o1) - 8 * o1)
        o5 = (24 * (o1 - 2) * (4 * o1 * o1 + o1 * o2 * (18 - 13 * o1) + o2 * o2 * (2 + o1 * (6 * o1 - 11)))
              / (16 * o1 * o1 * (o1 - 6) - 2 * o1 * o2 * (216 + 5 * o1 * (9 * o1 - 46))
                 + o2 * o2 * (o1 * (3 * o1 - 10) * (15 * o1 - 28) - 48)))

        def lim(om, c):
            a = c.abs()
            return torch.where(a > 0, om + (1 - om) * a / (a + clim * rho), torch.ones_like(om))

        den = (o1 - o2) * (o2 * (2 + 3 * o1) - 8 * o1)
        A = ((4 * o1 * o1 + 2 * o1 * o2 * (o1 - 6) + o2 * o2 * (o1 * (10 - 3 * o1) - 4)) / den).clamp(min=0)
        B = ((4 * o1 * o2 * (9 * o1 - 16) - 4 * o1 * o1 - 2 * o2 * o2 * (2 + 9 * o1 * (o1 - 2))) / den / 3).clamp(min=0)
        u, v, w = vel
        a, b, c = two
        S = {(0, 0, 0): rho, (1, 0, 0): -C[1, 0, 0], (0, 1, 0): -C[0, 1, 0], (0, 0, 1): -C[0, 0, 1]}
        for t in ((1, 1, 0), (1, 0, 1), (0, 1, 1)):
            S[t] = (1 - o1) * C[t]
        Dx = -0.5 * inv * (o1 * (2 * a - b - c) + o2 * (a + b + c - rho))
        Dy, Dz = Dx + 1.5 * o1 * inv * (a - b), Dx + 1.5 * o1 * inv * (a - c)
        X1 = (1 - o1) * (a - b) - 3 * rho * (1 - o1 / 2) * (u * u * Dx - v * v * Dy)
        X2 = (1 - o1) * (a - c) - 3 * rho * (1 - o1 / 2) * (u * u * Dx - w * w * Dz)
        X3 = rho * o2 + (1 - o2) * (a + b + c) - 3 * rho * (1 - o2 / 2) * (u * u * Dx + v * v * Dy + w * w * Dz)
        S[2, 0, 0] = (X1 + X2 + X3) / 3
        S[0, 2, 0], S[0, 0, 2] = S[2, 0, 0] - X1, S[2, 0, 0] - X2
        for p, q in (((1, 2, 0), (1, 0, 2)), ((2, 1, 0), (0, 1, 2)), ((2, 0, 1), (0, 2, 1))):
            X1 = (1 - lim(o3, C[p] + C[q])) * (C[p] + C[q])
            X2 = (1 - lim(o4, C[p] - C[q])) * (C[p] - C[q])
            S[p], S[q] = 0.5 * (X1 + X2), 0.5 * (X1 - X2)
        S[1, 1, 1] = (1 - lim(o5, C[1, 1, 1])) * C[1, 1, 1]
        vis = 1 / o1 - 0.5
        vA, vB = 2 * vis * A * rho / 3, -vis * B * rho / 3
        X1, X2, X3 = vA * (Dx - 2 * Dy + Dz), vA * (Dx + Dy - 2 * Dz), -2 * vA * (Dx + Dy + Dz)
        S[2, 2, 0], S[2, 0, 2], S[0, 2, 2] = (X1 + X2 + X3) / 3, (X3 - X1) / 3, (X3 - X2) / 3
        S[2, 1, 1] = vB * -3 * o1 * C[0, 1, 1] * inv
        S[1, 2, 1] = vB * -3 * o1 * C[1, 0, 1] * inv
        S[1, 1, 2] = vB * -3 * o1 * C[1, 1, 0] * inv
        n, two = products(S)
        for t, x in n.items():
            S[t] = S[t] + x * inv
        a, b, c = two
        # fifth and sixth order relax to zero: only the products remain (with the reference's own
        # choice of the fourth-order moment in the first product of each fifth-order one)
        S[1, 2, 2] = (S[0, 2, 2] * S[1, 2, 0] + b * S[1, 0, 2] + 4 * S[0, 1, 1] * S[1, 1, 1]
                      + 2 * (S[1, 0, 1] * S[0, 2, 1] + S[1, 1, 0] * S[0, 1, 2])) * inv
        S[2, 1, 2] = (S[2, 0, 2] * S[0, 1, 2] + c * S[2, 1, 0] + 4 * S[1, 0, 1] * S[1, 1, 1]
                      + 2 * (S[1, 1, 0] * S[1, 0, 2] + S[0, 1, 1] * S[2, 0, 1])) * inv
        S[2, 2, 1] = (S[2, 2, 0] * S[2, 0, 1] + a * S[0, 2, 1] + 4 * S[1, 1, 0] * S[1, 1, 1]
                      + 2 * (S[0, 1, 1] * S[2, 1, 0] + S[1, 0, 1] * S[1, 2, 0])) * inv
        S[2, 2, 2] = ((4 * S[1, 1, 1] ** 2 + a * S[0, 2, 2] + b * S[2, 0, 2] + c * S[2, 2, 0]
                       + 4 * (S[0, 1, 1] * S[2, 1, 1] + S[1, 0, 1] * S[1, 2, 1] + S[1, 1, 0] * S[1, 1, 2])
                       + 2 * (S[1, 2, 0] * S[1, 0, 2] + S[2, 1, 0] * S[0, 1, 2] + S[2, 0, 1] * S[0, 2, 1])) * inv
                      - (16 * S[1, 1, 0] * S[1, 0, 1] * S[0, 1, 1]
                         + 4 * (S[1, 0, 1] ** 2 * b + S[0, 1, 1] ** 2 * a + S[1, 1, 0] ** 2 * c)
                         + 2 * a * b * c) * inv * inv)
        K = torch.stack([S[t] for t in itertools.product(range(3), repeat=3)]).reshape((3, 3, 3) + self.shape)
        for ax in range(3):
            k0, k1, k2 = K.movedim(ax, 0)
            v = vel[ax]
            K = torch.stack([k0, k1 + v * k0, k2 + 2 * v * k1 + v * v * k0]).movedim(0, ax)
        return self.back @ K.reshape(27, -1)

    def sums(self):
        """The eight sums of lbffs_reduce: wall force, marker forcing, density excess, fluid cells."""
        fluid = ~self.solid.reshape(-1)
        G = self.G if self.xyz is not None else [torch.zeros(1, dtype=torch.float64, device=self.dev)] * 3
        rest = [((self.f.sum(0) - 1) * fluid).sum(), fluid.sum().double()]
        return torch.stack([g.sum() for g in self.force] + [g.sum() for g in G] + rest)

    def markers(self, xyz, motion):
        self.xyz, self.motion = self.put(xyz), motion

    def frame(self, x):
        """Axis foot, radial and tangential unit vectors and radius (with the reference's axis dot product)."""
        e0 = self.put(np.float32(self.motion["axis"]))
        OX = x - self.put(np.float32(self.motion["center"]))
        foot = (OX[:, 0] * e0[0] + OX[:, 1] * e0[1] + OX[:, 0] * e0[2])[:, None] * e0
        r = torch.linalg.norm(OX - foot, dim=1, keepdim=True)
        e1 = (OX - foot) / r
        return foot, e1, torch.linalg.cross(e0.expand_as(e1), e1), r

    def turn(self):
        """After a step: marker forcing from the trilinear velocity, its spread, the markers' motion, the force."""
        trans = self.put(np.float32(self.motion["trans"]))
        om = float(np.float32(self.motion["omega"]))
        _, _, e2, r = self.frame(self.xyz)
        wall = trans + r * om * e2
        base = self.xyz.long()
        n = torch.tensor(self.n, device=self.dev)
        box = []
        for d in itertools.product((0, 1), repeat=3):
            b = base + torch.tensor(d, device=self.dev)
            ok = ((base >= 0) & (base < n) & (b < n)).all(1)
            weight = torch.prod(1 - (b - self.xyz).abs(), dim=1) * ok
            b = torch.minimum(b.clamp(min=0), n - 1)
            box.append((b[:, 0] + n[0] * (b[:, 1] + n[1] * b[:, 2]), weight))
        flat = [v.reshape(-1) for v in self.vel]
        there = torch.stack([sum(v[ic] * wt for ic, wt in box) for v in flat], dim=1)
        self.forcing = wall - there
        self.G = [torch.zeros_like(flat[0]) for _ in range(3)]
        for a in range(3):
            for ic, wt in box:
                self.G[a].index_add_(0, ic, self.forcing[:, a] * wt)
        x = self.xyz + trans
        foot, e1, e2, r = self.frame(x)
        self.xyz = self.put(np.float32(self.motion["center"])) + foot + r * (math.cos(om) * e1 + math.sin(om) * e2)
        rho = 3 * self.rho.reshape(-1) * ~self.solid.reshape(-1)
        for q, d in enumerate(self.dirs):
            self.f[q] += rho * self.w[q] * sum(g * s for g, s in zip(self.G, d))
