"""Performance cases: what a program that simulates soft bodies with this package has it do.

A pass of a "frame" case is what a simulation loop does per output frame: `steps` implicit Euler
steps of every scene (replayed from a captured graph, as the serving loop and bench.py run them),
then positions and velocities read back.  A pass of the "plugin" case is one implicit Euler step
driven from outside through the component calls (addForce, addMDx, addDForce, projectResponse,
CGLinearSolver::solve) on the caller's device vectors, the way a SOFA solver drives a force field.

The bodies: clamped beams on regular grids cut into 5 or 6 tetrahedra per cube, their far face
driven by an oscillator (cubic cells, as the jobs of the served stream; SofaCUDA's two benchmark beams
hang free, one on a plane), mixes of such jobs of log-uniform size stepped together, and ellipsoids of jittered
cubes with one material per element and a consistent mass.  Materials, the starting deflection and
velocity, the drive and the jitter come from the seed.  The solver tolerances are below what the
iteration budgets reach, so every solve runs its budget.

The engines that compute elements in single precision (FP32, SPLIT, MIXED) are read back into
float32 arrays, the precision their callers keep; the FP64 engines into float64.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from sofa_amd import capi

GRAVITY = (0.0, -9.81, 0.0)
RAYLEIGH = 0.1          # stiffness and mass factors of every benchmark scene
SINGLE = ("fp32", "split", "mixed")


def listed():
    def frame(name, engine, body, **kw):
        return dict(dict(name=name, kind="frame", engine=engine, body=body, split=5, scenes=1, plane=False,
                         drive=True, iters=25, steps=1, stress=False), **kw)

    def beam(name, engine, nx, ny, nz, **kw):
        return frame(name, engine, "beam", nx=nx, ny=ny, nz=nz, **kw)

    return [
        # the 5x5x21 beam of the accuracy tests, parity engine: an interactive scene, one step a frame
        beam("beam_5_fp64", "fp64", 5, 5, 21),
        # SofaCUDA's benchmark beam10x10x40 (18,954 tets, CG 20), single precision as published
        beam("beam_10_fp32", "fp32", 10, 10, 40, split=6, iters=20, steps=2, drive=False),
        # SofaCUDA's benchmark beam16x16x76 (101,250 tets, CG 10) falling onto its plane
        beam("beam_16_plane_fp32", "fp32", 16, 16, 76, split=6, iters=10, steps=2, plane=True, drive=False),
        # the 1.31M-tetrahedron beam (33x33x257, CG 50): one scene that fills the GPU
        beam("beam_33_fp32", "fp32", 33, 33, 257, iters=50, steps=2),
        # a quarter-million-tetrahedron beam on the parity engine, with its stress field per frame
        beam("beam_21_fp64", "fp64", 21, 21, 129, steps=4, stress=True),
        # a mix of beam jobs in the reference's summation order (the benchmark's headline path)
        frame("mix_reference", "reference", "mix", scenes=16, steps=4),
        # the same mix in single precision: throughput serving
        frame("mix_fp32", "fp32", "mix", scenes=24, steps=2),
        # ellipsoids, one material per element, consistent mass: FP32 inner CG in FP64 refinement
        frame("ellipsoid_mixed", "mixed", "ellipsoid", nodes=40000, precond=2, iters=30, sweeps=3, steps=2),
        # ... FP32 elements on FP64 vectors
        frame("ellipsoid_split", "split", "ellipsoid", nodes=25000, steps=2),
        # ... all FP64 on the tiled kernels
        frame("ellipsoid_fp64_tiled", "fp64_tiled", "ellipsoid", nodes=60000, iters=30, steps=4),
        # ... block-Jacobi PCG on the parity engine
        frame("ellipsoid_pcg_fp64", "fp64", "ellipsoid", nodes=9000, precond=2, iters=60, steps=2),
        # a step driven through the component calls on float vectors
        dict(name="plugin_fp32", kind="plugin", engine="fp32", body="beam", split=5, scenes=1, plane=False,
             drive=False, nx=13, ny=13, nz=120, iters=25, steps=1, stress=False),
    ]


# cost of an element's share of a CG iteration, relative to the FP32 engine's
_WEIGHT = {"fp32": 1.0, "split": 1.4, "mixed": 1.4, "fp64_tiled": 2.5, "reference": 4.0, "fp64": 6.0}


def _elements(case):
    """The pass's tetrahedra over all scenes (of a mix, which depends on the seed: about)."""
    if case["body"] == "beam":
        return case["split"] * (case["nx"] - 1) * (case["ny"] - 1) * (case["nz"] - 1)
    if case["body"] == "mix":
        return 35000 * case["scenes"]
    return 6 * case["nodes"]


def _iterations(case):
    return case["iters"] * case.get("sweeps", 1)


def _cost(case):
    return _WEIGHT[case["engine"]] * _elements(case) * (_iterations(case) + 4) * case["steps"]


def draw(rng):
    most = 0.9 * max(_cost(c) for c in listed())
    while True:
        engine = rng.choice(("fp32", "fp32", "fp64", "fp64_tiled", "reference", "split", "mixed"))
        body = rng.choice(("beam", "beam", "ellipsoid", "mix"))
        case = dict(kind="frame", engine=engine, body=body, split=rng.choice((5, 6)), scenes=1, plane=False, drive=True,
                    iters=rng.randint(10, 30), steps=rng.choice((1, 2) if engine in SINGLE else (1, 2, 4)), stress=False)
        if body == "beam":
            nodes = math.exp(rng.uniform(math.log(500), math.log(280000)))
            nx, ny = rng.randint(3, 33), rng.randint(3, 33)
            nz = round(nodes / (nx * ny))
            if not max(4, nx, ny) <= nz <= 600:
                continue
            case.update(nx=nx, ny=ny, nz=nz, plane=rng.random() < 0.3, drive=rng.random() < 0.7)
            if engine == "fp32" and rng.random() < 0.3:
                case.update(kind="plugin", plane=False, drive=False, steps=1)
            elif engine == "fp64":
                case["stress"] = rng.random() < 0.3
        elif body == "mix":
            if engine == "mixed":
                continue
            case["scenes"] = rng.randint(3, 20)
        else:
            if engine == "reference":      # the reference order takes lumped masses only
                continue
            case["nodes"] = round(math.exp(rng.uniform(math.log(1500), math.log(60000))))
            if engine == "fp64" and rng.random() < 0.5:
                case["precond"] = rng.choice((1, 2))
        if engine == "mixed":
            case.update(precond=rng.choice((0, 1, 2)), iters=30, sweeps=rng.randint(1, 3))
        if _cost(case) <= most:
            return case


# ---- the bodies (plain numpy: exact() builds the same ones) ---------------------------------

_CORNERS = ((0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1))
_SPLIT = {5: ((0, 1, 3, 4), (1, 2, 3, 6), (1, 4, 5, 6), (3, 4, 6, 7), (1, 3, 4, 6)),
          6: ((0, 5, 1, 6), (0, 1, 3, 6), (1, 3, 6, 2), (6, 3, 0, 7), (6, 7, 0, 5), (7, 5, 4, 0))}


def _grid(n, lo, hi):
    """Points (x fastest) and cubes of a regular grid."""
    axes = [np.linspace(lo[k], hi[k], n[k]) for k in range(3)]
    z, y, x = np.meshgrid(axes[2], axes[1], axes[0], indexing="ij")
    points = np.stack([x.ravel(), y.ravel(), z.ravel()], 1)
    k, j, i = np.meshgrid(*[np.arange(m - 1) for m in (n[2], n[1], n[0])], indexing="ij")
    cubes = np.stack([(i + a) + n[0] * ((j + b) + n[1] * (k + c)) for a, b, c in _CORNERS], -1).reshape(-1, 8)
    return points, cubes


def _tets(cubes, split):
    return np.ascontiguousarray(cubes[:, np.array(_SPLIT[split])].reshape(-1, 4).astype(np.int32))


def _beam(case, rng, n, width, young, poisson):
    """A beam of cubic cells along z, its larger section side `width`, 1000 kg per cubic metre."""
    length = np.array([m - 1 for m in n]) * (width / (max(n[:2]) - 1))
    x0, cubes = _grid(n, (0, 0, 0), length)
    s = x0[:, 2] / length[2]
    bump = (6.75 * s * s * (1 - s) if case["drive"] else s * s)[:, None]
    amp = 0.01 * length[2] * rng.uniform(0.5, 1.5)
    turn = rng.uniform(0, 2 * math.pi)
    way = np.array([math.cos(turn), math.sin(turn), 0.0])
    body = dict(x0=x0, tets=_tets(cubes, case["split"]), young=young, poisson=poisson,
                fixed=np.nonzero(x0[:, 2] == 0)[0], driven=np.zeros(0, np.int64), x=x0 + amp * bump * way,
                v=rng.uniform(1, 3) * bump * way[[1, 0, 2]] + rng.normal(0, 1e-3, x0.shape), plane=None, dt=0.01,
                mass="uniform", mass_value=1000.0 * length.prod() / len(x0))
    if case["drive"]:
        body.update(driven=np.nonzero(x0[:, 2] == x0[:, 2].max())[0], amplitude=rng.uniform(0.002, 0.01),
                    frequency=rng.uniform(0.5, 5.0))
    for fixed in (body["fixed"], body["driven"]):
        body["x"][fixed], body["v"][fixed] = x0[fixed], 0.0
    return body


def _bodies(case, seed):
    rng = np.random.default_rng(seed)
    if case["body"] == "beam" and case["split"] == 6 and not case["drive"]:
        # SofaCUDA's scenes: 4 m section, total mass 50 spread by volume
        b = _beam(case, rng, (case["nx"], case["ny"], case["nz"]), 4.0, rng.uniform(1000, 2000), 0.3)
        b.update(mass="diagonal_total", mass_value=50.0, plane=(0.05, 1e4) if case["plane"] else None,
                 dt=0.04 if case["plane"] else 0.01)
        return [b]
    if case["body"] == "beam":
        b = _beam(case, rng, (case["nx"], case["ny"], case["nz"]), 1.0, 10 ** rng.uniform(5, 6), rng.uniform(0.3, 0.49))
        b.update(plane=(0.05, 1e4) if case["plane"] else None)
        return [b]
    if case["body"] == "mix":
        out = []
        sizes = np.random.default_rng(case["scenes"])     # the mix's sizes go with its scene count
        for _ in range(case["scenes"]):
            nodes = 10 ** sizes.uniform(math.log10(500), math.log10(50000))
            nxy = max(3, round((nodes / 4) ** (1 / 3)))
            out.append(_beam(case, rng, (nxy, nxy, max(4, round(nodes / nxy ** 2))), 1.0, 10 ** rng.uniform(5, 6),
                             rng.uniform(0.3, 0.49)))
        return out
    # an ellipsoid (0.15 x 0.10 x 0.08 m semi-axes) of jittered cubes, materials per element
    axes = np.array([0.15, 0.10, 0.08])
    h = (4 / 3 * math.pi * axes.prod() / case["nodes"]) ** (1 / 3)
    x0, cubes = _grid([2 * math.ceil(a / h) + 1 for a in axes], -axes, axes)
    cubes = cubes[((x0[cubes].mean(1) / axes) ** 2).sum(1) <= 1]
    used = np.unique(cubes)
    index = np.full(len(x0), -1)
    index[used] = np.arange(len(used))
    x0, tets = x0[used], _tets(index[cubes], 6)
    x0 = x0 + rng.uniform(-0.12 * h, 0.12 * h, x0.shape)
    bump = np.clip(1 - (x0[:, :1] / 0.13) ** 2, 0, None)
    fixed, driven = np.nonzero(x0[:, 0] < -0.13)[0], np.nonzero(x0[:, 0] > 0.13)[0]
    x = x0 + bump * rng.uniform(-0.01, 0.01, 3)
    v = bump * rng.uniform(-0.1, 0.1, 3) + rng.normal(0, 1e-4, x0.shape)
    for f in (fixed, driven):
        x[f], v[f] = x0[f], 0.0
    return [dict(x0=x0, tets=tets, young=10 ** rng.uniform(3, 5, len(tets)), poisson=rng.uniform(0.40, 0.49, len(tets)),
                 fixed=fixed, driven=driven, amplitude=0.005, frequency=1.0, x=x, v=v, plane=None, dt=0.01,
                 mass="consistent", mass_value=1050.0)]


# ---- the framework --------------------------------------------------------------------------

_ENGINE = {"fp64": capi.FP64, "fp32": capi.FP32, "mixed": capi.MIXED, "fp64_tiled": capi.FP64_TILED,
           "reference": capi.FP64_TILED, "split": capi.SPLIT}
_MASS = {"uniform": capi.MASS_UNIFORM, "diagonal_total": capi.MASS_DIAGONAL_TOTAL, "consistent": capi.MASS_MESHMATRIX}


def _tolerance(case):
    return 1e-18 if case.get("precond") else 1e-9     # PCG's is on r.z over b.b


def prepare(case, seed):
    eng = capi.Engine(0, _ENGINE[case["engine"]])
    if case["engine"] == "reference":
        eng.set_dot_order(True)
    bodies = _bodies(case, seed)
    for b in bodies:
        drive = None
        if len(b["driven"]):
            amp = np.zeros((len(b["driven"]), 3))
            amp[:, 0] = b["amplitude"]
            drive = dict(index=b["driven"], mean=b["x0"][b["driven"]], amplitude=amp,
                         pulsation=np.full(len(amp), 2 * math.pi * b["frequency"]), phase=np.zeros(len(amp)))
        s = eng.add_scene(b["x0"], b["tets"], b["young"], b["poisson"], b["fixed"], mass_kind=_MASS[b["mass"]],
                          mass_value=b["mass_value"], gravity=GRAVITY, dt=b["dt"], rayleigh_stiffness=RAYLEIGH,
                          rayleigh_mass=RAYLEIGH, cg_iterations=case["iters"], cg_tolerance=_tolerance(case),
                          cg_threshold=1e-30, oscillators=drive)
        if b["plane"]:
            eng.add_plane(s, d=b["plane"][0], stiffness=b["plane"][1])
        if case.get("precond"):
            eng.set_preconditioner(s, case["precond"])
        if case["engine"] == "mixed":
            eng.set_refinement(s, inner_iterations=case["iters"], inner_tolerance=0.0, max_sweeps=case["sweeps"])
    eng.commit()
    eng.set_graphs(True)
    state = dict(case=case, eng=eng, scenes=list(range(len(bodies))))
    if case["kind"] == "plugin":
        b, dev = bodies[0], dict(dtype=torch.float32, device="cuda")
        state.update(dt=b["dt"], x=torch.tensor(b["x"], **dev), v=torch.tensor(b["v"], **dev),
                     stream=torch.cuda.Stream())
        torch.cuda.synchronize()
    else:
        for s, b in enumerate(bodies):
            eng.write(s, b["x"], b["v"])
    return state


def run(state):
    case, eng = state["case"], state["eng"]
    if case["kind"] == "plugin":
        return _plugin_step(state)
    eng.step(state["scenes"], case["steps"])
    out = dict(x=[], v=[])
    single = case["engine"] in SINGLE
    for s in state["scenes"]:
        x, v, _ = eng.read(s)
        out["x"].append(x.astype(np.float32) if single else x)
        out["v"].append(v.astype(np.float32) if single else v)
    if case["stress"]:
        out["stress"], out["stress_nodes"] = eng.von_mises(0, 2)
    return out


def _plugin_step(state):
    """EulerImplicitSolver::solve on the caller's vectors, one component call per operation."""
    eng, x, v, h = state["eng"], state["x"], state["v"], state["dt"]
    with torch.cuda.stream(state["stream"]):
        s = state["stream"].cuda_stream
        f = torch.zeros_like(x)
        eng.mass_add_force(0, f.data_ptr(), s)
        eng.fem_add_force(0, x.data_ptr(), f.data_ptr(), s)
        b = f.clone()
        eng.mass_add_mdx(0, v.data_ptr(), b.data_ptr(), -RAYLEIGH, s)
        eng.fem_add_dforce(0, v.data_ptr(), b.data_ptr(), h + RAYLEIGH, s)
        b *= h
        eng.project_response(0, b.data_ptr(), s)
        dv = torch.empty_like(x)
        eng.cg_solve(0, 1 + h * RAYLEIGH, 0.0, -h * (h + RAYLEIGH), b.data_ptr(), dv.data_ptr(), s)
        new_v = v + dv
        new_x = x + h * new_v
    return dict(f=f, v=new_v, x=new_x)


def work(case):
    """An iteration reads the connectivity (16 B an element) and passes over 6 node vectors (r, p, q, x);
    an element's product with its stiffness takes about 160 operations, 2 of each vector entry."""
    e, n = _elements(case), _nodes(case)
    size = 4 if case["engine"] in ("fp32", "mixed") else 8
    passes = case["steps"] * (_iterations(case) + 2)
    return dict(bytes=passes * (16 * e + 18 * size * n), flops=passes * (160 * e + 30 * n))


def _nodes(case):
    if case["body"] == "beam":
        return case["nx"] * case["ny"] * case["nz"]
    return 10700 * case["scenes"] if case["body"] == "mix" else case["nodes"]


# ---- the same step in 64 bits ---------------------------------------------------------------

class _Body64:
    """Corotational linear tetrahedra ("large": the frame of edges ab and ac) with implicit Euler, in
    plain float64 torch operations."""

    def __init__(self, case, b):
        def t(a, dtype=torch.float64):
            return torch.as_tensor(np.ascontiguousarray(a)).to(device="cuda", dtype=dtype)
        self.case, self.b, self.h = case, b, b["dt"]
        self.tets = t(b["tets"], torch.int64)
        self.x0, self.x, self.v = t(b["x0"]), t(b["x"]), t(b["v"])
        self.n = len(self.x0)
        e = len(self.tets)
        young, nu = (t(np.broadcast_to(b[k], e)) for k in ("young", "poisson"))
        self.lam, self.mu = young * nu / ((1 + nu) * (1 - 2 * nu)), young / (2 * (1 + nu))
        p = self.x0[self.tets]
        edges = p[:, 1:] - p[:, :1]
        self.vol = torch.linalg.det(edges).abs() / 6
        self.grad = torch.linalg.inv(edges).transpose(1, 2)           # row i: the gradient of vertex i + 1
        self.frame0 = self.frame(self.x0)
        self.rest_edges = torch.matmul(edges, self.frame0.transpose(1, 2))
        ones = torch.ones(e, 4, dtype=torch.float64, device="cuda")
        if b["mass"] == "uniform":
            self.m = torch.full((self.n,), b["mass_value"], dtype=torch.float64, device="cuda")
        elif b["mass"] == "diagonal_total":
            m = self.gather(ones[:, :, None] * (self.vol / 4)[:, None, None])[:, 0]
            self.m = m * (b["mass_value"] / m.sum())
        else:
            self.m = self.gather(ones[:, :, None] * (b["mass_value"] * self.vol / 4)[:, None, None])[:, 0]
        self.held = torch.zeros(self.n, dtype=torch.bool, device="cuda")
        self.held[t(b["fixed"], torch.int64)] = True
        self.driven = t(b["driven"], torch.int64)
        self.held[self.driven] = True
        self.dv, self.time, self.first = torch.zeros_like(self.x), 0.0, True

    def gather(self, c):
        """(E, 4, k) vertex values summed into (n, k)."""
        out = torch.zeros(self.n, c.shape[2], dtype=torch.float64, device="cuda")
        return out.index_add_(0, self.tets.reshape(-1), c.reshape(-1, c.shape[2]))

    def frame(self, x):
        p = x[self.tets]
        ex = p[:, 1] - p[:, 0]
        ex = ex / ex.norm(dim=1, keepdim=True)
        ez = torch.linalg.cross(ex, p[:, 2] - p[:, 0])
        ez = ez / ez.norm(dim=1, keepdim=True)
        return torch.stack([ex, torch.linalg.cross(ez, ex), ez], 1)   # rows

    def stress_forces(self, g, strain):
        """Vertex forces of the strains (E, 3, 3), both in the same frame as the gradients g (E, 3, 3)."""
        eye = torch.eye(3, dtype=torch.float64, device="cuda")
        sigma = 2 * self.mu[:, None, None] * strain + (self.lam * strain.diagonal(dim1=1, dim2=2).sum(1))[:, None, None] * eye
        f = torch.matmul(g, sigma) * self.vol[:, None, None]
        return torch.cat([-f.sum(1, keepdim=True), f], 1)

    @staticmethod
    def sym(g, u):
        """The symmetric part of sum_i u_i g_i^T."""
        a = torch.matmul(u.transpose(1, 2), g)
        return (a + a.transpose(1, 2)) / 2

    def force(self):
        """Elastic force and weight; keeps the gradients turned with the elements."""
        now = self.frame(self.x)
        p = self.x[self.tets]
        edges = torch.matmul(p[:, 1:] - p[:, :1], now.transpose(1, 2))
        local = torch.matmul(self.grad, self.frame0.transpose(1, 2))
        f = self.stress_forces(local, self.sym(local, edges - self.rest_edges))
        self.turned = torch.matmul(local, now)
        out = -self.gather(torch.matmul(f, now))
        out += self.m[:, None] * torch.tensor(GRAVITY, dtype=torch.float64, device="cuda")
        self.touch = torch.zeros_like(self.held)
        if self.b["plane"]:
            d, k = self.b["plane"]
            dist = self.x[:, 1] - d
            self.touch = dist < 0
            push = torch.zeros_like(out)
            push[:, 1] = -k * dist
            out += torch.where(self.touch[:, None], push + self.v * (5.0 * dist)[:, None], torch.zeros_like(out))
        return out

    def k_mul(self, u):
        p = u[self.tets]
        return self.gather(self.stress_forces(self.turned, self.sym(self.turned, p[:, 1:] - p[:, :1])))

    def m_mul(self, u):
        if self.b["mass"] != "consistent":
            return self.m[:, None] * u
        p = u[self.tets]
        return self.gather((p + p.sum(1, keepdim=True)) * (self.b["mass_value"] * self.vol / 20)[:, None, None])

    def plane_mul(self, u):
        out = torch.zeros_like(u)
        if self.b["plane"]:
            out[:, 1] = torch.where(self.touch, self.b["plane"][1] * u[:, 1], torch.zeros_like(u[:, 1]))
        return out

    def project(self, u):
        u[self.held] = 0.0
        return u

    def a_mul(self, u):
        h = self.h
        return self.project((1 + h * RAYLEIGH) * self.m_mul(u) + h * (h + RAYLEIGH) * (self.k_mul(u) + self.plane_mul(u)))

    def preconditioner(self):
        """The inverse of A's diagonal (kind 1) or of its 3x3 diagonal blocks (kind 2)."""
        kind, h = self.case.get("precond", 0), self.h
        if not kind:
            return lambda r: r
        g = torch.cat([-self.turned.sum(1, keepdim=True), self.turned], 1)
        mu, lam = (a[:, None, None, None] for a in (self.mu, self.lam))
        outer = g[:, :, :, None] * g[:, :, None, :]
        eye = torch.eye(3, dtype=torch.float64, device="cuda")
        blocks = ((lam + mu) * outer + mu * (g * g).sum(2)[:, :, None, None] * eye) * self.vol[:, None, None, None]
        blocks = h * (h + RAYLEIGH) * self.gather(blocks.reshape(len(g), 4, 9)).reshape(-1, 3, 3)
        m = self.m if self.b["mass"] != "consistent" else self.m * 0.4     # the consistent mass's diagonal: V/10 of V/4
        blocks = blocks + ((1 + h * RAYLEIGH) * m)[:, None, None] * eye
        blocks[self.held] = eye
        if kind == 1:
            d = blocks.diagonal(dim1=1, dim2=2)
            return lambda r: r / d
        inv = torch.linalg.inv(blocks)
        return lambda r: torch.matmul(inv, r[:, :, None])[:, :, 0]

    def cg(self, b, x, r, iters, pre, tol2):
        """`iters` (preconditioned) CG iterations from x with residual r; stops at r.z <= tol2."""
        z = pre(r)
        rho, p = (r * z).sum(), z
        for _ in range(iters):
            if not float(rho) > tol2:
                break
            q = self.a_mul(p)
            alpha = rho / (p * q).sum()
            x, r = x + alpha * p, r - alpha * q
            z = pre(r)
            old, rho = rho, (r * z).sum()
            p = z + (rho / old) * p
        return x

    def right_side(self):
        f = self.force()
        b = f - RAYLEIGH * self.m_mul(self.v) - (self.h + RAYLEIGH) * (self.k_mul(self.v) + self.plane_mul(self.v))
        return f, self.project(b * self.h)

    def solve(self, b):
        case, bb = self.case, float((b * b).sum())
        pre, tol = self.preconditioner(), _tolerance(case)
        if case["engine"] == "mixed":
            x = torch.zeros_like(b)
            for _ in range(case["sweeps"]):
                r = b - self.a_mul(x)
                x = x + self.cg(b, torch.zeros_like(b), r, case["iters"], pre, 0.0)
            return x
        if case.get("precond"):
            self.dv = self.cg(b, self.dv, b - self.a_mul(self.dv), case["iters"], pre, tol * bb)
            return self.dv
        return self.cg(b, torch.zeros_like(b), b, case["iters"], pre, tol * tol * bb)

    def step(self):
        dv = self.solve(self.right_side()[1])
        self.v = self.v + dv
        self.x = self.x + self.h * self.v
        if len(self.driven):
            w, a = 2 * math.pi * self.b["frequency"], self.b["amplitude"]
            self.x[self.driven] = self.x0[self.driven]
            self.x[self.driven, 0] += a * math.sin(w * self.time)
            self.v[self.driven] = 0.0
            self.v[self.driven, 0] = a * w * math.cos(w * self.time)
        self.time += self.h

    def stress(self):
        """Von Mises stress of the Green strain per element, and its mean around each node."""
        p, p0 = self.x[self.tets], self.x0[self.tets]
        u = (p - p0)[:, 1:] - (p - p0)[:, :1]
        a = torch.matmul(u.transpose(1, 2), self.grad)
        s = (a + a.transpose(1, 2) + torch.matmul(a.transpose(1, 2), a)) / 2
        s = 2 * self.mu[:, None, None] * s + (self.lam * s.diagonal(dim1=1, dim2=2).sum(1))[:, None, None] * torch.eye(
            3, dtype=torch.float64, device="cuda")
        dev = s - s.diagonal(dim1=1, dim2=2).mean(1)[:, None, None] * torch.eye(3, dtype=torch.float64, device="cuda")
        vm = torch.sqrt(1.5 * (dev * dev).sum((1, 2)))
        one = torch.ones(len(vm), 4, 1, dtype=torch.float64, device="cuda")
        around = self.gather(one * vm[:, None, None]) / self.gather(one).clamp(min=1)
        return vm, around[:, 0]


def exact(case, seed):
    bodies = _bodies(case, seed)
    if case["kind"] == "plugin":
        s = _Body64(case, {**bodies[0], **{k: bodies[0][k].astype(np.float32).astype(np.float64) for k in "xv"}})
        f, b = s.right_side()
        v = s.v + s.solve(b)
        return dict(f=f, v=v, x=s.x + s.h * v)
    out = dict(x=[], v=[])
    for b in bodies:
        s = _Body64(case, b)
        for _ in range(case["steps"]):
            s.step()
        out["x"].append(s.x.cpu().numpy())
        out["v"].append(s.v.cpu().numpy())
    if case["stress"]:
        out["stress"], out["stress_nodes"] = (a.cpu().numpy() for a in s.stress())
    return out
