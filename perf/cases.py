"""The workloads by which this library's speed is judged.

Every case goes through the entry points that a program calls (the drivers in
sgipc.system, sgipc.batch, sgipc.hybrid and sgipc.sim, and the C ABI below
them) on seeded synthetic scenes.  Kinds:

  newton       one Newton iteration on a fixed iterate: gradient and Hessian
               assembly, convert, MAS build and MAS-PCG.  `cube`: a pinned
               cube without contacts; `two_box`: two stacked boxes in contact
  system       assembly and convert alone: the gradient and the block matrix
  precond      the MAS build on a converted matrix, and one apply
  detect       contact detection: LBVH broad phase and narrow phase
  line_search  what an accepted step costs besides the solve: energies, the
               CCD step bound and the step
  batch        one Newton iteration of independent boxes on a ground plane,
               every scene with its own PCG, in one batched solve
  hybrid       affine bodies resting on a soft slab: detection and one
               coupled Newton iteration
  rollout      a few implicit time steps and the gradient of their loss

Sizes are those of the repository's tests and benchmark (cubes of 4 and 10
cells, boxes of 40, the batch of uneven boxes, the lattice of affine cubes,
the cantilever) and odd ones between.
"""
import ctypes as C
import dataclasses
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "stiff-gipc_amd"))

from sgipc import capi, scene  # noqa: E402
from sgipc.batch import BatchedNewton  # noqa: E402
from sgipc.hybrid import HybridSystem  # noqa: E402
from sgipc.sim import GroundSim, RolloutFunction  # noqa: E402
from sgipc.system import NewtonSystem, _p  # noqa: E402

# ---- the cases ---------------------------------------------------------------


def listed():
    return [
        # the smallest call: a cube of 125 vertices, where launches and host
        # round trips count; the reference's own stop rule, FP64
        dict(name="newton_cube_4_fp64", kind="newton", scene="cube", cells=4, bank=16, precision="fp64"),
        # the no-contact FP64 workload at its documented size (1,331 vertices)
        dict(name="newton_cube_10_fp64", kind="newton", scene="cube", cells=10, bank=16, precision="fp64"),
        # an ordinary interactive scene with contacts, of odd size
        dict(name="newton_two_box_13_mixed", kind="newton", scene="two_box", cells=13, bank=16, precision="mixed"),
        # the headline workload (137,842 vertices, 640,000 tets) in both forms
        dict(name="newton_two_box_40_fp64", kind="newton", scene="two_box", cells=40, bank=16, precision="fp64"),
        dict(name="newton_two_box_40_mixed", kind="newton", scene="two_box", cells=40, bank=16, precision="mixed"),
        # assembly and convert alone, for a program with its own solver
        dict(name="system_two_box_40", kind="system", scene="two_box", cells=40),
        # the preconditioner alone, at FP32 apply precision, of odd size
        dict(name="precond_two_box_27_fp32", kind="precond", scene="two_box", cells=27, bank=16, precision="fp32"),
        # contact detection, which every Newton iteration of a simulation runs
        dict(name="detect_two_box_40", kind="detect", scene="two_box", cells=40),
        # the line search's part of an iteration, of odd size
        dict(name="line_search_two_box_27", kind="line_search", scene="two_box", cells=27),
        # many uneven scenes at once (training data, design sweeps)
        dict(name="batch_48_mixed", kind="batch", scenes=48, n_min=500, n_max=5000, precision="mixed"),
        # stiff bodies on soft ground
        dict(name="hybrid_64_bodies", kind="hybrid", lattice=4, nx=50, ny=10, nz=50),
        # forward and backward through time: the differentiable cantilever
        dict(name="rollout_cantilever_20", kind="rollout", nx=20, ny=4, nz=4, steps=2),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["newton"] * 4 + ["system", "precond", "detect", "line_search", "batch", "hybrid", "rollout"])
    sc = rng.choice(["cube", "two_box", "two_box"])
    cells = _log_int(rng, 3, 48) if sc == "cube" else _log_int(rng, 4, 38)
    if kind in ("newton", "precond"):
        bank = rng.choice([16, 16, 16, 32])
        precision = rng.choice(["fp64", "mixed"] if kind == "newton" else ["fp64", "fp32"])
        return dict(kind=kind, scene=sc, cells=min(cells, 24) if bank == 32 else cells, bank=bank, precision=precision)
    if kind == "system":
        return dict(kind=kind, scene=sc, cells=cells)
    if kind in ("detect", "line_search"):
        return dict(kind=kind, scene="two_box", cells=_log_int(rng, 4, 38))
    if kind == "batch":
        n_min = _log_int(rng, 100, 800)
        return dict(kind=kind, scenes=_log_int(rng, 2, 64), n_min=n_min, n_max=n_min + _log_int(rng, 100, 3500),
                    precision=rng.choice(["fp64", "mixed", "mixed"]))
    if kind == "hybrid":
        return dict(kind=kind, lattice=rng.randint(1, 4), nx=_log_int(rng, 12, 56), ny=rng.randint(3, 10),
                    nz=_log_int(rng, 12, 56))
    return dict(kind=kind, nx=_log_int(rng, 6, 24), ny=rng.randint(2, 4), nz=rng.randint(2, 4), steps=rng.randint(1, 3))


def work(case):
    """Inputs read once and outputs written once, in bytes; floating-point
    operations that every method has to spend (one pass over the tets)."""
    kind = case["kind"]
    if kind in ("newton", "system", "precond", "detect", "line_search"):
        m = case["cells"]
        boxes = 2 if case["scene"] == "two_box" else 1
        n, T = boxes * (m + 1) ** 3, boxes * 5 * m ** 3
        faces = boxes * 12 * m * m
    elif kind == "batch":
        scenes = _batch_base(case["scenes"], case["n_min"], case["n_max"])
        n, T, faces = sum(s.n for s in scenes), sum(s.T for s in scenes), 0
    else:
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        n, T = (nx + 1) * (ny + 1) * (nz + 1), 5 * nx * ny * nz
        faces = 4 * (nx * ny + ny * nz + nx * nz)
    K = 7.0 * n  # upper blocks of a five-tet grid, about
    tets = T * (16 + 72 + 8 + 16.0)              # indices, DmInv, volume, two moduli
    verts = n * (3 * 24 + 8 + 4.0)               # x, x_rest or x_tilde, mass, pin flag, one output vector
    if kind == "system":
        return {"bytes": tets + verts + 80 * K, "flops": 3000.0 * T}
    if kind == "precond":
        return {"bytes": 80 * K + 48 * n, "flops": 2 * 48 ** 3 * n / 16.0}
    if kind == "detect":
        return {"bytes": 24.0 * n + 12 * faces + 8 * 1.5 * faces + 16 * 12.0 * case["cells"] ** 2, "flops": 30.0 * faces}
    if kind == "line_search":
        return {"bytes": tets + 5 * 24.0 * n + 20 * faces, "flops": 200.0 * T}
    if kind == "rollout":
        return {"bytes": case["steps"] * 2 * (tets + verts), "flops": case["steps"] * 6000.0 * T}
    return {"bytes": tets + verts, "flops": 3000.0 * T + 250.0 * n}


def tolerance(case):
    kind = case["kind"]
    if kind == "detect":
        return "exact"                          # whole numbers: vertex ids, ranks and counts
    if kind == "system":
        return {"rel": 1e-12, "max": 1e-9}      # FP64 sums
    if kind == "precond":
        # FP64, or FP32 inverses and products (6e-8 from 64 bits as measured)
        return {"rel": 1e-12, "max": 1e-10} if case["precision"] == "fp64" else {"rel": 3e-7, "max": 1e-5}
    if kind == "line_search":
        return {"rel": 1e-12, "max": 1e-10}
    if kind == "rollout":
        return {"rel": 1e-9, "max": 1e-7}       # Newton to 1e-11, PCG to 1e-10, per step
    if kind == "newton" and case["scene"] == "cube" and case["precision"] == "fp64":
        return {"rel": 1e-9, "max": 1e-7}       # the same PCG iterate: equal iteration counts, FP64
    # a solve to 1e-6 of the right-hand side: two correct solvers may stop at
    # neighbouring iterates, each about 2e-5 from the solution as measured
    return {"rel": 1e-4, "max": 2e-3}


# ---- inputs --------------------------------------------------------------------


@functools.lru_cache(maxsize=4)
def _base(kind, cells, bank):
    return scene.cube_scene(cells, bank=bank) if kind == "cube" else scene.two_box_scene(cells, bank=bank)


@functools.lru_cache(maxsize=2)
def _surface(kind, cells, bank):
    return scene.surface_primitives(_base(kind, cells, bank).tets)


@functools.lru_cache(maxsize=2)
def _batch_base(n_scenes, n_min, n_max):
    return tuple(scene.batch_scenes(n_scenes, seed=5, n_min=n_min, n_max=n_max))


@functools.lru_cache(maxsize=2)
def _hybrid_base(lattice, nx, ny, nz):
    return scene.hybrid_scene((nx, ny, nz), lattice=lattice)


@functools.lru_cache(maxsize=2)
def _cantilever_base(nx, ny, nz):
    return scene.cantilever_scene(nx, ny, nz)


def _scene(case, seed):
    """The scene of a seed: its own iterate and velocities on a shared mesh."""
    bank = case.get("bank", 16)
    base = _base(case["scene"], case["cells"], bank)
    rng = np.random.default_rng(seed)
    xr, free = base.x_rest, base.btype == 0
    noise = rng.normal(0.0, 0.01 / case["cells"], size=xr.shape)
    if case["scene"] == "two_box":  # the facing faces keep their distance
        gap = base.meta["gap"]
        noise[(np.abs(xr[:, 1] - 1.0) < 1e-12) | (np.abs(xr[:, 1] - 1.0 - gap) < 1e-12), 1] = 0.0
    x = xr + noise * free[:, None]
    if case["kind"] == "system" and seed != 0:  # iterates around the one whose contact pairs are known
        noise = 0.1 * noise + _scene(case, 0).x - xr
    v = rng.uniform(-0.5, 0.5, size=xr.shape) * (1.0 if case["scene"] == "two_box" else 0.1)
    xt = x + (base.dt * v + base.dt ** 2 * np.array([0.0, -9.8, 0.0])) * free[:, None]
    return dataclasses.replace(base, x=x, x_tilde=xt)


def _batch_scenes(case, seed):
    rng = np.random.default_rng(seed)
    out = []
    for s in _batch_base(case["scenes"], case["n_min"], case["n_max"]):
        noise = rng.normal(0.0, 0.01 * 0.5 / max(s.meta["cells"]), size=s.x_rest.shape)
        noise[s.x_rest[:, 1] < 0.5 * s.meta["dhat_dist"] + 1e-12, 1] = 0.0
        x = s.x_rest + noise
        v = rng.uniform(-0.1, 0.1, size=3)
        out.append(dataclasses.replace(s, x=x, x_tilde=x + s.dt * v + s.dt ** 2 * np.array([0.0, -9.8, 0.0])))
    return out


class _Surface:
    """Surface primitives and candidate buffers of a scene on the GPU."""

    def __init__(self, case, dev, per_primitive=4):
        faces, edges, verts = _surface(case["scene"], case["cells"], case.get("bank", 16))
        i32 = dict(dtype=torch.int32, device=dev)
        self.nf, self.ne, self.nv = len(faces), len(edges), len(verts)
        self.faces = torch.tensor(faces.astype(np.int32).reshape(-1), **i32)
        self.edges = torch.tensor(edges.astype(np.int32).reshape(-1), **i32)
        self.verts = torch.tensor(verts.astype(np.int32), **i32)
        self.cap = per_primitive * (self.nv + self.ne) + 1024
        self.pt = torch.zeros(4 * self.cap, **i32)
        self.ee = torch.zeros(4 * self.cap, **i32)
        self.pairs = torch.zeros(8 * self.cap, **i32)
        self.mat_index = torch.zeros(2 * self.cap, **i32)

    def detect(self, s):
        """Broad and narrow phase at s.x: candidate and pair counts."""
        npt, nee, npair, counts = C.c_int(), C.c_int(), C.c_int(), np.zeros(3, np.int32)
        s.ctx.call("sgipc_broad_phase", self.nv, _p(self.verts), self.nf, _p(self.faces), self.ne, _p(self.edges),
                   _p(s.x), _p(s.btype), None, float(s.sc.dhat), _p(self.pt), self.cap, C.byref(npt), _p(self.ee),
                   self.cap, C.byref(nee))
        s.ctx.call("sgipc_classify_contacts", npt.value, _p(self.pt), nee.value, _p(self.ee), _p(s.x), _p(s.x_rest),
                   float(s.sc.dhat), _p(self.pairs), _p(self.mat_index), 2 * self.cap, C.byref(npair),
                   counts.ctypes.data)
        return npt.value, nee.value, npair.value, counts


def _newton_system(case, seed):
    sc = _scene(case, seed)
    pc = capi.PRECOND_MAS_FP32 if case.get("precision") in ("mixed", "fp32") else capi.PRECOND_MAS
    s = NewtonSystem(sc, "cuda:0", precond=pc)
    if case["scene"] == "two_box":
        surf = _Surface(case, s.dev)
        if case["kind"] == "system":  # the pair list of a nearby iterate: the matrix keeps its pattern
            x = s.x.clone()
            s.x.copy_(torch.tensor(_scene(case, 0).x.reshape(-1)))
        _, _, n, counts = surf.detect(s)
        if case["kind"] == "system":
            s.x.copy_(x)
        s.n_pairs, s.counts = n, counts
        s.pairs = surf.pairs[:4 * n].clone() if n else None
        s.mat_index = surf.mat_index[:n].clone() if n else None
        s.n_contact_triplets = 4 * int(counts[0]) + 9 * int(counts[1]) + 16 * int(counts[2])
        s._set_capacity(10 * s.T + s.n + s.n_contact_triplets)
    return s


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case, "kind": kind}
    if kind in ("newton", "system"):
        st["sys"] = _newton_system(case, seed)
    elif kind == "precond":
        s = st["sys"] = _newton_system(case, seed)
        s.assemble()
        s.convert()
        st["r"] = torch.tensor(np.random.default_rng(seed + 1).normal(size=3 * s.n), device=s.dev)
        st["z"] = torch.zeros_like(st["r"])
    elif kind == "detect":
        s = st["sys"] = NewtonSystem(_scene(case, seed), "cuda:0")
        st["surf"] = _Surface(case, s.dev)
    elif kind == "line_search":
        s = st["sys"] = _newton_system(case, seed)
        st["surf"] = _Surface(case, s.dev, 32)
        st["dir"] = s.x - s.x_tilde           # x - alpha dir: towards the inertial target
        st["x_new"] = torch.zeros_like(s.x)
    elif kind == "batch":
        st["sys"] = BatchedNewton(_batch_scenes(case, seed), "cuda:0",
                                  precond=capi.PRECOND_MAS_FP32 if case["precision"] == "mixed" else capi.PRECOND_MAS)
    elif kind == "hybrid":
        st["sys"] = HybridSystem(_hybrid_scene(case, seed), "cuda:0", precond=capi.PRECOND_MAS_FP32)
    else:
        sc, log_E, v0, target = _rollout_inputs(case, seed)
        st["sys"] = GroundSim(sc, "cuda:0")
        st["log_E"], st["v0"], st["target"] = (torch.tensor(a, device="cuda:0") for a in (log_E, v0, target))
    return st


def _hybrid_scene(case, seed):
    base = _hybrid_base(case["lattice"], case["nx"], case["ny"], case["nz"])
    rng = np.random.default_rng(seed)
    fem = base.fem
    free = fem.btype == 0
    x = fem.x_rest + rng.normal(0.0, 0.01 / case["nx"], size=fem.x_rest.shape) * free[:, None]
    top = fem.x_rest[:, 1] > fem.x_rest[:, 1].max() - 1e-9
    x[top, 1] = fem.x_rest[top, 1]
    g = np.array([0.0, -9.8, 0.0])
    xt = x + fem.dt ** 2 * g * free[:, None]
    qt = base.q_tilde.copy()
    qt[:, :3] += fem.dt * rng.uniform(-0.1, 0.1, size=(base.nb, 3))
    return dataclasses.replace(base, fem=dataclasses.replace(fem, x=x, x_tilde=xt), q_tilde=qt)


def _rollout_inputs(case, seed):
    sc = _cantilever_base(case["nx"], case["ny"], case["nz"])
    rng = np.random.default_rng(seed)
    log_E = rng.normal(math.log(1e5), 0.2, size=sc.T)
    v0 = rng.uniform(-0.1, 0.1, size=(sc.n, 3)) * (sc.btype == 0)[:, None]
    return sc, log_E, v0, sc.x_rest + rng.normal(0.0, 0.01, size=(sc.n, 3))


# ---- one pass --------------------------------------------------------------------


def run(st):
    kind, case, s = st["kind"], st["case"], st["sys"]
    if kind == "newton":
        if case["scene"] == "cube" and case["precision"] == "fp64":
            s.newton_step(tol=1e-4, stop_rule=capi.STOP_REF_RZ)
        else:
            s.newton_step(tol=1e-6, stop_rule=capi.STOP_TRUE_REL, max_iter=100000,
                          precision=capi.PRECISION_MIXED if case["precision"] == "mixed" else capi.PRECISION_FP64)
        return {"b": s.b, "dx": s.dx}
    if kind == "system":
        s.assemble()
        K = s.convert()
        return {"b": s.b, "rows": s.tr[:K], "cols": s.tc[:K], "vals": s.tv[:9 * K]}
    if kind == "precond":
        s.build_precond()
        s.ctx.call("sgipc_precond_apply", _p(st["r"]), _p(st["z"]))
        return {"z": st["z"]}
    if kind == "detect":
        f = st["surf"]
        npt, nee, n, counts = f.detect(s)
        return {"pt": f.pt, "ee": f.ee, "pairs": f.pairs, "mat_index": f.mat_index, "counts": counts,
                "sizes": np.array([npt, nee, n])}
    if kind == "line_search":
        return _line_search(st, s)
    if kind == "batch":
        s.newton_step(precision=capi.PRECISION_MIXED if case["precision"] == "mixed" else capi.PRECISION_FP64,
                      tol=1e-6)
        return {"b": s.sys.b, "dx": s.sys.dx}
    if kind == "hybrid":
        s.detect()
        s.newton_step(tol=1e-6)
        return {"b": s.b, "dx": s.dx}
    le, v0 = st["log_E"].clone().requires_grad_(True), st["v0"].clone().requires_grad_(True)
    xT = RolloutFunction.apply(le, v0, s, case["steps"], 5)
    ((xT - st["target"]) ** 2).sum().backward()
    return {"x": xT.detach(), "grad_log_E": le.grad, "grad_v0": v0.grad}


def _line_search(st, s):
    f, sc, d, xn = st["surf"], s.sc, st["dir"], st["x_new"]
    e0 = s.energies()
    npt, nee, alpha = C.c_int(), C.c_int(), C.c_double(1.0)
    s.ctx.call("sgipc_broad_phase_ccd", f.nv, _p(f.verts), f.nf, _p(f.faces), f.ne, _p(f.edges), _p(s.x), _p(d), 1.0,
               _p(s.btype), None, float(sc.dhat), _p(f.pt), f.cap, C.byref(npt), _p(f.ee), f.cap, C.byref(nee))
    s.ctx.call("sgipc_ccd_step_bound", npt.value, _p(f.pt), nee.value, _p(f.ee), _p(s.x), _p(d), 0.8, C.byref(alpha))
    s.ctx.call("sgipc_step_forward", s.n, _p(xn), _p(s.x), _p(d), _p(s.btype), alpha.value, 0)
    ek, ef = C.c_double(), C.c_double()
    s.ctx.call("sgipc_kinetic_energy", s.n, _p(xn), _p(s.x_tilde), _p(s.mass), C.byref(ek))
    s.ctx.call("sgipc_fem_energy", s.T, _p(xn), _p(s.tets), _p(s.DmInv), _p(s.vol), _p(s.mu), _p(s.lam), float(sc.dt),
               C.byref(ef))
    return {"energies": np.array([e0["kinetic"], e0["elastic"], e0["barrier"]]), "alpha": np.float64(alpha.value),
            "x_new": xn, "kinetic": np.float64(ek.value), "elastic": np.float64(ef.value)}


# ---- the same results in 64 bits, from their definitions ---------------------------


def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _t(a):
    return torch.tensor(np.ascontiguousarray(a), device=_dev())


class _Tets:
    """SNK1 energy, gradient and Hessian of a scene's tets (dt^2-scaled)."""

    def __init__(self, sc, mu=None, lam=None):
        self.n, self.dt = sc.n, sc.dt
        self.tets = _t(sc.tets.astype(np.int64))
        D = _t(sc.DmInv).reshape(-1, 3, 3)
        self.B = torch.cat([-D.sum(1, keepdim=True), D], 1)          # (T, 4, 3): F = x^T B
        self.vol = _t(sc.vol)
        self.mu, self.lam = (_t(sc.mu) if mu is None else mu), (_t(sc.lam) if lam is None else lam)
        self.free = _t(sc.btype == 0)

    def F(self, x):
        return torch.einsum("tai,taj->tij", x[self.tets], self.B)

    def energy(self, x):
        F = self.F(x)
        Jm = torch.linalg.det(F) - 1.0 - self.mu / self.lam
        e = 0.5 * (self.mu * ((F * F).sum((1, 2)) - 3.0) + self.lam * Jm * Jm)
        return self.dt ** 2 * (e * self.vol).sum()

    def _cof(self, F):
        return torch.stack([torch.linalg.cross(F[:, 1], F[:, 2]), torch.linalg.cross(F[:, 2], F[:, 0]),
                            torch.linalg.cross(F[:, 0], F[:, 1])], 1)

    def gradient(self, x):
        F = self.F(x)
        P = self.mu[:, None, None] * F + (self.lam * (torch.linalg.det(F) - 1.0) - self.mu)[:, None, None] * self._cof(F)
        g = torch.einsum("t,taj,tij->tai", self.dt ** 2 * self.vol, self.B, P)
        return torch.zeros((self.n, 3), dtype=g.dtype, device=g.device).index_add_(0, self.tets.reshape(-1),
                                                                                   g.reshape(-1, 3))

    def hessian(self, x, project=True):
        """(rows, cols, blocks) of all 16 vertex pairs per tet; blocks of pinned vertices are zero."""
        out, step = [], 200000
        eps = torch.zeros((3, 3, 3), dtype=torch.float64, device=x.device)
        for i, j, k in ((0, 1, 2), (1, 2, 0), (2, 0, 1)):
            eps[i, j, k], eps[i, k, j] = 1.0, -1.0
        for a in range(0, self.tets.shape[0], step):
            sl = slice(a, a + step)
            F = self.F(x)[sl]
            g = self._cof(F).reshape(-1, 9)
            k = self.lam[sl] * (torch.linalg.det(F) - 1.0) - self.mu[sl]
            H = self.lam[sl, None, None] * g[:, :, None] * g[:, None, :]
            H = H + k[:, None, None] * torch.einsum("ikm,jln,tmn->tijkl", eps, eps, F).reshape(-1, 9, 9)
            H = H + self.mu[sl, None, None] * torch.eye(9, dtype=H.dtype, device=H.device)
            if project:
                w, Q = np.linalg.eigh(H.cpu().numpy())
                H = _t((Q * np.maximum(w, 0.0)[:, None, :]) @ Q.transpose(0, 2, 1))
            H = H.reshape(-1, 3, 3, 3, 3)
            B = self.B[sl]
            H = torch.einsum("taj,tijkl->taikl", B, H)
            H = torch.einsum("taikl,tbl->tabik", H, B) * (self.dt ** 2 * self.vol[sl])[:, None, None, None, None]
            t = self.tets[sl]
            fr = self.free[t].double()
            H = H * (fr[:, :, None] * fr[:, None, :])[:, :, :, None, None]
            r = t[:, :, None].expand(-1, 4, 4)
            out.append((r.reshape(-1), r.transpose(1, 2).reshape(-1), H.reshape(-1, 3, 3)))
        return tuple(torch.cat(v) for v in zip(*out))


def _ln_terms(I):
    l = torch.log(I)
    return l, (I - 1) * (I + I * l - 1), \
        4 * I + l - 3 * I * I * l * l + 6 * I * l - 2 * I * I + I * l * l - 7 * I * I * l - 2


class _Pairs:
    """The contact barrier of a list of encoded pairs."""

    def __init__(self, sc, pairs):
        q = pairs.long()
        a, b, c, d = q.unbind(1)
        neg = a < 0
        self.groups = []  # (distance kind, vertex ids, mollifier edges as slots or None)
        f = lambda v: torch.where(v < 0, -v - 1, v)
        for kind, sel, edges in (("ee", ~neg & (d >= 0), None), ("ee", ~neg & (d < 0), (0, 1, 2, 3)),
                                 ("pp", neg & (c < 0) & (b < 0), (0, 2, 1, 3)), ("pp", neg & (c < 0) & (b >= 0), None),
                                 ("pe", neg & (c >= 0) & (d < 0) & (b < 0), (0, 3, 1, 2)),
                                 ("pe", neg & (c >= 0) & (d < 0) & (b >= 0), None),
                                 ("pt", neg & (c >= 0) & (d >= 0), None)):
            if bool(sel.any()):
                nv = 4 if edges else {"pp": 2, "pe": 3}.get(kind, 4)
                self.groups.append((kind, f(q[sel])[:, :nv], edges))
        self.sc, self.xr = sc, _t(sc.x_rest)

    def _dist2(self, kind, X):
        cr, dot = torch.linalg.cross, lambda u, v: (u * v).sum(1)
        if kind == "pp":
            return dot(X[:, 0] - X[:, 1], X[:, 0] - X[:, 1])
        if kind == "pe":
            n = cr(X[:, 1] - X[:, 0], X[:, 2] - X[:, 0])
            e = X[:, 2] - X[:, 1]
            return dot(n, n) / dot(e, e)
        if kind == "pt":
            n, w = cr(X[:, 2] - X[:, 1], X[:, 3] - X[:, 1]), X[:, 0] - X[:, 1]
        else:
            n, w = cr(X[:, 1] - X[:, 0], X[:, 3] - X[:, 2]), X[:, 2] - X[:, 0]
        return dot(w, n) ** 2 / dot(n, n)

    def parts(self, x):
        """Per group: vertex ids, energies, gradients (m, nv, 3), Hessians (m, nv, nv, 3, 3)."""
        dh, kap = float(self.sc.dhat), float(self.sc.kappa)
        for kind, v, edges in self.groups:
            X = x[v].clone().requires_grad_(True)
            s = torch.sqrt(self._dist2(kind, X) / dh)
            gs, = torch.autograd.grad(s.sum(), X, retain_graph=True)
            s = s.detach()
            I = s * s
            l, u, w = _ln_terms(I)
            E = kap * dh * dh * (I - 1) ** 2 * l * l
            if edges is None:
                g = gs * (4 * kap * dh * dh * l * u / I * s)[:, None, None]
                I0 = torch.where(I < 1e-6, torch.full_like(I, 1e-6), I)
                l0 = -4 * kap * dh * dh * _ln_terms(I0)[2] / I0
                H = torch.einsum("m,mai,mbj->mabij", l0, gs, gs)
            else:
                p, q, r, t = edges
                cc = torch.linalg.cross(X[:, q] - X[:, p], X[:, t] - X[:, r])
                I1 = (cc * cc).sum(1)
                ok = I1.detach() > 0
                cn = torch.sqrt(torch.where(ok, I1, torch.ones_like(I1)))
                gc, = torch.autograd.grad(cn.sum(), X)
                I1, cn = I1.detach(), cn.detach()
                r0, r1 = self.xr[v[:, p]] - self.xr[v[:, q]], self.xr[v[:, r]] - self.xr[v[:, t]]
                eps = 1e-3 * (r0 * r0).sum(1) * (r1 * r1).sum(1)
                E = torch.where(ok, -I1 * (I1 - 2 * eps) / eps ** 2 * E, torch.zeros_like(E))
                p1 = -4 * kap * dh * dh * l * l * (I1 - eps) * (I - 1) ** 2 / eps ** 2
                p2 = -4 * kap * dh * dh * I1 * l * (I1 - 2 * eps) * u / (I * eps ** 2)
                z = ok.double()[:, None, None]
                g = z * (gc * (cn * p1)[:, None, None] + gs * (s * p2)[:, None, None])
                M = torch.zeros((len(I), 2, 2), dtype=I.dtype, device=I.device)
                M[:, 0, 0] = -4 * kap * dh * dh * l * l * (I - 1) ** 2 * (3 * I1 - eps) / eps ** 2
                M[:, 1, 1] = 4 * kap * dh * dh * I1 * (I1 - 2 * eps) * w / (I * eps ** 2)
                M[:, 0, 1] = M[:, 1, 0] = -16 * kap * dh * dh * cn * s * l * (I1 - eps) * u / (I * eps ** 2)
                e, Q = np.linalg.eigh(M.cpu().numpy())
                M = _t((Q * np.maximum(e, 0.0)[:, None, :]) @ Q.transpose(0, 2, 1))
                G = torch.stack([gc, gs], 1) * z[:, None]
                H = torch.einsum("mcai,mcd,mdbj->mabij", G, M, G)
            yield v, E, g, H


def _coalesce(n, parts):
    """Sums (rows, cols, blocks) lists into unique blocks: sorted keys and values."""
    r, c, B = (torch.cat(v) for v in zip(*parts))
    key, inv = torch.unique(r * n + c, return_inverse=True)
    return key // n, key % n, torch.zeros((len(key), 3, 3), dtype=B.dtype, device=B.device).index_add_(0, inv, B)


def _pairs_of(case, seed):
    """The encoded contact pairs of a scene: an input of the later stages."""
    if case.get("scene") != "two_box":
        return None
    s = NewtonSystem(_scene(case, 0 if case["kind"] == "system" else seed), "cuda:0")
    f = _Surface(case, s.dev)
    n = f.detect(s)[2]
    return f.pairs[:4 * n].reshape(-1, 4).clone()


def _system(sc, pairs=None, close=None):
    """Gradient and all blocks (both triangles) of a scene's Newton system."""
    x, n = _t(sc.x), sc.n
    fem, mass = _Tets(sc), _t(sc.mass)
    g = mass[:, None] * (x - _t(sc.x_tilde)) + fem.gradient(x)
    i = torch.arange(n, device=x.device)
    parts = [fem.hessian(x), (i, i, mass[:, None, None] * torch.eye(3, dtype=x.dtype, device=x.device))]
    if pairs is not None:
        free = fem.free.double()
        for v, _, gp, H in _Pairs(sc, pairs).parts(x):
            g.index_add_(0, v.reshape(-1), gp.reshape(-1, 3))
            nv = v.shape[1]
            H = H * (free[v][:, :, None] * free[v][:, None, :])[:, :, :, None, None]
            r = v[:, :, None].expand(-1, nv, nv)
            parts.append((r.reshape(-1), r.transpose(1, 2).reshape(-1), H.reshape(-1, 3, 3)))
    if close is not None:
        gg, hh = _ground(sc, x, close)
        g[:, 1] += gg
        B = torch.zeros((n, 3, 3), dtype=x.dtype, device=x.device)
        B[:, 1, 1] = hh
        parts.append((i, i, B))
    return g * fem.free[:, None], _coalesce(n, parts)


def _ground(sc, x, close):
    """Gradient and second derivative in y of the ground barrier (plane y = 0), per vertex."""
    d = x[:, 1].clone().requires_grad_(True)
    s, dh = d * d, float(sc.dhat)
    near = close & (s.detach() <= dh)
    s = torch.where(near, s, torch.full_like(s, dh))
    e = float(sc.kappa) * (-(s - dh) ** 2 * torch.log(s / dh)) * (_t(sc.btype == 0))
    g, = torch.autograd.grad(e.sum(), d, create_graph=True)
    h, = torch.autograd.grad(g.sum(), d)
    return g.detach(), h


def _solve(n, blocks, b):
    """A x = b to round-off: dense for small systems, block-Jacobi CG with
    restarts on the true residual otherwise."""
    r, c, B = blocks
    if n <= 2500:
        A = torch.zeros((n, n, 3, 3), dtype=B.dtype, device=B.device)
        A[r, c] = B
        A = A.permute(0, 2, 1, 3).reshape(3 * n, 3 * n)
        return torch.linalg.solve(A.cpu(), b.reshape(-1).cpu()).to(b.device)
    i = torch.arange(3, device=B.device)
    rows = (3 * r[:, None, None] + i[None, :, None]).expand(-1, 3, 3).reshape(-1)
    cols = (3 * c[:, None, None] + i[None, None, :]).expand(-1, 3, 3).reshape(-1)
    A = torch.sparse_coo_tensor(torch.stack([rows, cols]), B.reshape(-1), (3 * n, 3 * n)).coalesce().to_sparse_csr()
    D = torch.linalg.inv(B[r == c])
    b = b.reshape(-1)
    x = torch.zeros_like(b)
    for _ in range(4):
        res = b - A.mv(x)
        if float(res.norm()) <= 1e-14 * float(b.norm()):
            break
        y, q = torch.zeros_like(b), res.clone()
        goal = 1e-10 * float(q.norm())
        z = torch.bmm(D, q.reshape(-1, 3, 1)).reshape(-1)
        p, rz = z.clone(), torch.dot(q, z)
        for k in range(20000):
            Ap = A.mv(p)
            al = rz / torch.dot(p, Ap)
            y += al * p
            q -= al * Ap
            if k % 50 == 49 and float(q.norm()) <= goal:
                break
            z = torch.bmm(D, q.reshape(-1, 3, 1)).reshape(-1)
            rz, old = torch.dot(q, z), rz
            p = z + (rz / old) * p
        x = x + y
    return x


def _mas(sc, pairs, blocks, r):
    """The multilevel additive Schwarz apply from its definition: nodes of a
    level are grouped by bank, connected nodes of a bank form a node of the
    next level, and every bank of every level adds its exact inverse."""
    bank, n, dev = sc.bank, sc.n, r.device
    part = _t(sc.part.astype(np.int64))
    first = torch.searchsorted(part, part)
    node = part * bank + torch.arange(n, device=dev) - first
    t = _t(sc.tets.astype(np.int64))
    e = [t[:, [i, j]] for i in range(4) for j in range(i)]
    if pairs is not None:
        for _, v, _ in _Pairs(sc, pairs).groups:
            e += [v[:, [i, j]] for i in range(v.shape[1]) for j in range(i)]
    e = torch.unique(torch.cat(e), dim=0)
    size = bank * (int(part[-1]) + 1)
    m, levels = -(-max(size, n) // bank) * bank, 2
    while m > bank:
        m, levels = -(-(m // bank) // bank) * bank, levels + 1
    z = torch.zeros((n, 3), dtype=r.dtype, device=dev)
    r = r.reshape(n, 3)
    for _ in range(min(levels, 6)):
        nb = -(-size // bank)
        I, J = node[blocks[0]], node[blocks[1]]
        same = I // bank == J // bank
        A = torch.zeros((nb * bank * bank, 3, 3), dtype=r.dtype, device=dev)
        A.index_add_(0, I[same] * bank + J[same] % bank, blocks[2][same])
        A = A.reshape(nb, bank, bank, 3, 3).permute(0, 1, 3, 2, 4).reshape(nb, 3 * bank, 3 * bank)
        dia = torch.diagonal(A, dim1=1, dim2=2)
        dia += (dia == 0).double()
        R = torch.zeros((nb * bank, 3), dtype=r.dtype, device=dev).index_add_(0, node, r)
        z += torch.linalg.solve(A, R.reshape(nb, 3 * bank, 1)).reshape(-1, 3)[node]
        label = torch.arange(size, device=dev)
        ea, eb = node[e[:, 0]], node[e[:, 1]]
        ok = (ea // bank == eb // bank) & (ea != eb)
        ea, eb = ea[ok], eb[ok]
        for _ in range(bank):
            low = torch.minimum(label[ea], label[eb])
            label.scatter_reduce_(0, ea, low, "amin")
            label.scatter_reduce_(0, eb, low, "amin")
        used, node = torch.unique(label[node], return_inverse=True)
        size = len(used)
    return z.reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("detect", "hybrid"):
        return None  # whole numbers; two coupled kinds of unknowns, over 20 seconds
    if kind == "rollout":
        return _exact_rollout(case, seed)
    if kind == "batch":
        b, dx = [], []
        for s in _batch_scenes(case, seed):
            close = torch.zeros(s.n, dtype=torch.bool, device=_dev())
            close[_t(s.meta["surf"].astype(np.int64))] = True
            g, blocks = _system(s, close=close)
            b.append(g.reshape(-1))
            dx.append(_solve(s.n, blocks, g))
        return {"b": torch.cat(b), "dx": torch.cat(dx)}
    sc, pairs = _scene(case, seed), _pairs_of(case, seed)
    if kind == "line_search":
        x = _t(sc.x)
        e = np.array([float(0.5 * (_t(sc.mass) * ((x - _t(sc.x_tilde)) ** 2).sum(1)).sum()),
                      float(_Tets(sc).energy(x)),
                      float(sum(E.sum() for _, E, _, _ in _Pairs(sc, pairs).parts(x)))])
        return {"energies": e, "alpha": None, "x_new": None, "kinetic": None, "elastic": None}
    g, blocks = _system(sc, pairs)
    if kind == "system":
        r, c, B = blocks
        up = r <= c
        return {"b": g.reshape(-1), "rows": None, "cols": None, "vals": B[up].transpose(1, 2).reshape(-1)}
    if kind == "precond":
        rhs = _t(np.random.default_rng(seed + 1).normal(size=3 * sc.n))
        return {"z": _mas(sc, pairs, blocks, rhs)}
    return {"b": g.reshape(-1), "dx": _solve(sc.n, blocks, g)}


def _exact_rollout(case, seed):
    sc, log_E, v0, target = _rollout_inputs(case, seed)
    le = _t(log_E)
    cm, cl = scene_moduli(sc.meta["nu"])
    E = torch.exp(le)
    fem = _Tets(sc, cm * E, cl * E)
    n, dt, mass, free = sc.n, sc.dt, _t(sc.mass)[:, None], fem.free[:, None].double()
    close = torch.zeros(n, dtype=torch.bool, device=_dev())
    close[_t(sc.meta["surf"].astype(np.int64))] = True
    grav = torch.tensor([0.0, sc.meta["gravity"], 0.0], dtype=torch.float64, device=_dev())
    eye = torch.eye(3, dtype=torch.float64, device=_dev())
    i = torch.arange(n, device=_dev())

    def dense(x, project):
        B = mass[:, :, None] * eye
        B = B.clone()
        B[:, 1, 1] += _ground(sc, x, close)[1]
        r, c, B = _coalesce(n, [fem.hessian(x, project), (i, i, B)])
        A = torch.zeros((n, n, 3, 3), dtype=B.dtype, device=B.device)
        A[r, c] = B
        return A.permute(0, 2, 1, 3).reshape(3 * n, 3 * n).cpu()

    def gradient(x, xt):
        g = mass * (x - xt) + fem.gradient(x)
        g[:, 1] += _ground(sc, x, close)[0]
        return g * free

    x, v = _t(sc.x_rest), _t(v0) * free
    states = []
    for _ in range(case["steps"]):
        xt = x + (dt * v + dt * dt * grav) * free
        y = x.clone()
        for _ in range(40):
            d = torch.linalg.solve(dense(y, True), gradient(y, xt).reshape(-1).cpu()).to(y.device).reshape(n, 3) * free
            al = 1.0
            while bool(((y - al * d)[close, 1] <= 0.2 * y[close, 1]).any()):
                al *= 0.5
            y = y - al * d
            if al == 1.0 and float(d.abs().max()) < 1e-13:
                break
        v = (y - x) / dt
        x = y
        states.append(x)
    gx, gv = 2.0 * (x - _t(target)) * free, torch.zeros_like(x)
    g_le = torch.zeros_like(le)
    for y in reversed(states):
        lam = torch.linalg.solve(dense(y, False), (gx + gv / dt).reshape(-1).cpu()).to(y.device).reshape(n, 3) * free
        F, lamF = fem.F(y), fem.F(lam)
        P = fem.mu[:, None, None] * F + (fem.lam * (torch.linalg.det(F) - 1.0) - fem.mu)[:, None, None] * fem._cof(F)
        g_le -= dt * dt * fem.vol * (P * lamF).sum((1, 2))  # P is linear in E
        ml = mass * lam
        gx, gv = ml - gv / dt * free, dt * ml
    return {"x": x, "grad_log_E": g_le, "grad_v0": gv}


def scene_moduli(nu):
    """(mu', lambda') per unit of Young's modulus of the SNK1 energy."""
    m, l = 1.0 / (2 * (1 + nu)), nu / ((1 + nu) * (1 - 2 * nu))
    return 4 * m / 3, l + 5 * m / 6
