"""The work that a user of this framework has it do, as measurable cases.

Every case goes through the public entry points: fdf_amd.swarm.PicGpu, the
reference's per-step interface, or the C-ABI it binds (fdf_amd._lib), with
arrays that the program keeps.  The kinds of case ("kind"):

  run       a short whole run from host arrays: upload, locate, interpolate,
            steps, download of the swarm and of the cell or face fields
  setup     a program's start: seed from the reference's random stream,
            locate from the reference's start cell, interpolate, download
  coupled   one-step calls, each after the flow solver has handed over a new
            field on the device
  advance   many steps in one call from positions on the device, downloaded
            at the end; the learned guess finds the first cells ("guess")
  fields    the same with the field prepared before every step (boundaries,
            Contra2Cart), few particles on a large grid
  stages    the reference's sweeps called one by one, two steps
  locate    picgpu_locate_device_noalloc on particles that the caller keeps
            on the device and has moved by up to a cell or two
  relocate  fresh positions on the device located from the learned guess and
            deposited onto cells and faces
  train     training the learned guess on a located swarm

Grids: "box" is the unit cube with equal cells, "cube" the unit cube with
displaced nodes, "tube" the bent pipe (fdf_amd/workloads.py).
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from fdf_amd import _lib as L
from fdf_amd import mlp
from fdf_amd import workloads as W
from fdf_amd.boundary import channel
from fdf_amd.swarm import PicGpu

DEV = "cuda" if torch.cuda.is_available() else "cpu"
CAP = 1000  # the walk's MAX_TRAVERSAL
PARTICLE_VOLUME = 1e-9


def _case(kind, grid, precision, IM, JM, KM, n, steps=1, rk2=False, faces=False, guess=False, **kw):
    return dict(kind=kind, grid=grid, precision=precision, IM=IM, JM=JM, KM=KM, n=n, steps=steps, rk2=rk2,
                faces=faces, guess=guess, **kw)


def listed():
    return [
        # the smallest simulation of the repository's configurations: ten thousand particles, ten steps
        dict(_case("run", "box", "fp64", 20, 20, 280, 10_000, steps=10), name="run small box fp64"),
        # a restart in the bent pipe with known cells, RK2 and face volume fractions
        dict(_case("run", "tube", "fp64", 48, 48, 250, 400_000, steps=50, rk2=True, faces=True),
             name="run restart tube fp64"),
        # the start of a run: seeded in the volume, located from cell (0,0,0)
        dict(_case("setup", "cube", "fp64", 63, 47, 129, 300_000), name="setup seeded cube fp64"),
        # a coupled solver's time loop: a new field, one step, a new field ...
        dict(_case("coupled", "cube", "fp64", 64, 64, 96, 500_000, steps=8), name="coupled one-step calls fp64"),
        # ordinary FP32 run on a ragged grid
        dict(_case("advance", "cube", "fp32", 61, 45, 131, 262_144, steps=64, rk2=True, faces=True),
             name="advance ragged cube fp32"),
        # the headline workload's shape (RK2, face deposition, two particles a cell), an eighth of its size
        dict(_case("advance", "cube", "fp32", 128, 128, 512, 16_777_216, steps=40, rk2=True, faces=True, guess=True),
             name="advance large cube fp32"),
        # the per-step field preparation in front of the particle step
        dict(_case("fields", "cube", "fp32", 128, 128, 192, 400_000, steps=16, rk2=True), name="fields each step fp32"),
        # the reference's sweeps replaced one by one
        dict(_case("stages", "cube", "fp64", 80, 72, 100, 800_000, steps=2), name="stage-wise sweeps fp64"),
        # a serving loop's small batch, and a large one
        dict(_case("locate", "cube", "fp32", 40, 40, 60, 3_000), name="locate device small fp32"),
        dict(_case("locate", "cube", "fp64", 128, 128, 256, 8_388_608), name="locate device large fp64"),
        # fresh positions every step, found from the learned guess, counted and deposited
        dict(_case("relocate", "tube", "fp32", 64, 64, 256, 6_000_000, guess=True), name="relocate guess tube fp32"),
        # training the guess
        dict(_case("train", "cube", "fp32", 64, 64, 64, 200_000, batch=4096, iters=200), name="train guess"),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["run", "setup", "coupled", "advance", "fields", "stages", "locate", "relocate", "train"])
    precision = rng.choice(["fp64", "fp32"])
    IM, JM, KM = size(12, 96), size(12, 96), size(12, 200)
    n = size(3_000, 2_000_000)
    if kind == "run":
        grid = rng.choice(["box", "tube"])
        if grid == "tube":
            IM = JM = 2 * size(8, 30)
        return _case(kind, grid, precision, IM, JM, KM, min(n, 600_000), steps=size(3, 60), rk2=rng.random() < 0.5,
                     faces=rng.random() < 0.5)
    if kind == "setup":
        return _case(kind, "cube", precision, IM, JM, KM, min(n, 600_000))
    if kind == "coupled":
        return _case(kind, "cube", precision, IM, JM, KM, n // 2, steps=size(2, 12), rk2=rng.random() < 0.5,
                     faces=rng.random() < 0.5)
    if kind in ("advance", "fields"):
        return _case(kind, "cube", precision, IM, JM, KM, n, steps=size(4, 64), rk2=rng.random() < 0.7,
                     faces=rng.random() < 0.6, guess=kind == "advance" and n > 500_000)
    if kind == "stages":
        return _case(kind, "cube", precision, IM, JM, KM, n // 2, steps=2)
    if kind == "locate":
        return _case(kind, "cube", precision, IM, JM, KM, size(500, 8_000_000))
    if kind == "relocate":
        IM = JM = 2 * size(12, 36)
        return _case(kind, "tube", precision, IM, JM, size(60, 300), n, guess=True)
    return _case(kind, "cube", precision, IM, JM, KM, size(20_000, 400_000), batch=32 * size(16, 400),
                 iters=size(20, 200))


# ---------------------------------------------------------------- inputs
def _inputs(case, seed):
    """Grid, field(s), positions and what else a case takes, from the seed
    alone, as tensors on the device (used by prepare and by exact)."""
    xp = W.namespace("torch", DEV)
    IM, JM, KM, n = (int(case[k]) for k in ("IM", "JM", "KM", "n"))
    gen = torch.Generator(device=DEV).manual_seed(seed)

    def rand(*shape):
        return torch.rand(*shape, generator=gen, device=DEV, dtype=torch.float64)

    d = dict(IM=IM, JM=JM, KM=KM, n=n, cells=None, gen=gen)
    if case["grid"] == "tube":
        d["coor"] = W.tube_grid(IM, JM, KM, xp=xp)
        d["ucat"] = W.ucat_poiseuille(d["coor"], IM, JM, KM, seed=seed, noise=0.05, xp=xp)
        th = rand(n)
        rho, ph = 0.99 * W.TUBE_A * torch.sqrt(rand(n)), 2 * math.pi * rand(n)
        rr = W.TUBE_R + rho * torch.cos(ph)
        d["pos"] = torch.stack([rr * torch.cos(-W.TUBE_SWEEP * th), rr * torch.sin(-W.TUBE_SWEEP * th),
                                rho * torch.sin(ph)], dim=1)
        d["dt"] = 0.5 * W.TUBE_R * W.TUBE_SWEEP / KM
        # the cell around each point in the O-grid: its ring, the place on the ring, the section along the axis
        half = IM // 2
        s = rho / W.TUBE_A
        t = 1.0 - torch.log(W.TUBE_RATIO ** half - s * (W.TUBE_RATIO ** half - 1.0)) / (half * math.log(W.TUBE_RATIO))
        top = torch.maximum(torch.cos(ph).abs(), torch.sin(ph).abs())
        at = [((1.0 + t * f(ph) / top) * half).floor().clamp(0, IM - 1) for f in (torch.cos, torch.sin)]
        d["cells"] = torch.stack([at[0], at[1], (th * KM).floor().clamp(0, KM - 1)], dim=1).to(torch.int64)
    elif case["grid"] == "box":
        d["coor"] = W.uniform_grid(IM, JM, KM, xp=xp)
        d["ucat"] = W.ucat_uniform(IM, JM, KM, (0.05, -0.02, 1.0), xp=xp)
        d["dt"] = 0.01
        d["pos"] = rand(n, 3)
    else:
        d["coor"] = W.perturbed_cube(IM, JM, KM, seed=seed, xp=xp)
        d["ucat"] = W.ucat_random_fourier(d["coor"], IM, JM, KM, seed=seed, nmodes=16, xp=xp)
        d["dt"] = 0.5 / max(IM, JM, KM) / float(d["ucat"].abs().max())
        d["pos"] = rand(n, 3)
    if case["kind"] == "coupled":
        d["ucat2"] = 0.9 * d["ucat"]
    if case["kind"] == "run":
        d["P"] = 101325.0 + 50.0 * rand(n)
    if case["kind"] == "locate":
        # start cells: where the particles were before they moved by up to 1.5 cells along each axis
        dims = torch.tensor([IM, JM, KM], device=DEV, dtype=torch.float64)
        d["cells"] = torch.minimum((d["pos"] * dims + 3.0 * rand(n, 3) - 1.5).floor().clamp(min=0), dims - 1).to(
            torch.int64)
    if case["kind"] == "fields":
        d["ucont"] = W.contravariant_from_cartesian(d["coor"], d["ucat"], IM, JM, KM).contiguous()
    return d


class State:
    pass


def _pack(d):
    c = d["cells"]
    return (c[:, 0] + d["IM"] * (c[:, 1] + d["JM"] * c[:, 2])).to(torch.int32)


def prepare(case, seed):
    d = _inputs(case, seed)
    s = State()
    s.case, s.d, s.seed = case, d, seed
    s.ctx = g = PicGpu(precision=case["precision"])
    g.upload_grid_device(d["IM"], d["JM"], d["KM"], d["coor"].data_ptr())
    g.upload_ucat_device(d["ucat"].data_ptr())
    g.set_particle_volume(PARTICLE_VOLUME)
    kind, n = case["kind"], d["n"]
    if kind == "run":
        s.host = {k: d[k].cpu().numpy() for k in ("pos", "P")}
        s.host["cell"] = None if d["cells"] is None else d["cells"].cpu().numpy()
    s.out = {"pos": np.zeros((n, 3)), "pid": np.zeros(n, np.int64)}
    if n <= 1_000_000:  # of the largest swarms only where the particles are
        s.out["vel"] = np.zeros((n, 3))
    if kind == "run":
        s.out.update(weight=np.zeros((n, 3)), cell=np.zeros((n, 3), np.int64), status=np.zeros(n, np.int64))
    if kind == "fields":
        g.compute_metrics()
        g.BoundarySystem_Create(channel(inlet_face=4, speed=0.5))
        g.upload_ucont_device(d["ucont"].data_ptr())
    if kind == "locate":
        real = torch.float64 if case["precision"] == "fp64" else torch.float32
        s.start, s.cell = _pack(d), torch.empty(n, dtype=torch.int32, device=DEV)
        s.status = torch.empty(n, dtype=torch.int32, device=DEV)
        s.weight = torch.zeros(n, 3, dtype=real, device=DEV)
        g.init_particles_device(1, d["pos"].data_ptr())
        g.LocateAllParticlesInGrid()  # lays out the grid's face planes
    if case["guess"]:
        pairs = dict(d, pos_dev=d["pos"])
        if case["grid"] == "tube":  # pairs from points whose cells are known, as a restart has them
            g.upload_particles(d["pos"][:100_000].cpu().numpy(), cell=d["cells"][:100_000].cpu().numpy())
            g.LocateAllParticlesInGrid()
            g.mlp_train(max_pairs=100_000, batch=4096, iters=2500, seed=seed % 1000)
            g.mlp_enable(True)
        else:
            mlp.train_from_walk(g, pairs, n_pairs=100_000, iters=1000, rounds=2, seed=seed % 1000)
    if kind == "train":
        g.init_particles_device(n, d["pos"].data_ptr())
        g.LocateAllParticlesInGrid()
        s.params = mlp.initial_params(seed % 1000)
    g.synchronize()
    return s


# ---------------------------------------------------------------- one pass
def _kept_download(s):
    """The swarm into the arrays that the program keeps; what it has lost leaves their tail empty."""
    m = s.ctx.n
    ptr = [s.out[k].ctypes.data_as(C.c_void_p) if k in s.out else None
           for k in ("pos", "vel", "cell", "weight", "status", "pid")]
    L.check(s.ctx.lib.picgpu_download_particles(s.ctx.h, *ptr))
    for v in s.out.values():
        v[m:] = 0
    return dict(s.out)


def _face_fractions(g):
    return [g.field(L.FIELD_IFACE_VOLFRAC + a) for a in range(3)]


def run(s):
    c, d, g = s.case, s.d, s.ctx
    kind, n, dt = c["kind"], d["n"], d["dt"]
    if kind == "run":
        g.upload_particles(s.host["pos"], cell=s.host["cell"], P=s.host["P"])
        g.LocateAllParticlesInGrid()
        g.InterpolateAllFieldsToSwarm()
        g.AdvanceSimulation(dt, c["steps"], rk2=c["rk2"], deposit_cells=True, deposit_faces=c["faces"])
        out = _kept_download(s)
        out["count"] = g.field(L.FIELD_PARTICLE_COUNT)
        if c["faces"]:
            out["faces"] = _face_fractions(g)
        else:
            out["P"] = g.field(L.FIELD_P_AVERAGE)
        return out
    if kind == "setup":
        g.InitializeParticleBasicProperties(n, volumetric=True, seed=s.seed % 100_000)
        g.LocateAllParticlesInGrid()
        g.InterpolateAllFieldsToSwarm()
        return g.download_particles()
    if kind == "coupled":
        g.init_particles_device(n, d["pos"].data_ptr())
        g.LocateAllParticlesInGrid()
        g.InterpolateAllFieldsToSwarm()
        for k in range(c["steps"]):
            g.upload_ucat_device(d["ucat2" if k % 2 else "ucat"].data_ptr())
            g.AdvanceSimulation(dt, 1, rk2=c["rk2"], deposit_cells=True, deposit_faces=c["faces"])
        out = _kept_download(s)
        out["count"] = g.field(L.FIELD_PARTICLE_COUNT)
        return out
    if kind in ("advance", "fields"):
        if kind == "fields":
            g.SetEulerianFields(1)
        g.init_particles_device(n, d["pos"].data_ptr())
        g.LocateAllParticlesInGrid()
        g.InterpolateAllFieldsToSwarm()
        g.AdvanceSimulation(dt, c["steps"], rk2=c["rk2"], deposit_cells=not c["faces"], deposit_faces=c["faces"],
                            fields=kind == "fields")
        out = _kept_download(s)
        if n <= 1_000_000:
            if c["faces"]:
                out["faces"] = _face_fractions(g)
            else:
                out["count"] = g.field(L.FIELD_PARTICLE_COUNT)
        return out
    if kind == "stages":
        g.init_particles_device(n, d["pos"].data_ptr())
        g.LocateAllParticlesInGrid()
        g.InterpolateAllFieldsToSwarm()
        for _ in range(c["steps"]):
            g.ResetAllParticleStatuses()
            g.UpdateAllParticlePositions(dt)
            g.LocateAllParticlesInGrid()
            g.CheckAndRemoveLostParticles()
            g.CheckAndRemoveOutOfBoundsParticles()
            g.InterpolateAllFieldsToSwarm()
            g.ScatterAllParticleFieldsToEulerFields()
            g.DepositParticlesToFaces(PARTICLE_VOLUME)
        return {"count": g.field(L.FIELD_PARTICLE_COUNT), "P": g.field(L.FIELD_P_AVERAGE),
                "faces": _face_fractions(g)}
    if kind == "locate":
        s.cell.copy_(s.start)
        s.status.zero_()
        torch.cuda.current_stream().synchronize()  # the library runs on a stream of its own
        L.check(g.lib.picgpu_locate_device_noalloc(g.h, n, d["pos"].data_ptr(), s.cell.data_ptr(),
                                                   s.weight.data_ptr(), s.status.data_ptr(), None))
        g.synchronize()
        return {"cell": s.cell, "weight": s.weight, "status": s.status}
    if kind == "relocate":
        g.init_particles_device(n, d["pos"].data_ptr())
        g.LocateAllParticlesInGrid()
        g.InterpolateAllFieldsToSwarm()
        g.ScatterAllParticleFieldsToEulerFields()
        g.DepositParticlesToFaces(PARTICLE_VOLUME)
        return {"count": g.field(L.FIELD_PARTICLE_COUNT), "faces": _face_fractions(g)}
    g.mlp_set_params(s.params)
    loss = g.mlp_train(max_pairs=n, batch=c["batch"], iters=c["iters"], seed=11)
    return {"params": g.mlp_get_params(), "loss": np.float32(loss)}


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    n, steps = case["n"], case["steps"]
    cells = case["IM"] * case["JM"] * case["KM"]
    r = 8 if case["precision"] == "fp64" else 4
    kind = case["kind"]
    swarm = n * (24 + 6 * r + 4 + 4 + 8 + r)  # position, velocity, weights, cell, status, PID, P
    locate = n * (24 + 4 + 3 * r + 8) + 24 * cells
    # a step reads and writes position and cell, reads the field and the nodes, and writes what it deposits
    step = n * 2 * 32 + cells * (3 * r + 3 * r + 24) + (3 * cells * 4 * r if case["faces"] else 8 * cells)
    host = n * (3 * 24 + 24 + 8 + 8)  # a downloaded swarm
    flops = n * (2 if case["rk2"] else 1) * 180.0
    if kind == "train":
        per = 3 * 2 * (64 * 64 + 6 * 64)
        return {"bytes": float(case["iters"] * (case["batch"] * 24 + 2 * 18_500)),
                "flops": float(case["iters"]) * case["batch"] * per}
    if kind == "locate":
        return {"bytes": float(locate), "flops": n * 80.0}
    if kind == "setup":
        return {"bytes": float(swarm + locate + cells * 6 * r + host), "flops": n * 300.0}
    if kind == "relocate":
        return {"bytes": float(2 * swarm + locate + cells * (6 * r + 32)), "flops": n * 10_000.0}
    if kind == "stages":
        per = locate + swarm + cells * (6 * r + 8 + 12 * r) + n * (24 + 3 * r) * 2
        return {"bytes": float(steps * per + cells * 5 * 8), "flops": steps * n * 250.0}
    if kind == "coupled":
        return {"bytes": float(swarm + locate + steps * (step + cells * (24 + 3 * r)) + n * 56 + cells * 8),
                "flops": steps * flops}
    if kind == "fields":
        return {"bytes": float(swarm + locate + steps * (step + cells * (72 + 3 * r)) + n * 56),
                "flops": steps * (flops + cells * 250.0)}
    if kind == "advance":
        return {"bytes": float(swarm + locate + steps * step + n * 56), "flops": steps * flops}
    return {"bytes": float(2 * host + locate + steps * step + cells * 32), "flops": steps * flops}


# ---------------------------------------------------------------- the same in 64 bits, in plain torch
VERTEX = [(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 1, 1), (1, 1, 1), (1, 0, 1), (0, 0, 1)]
FACE = {"back": (0, 3, 2, 1), "front": (4, 7, 6, 5), "bottom": (0, 1, 6, 7), "top": (3, 4, 5, 2),
        "left": (0, 7, 4, 3), "right": (1, 2, 5, 6)}
EDGE = [(0, 1), (1, 2), (2, 3), (3, 0), (4, 5), (5, 6), (6, 7), (7, 4), (0, 7), (1, 6), (2, 5), (3, 4)]


class _Exact:
    """The particle loop by the walking search's definition: distances to the
    six face planes, a step through every face the point is beyond."""

    def __init__(self, d):
        self.IM, self.JM, self.KM = d["IM"], d["JM"], d["KM"]
        self.dims = torch.tensor([self.IM, self.JM, self.KM], device=DEV)
        self.X = d["coor"].reshape(-1, 3)
        self.lo, self.hi = self.X.min(0).values - 1e-6, self.X.max(0).values + 1e-6

    def node(self, c, off):
        return (c[:, 0] + off[0]) + (self.IM + 1) * ((c[:, 1] + off[1]) + (self.JM + 1) * (c[:, 2] + off[2]))

    def distances(self, p, c):
        V = [self.X[self.node(c, o)] for o in VERTEX]
        h = sum((V[b] - V[a]).norm(dim=1) for a, b in EDGE) / 12
        centre = sum(V) / 8
        out = {}
        for name, (a, b, e, f) in FACE.items():
            nrm = torch.linalg.cross(V[b] - V[a], V[f] - V[a])
            fc = 0.25 * (V[a] + V[b] + V[e] + V[f])
            nrm = torch.where(((nrm * (centre - fc)).sum(1) > 1e-9)[:, None], -nrm, nrm)
            dist = ((fc - p) * nrm).sum(1) / nrm.norm(dim=1)
            out[name] = torch.where(dist.abs() < 1e-11 * h, torch.zeros_like(dist), dist)
        return out

    def walk(self, p, c):
        """Owning cells, weights and whether each point was found, from start cells c."""
        c, m = c.clone(), p.shape[0]
        w, found = torch.zeros_like(p), torch.zeros(m, dtype=torch.bool, device=DEV)
        live = torch.arange(m, device=DEV)
        seen, power, lam = torch.full((m,), -1, device=DEV, dtype=torch.int64), 1, 0
        for _ in range(CAP):
            ci = c[live]
            lin = ci[:, 0] + self.IM * (ci[:, 1] + self.JM * ci[:, 2])
            ok = ((ci >= 0) & (ci < self.dims)).all(1) & (lin != seen[live])  # a revisited cell: the walk is periodic
            live, ci, lin = live[ok], ci[ok], lin[ok]
            if live.numel() == 0:
                break
            lam += 1
            if lam == power:
                seen[live], power, lam = lin, 2 * power, 0
            t = self.distances(p[live], ci)
            stack = torch.stack(list(t.values()))
            accept = (stack.min(0).values >= 0) | (stack == 0).any(0)
            a = {k: v[accept].clamp(min=1e-14) for k, v in t.items()}
            w[live[accept]] = torch.stack([a["left"] / (a["left"] + a["right"]), a["bottom"] / (a["bottom"] + a["top"]),
                                           a["back"] / (a["front"] + a["back"])], dim=1)
            found[live[accept]] = True
            move = torch.stack([self.sign(t["right"], t["left"], False), self.sign(t["top"], t["bottom"], False),
                                self.sign(t["front"], t["back"], True)], dim=1)
            live, ci, move = live[~accept], ci[~accept], move[~accept]
            c[live] = ci + move
        return c, w, found

    @staticmethod
    def sign(up, down, up_first):
        u, v = (up < 0).long(), (down < 0).long()
        return torch.where(u > 0, u, -v) if up_first else torch.where(v > 0, -v, u)

    def corners(self, ucat):
        """Node means of the cells around each node."""
        u = ucat.reshape(self.KM + 1, self.JM + 1, self.IM + 1, 3)[:-1, :-1, :-1]
        s = torch.zeros(self.KM + 1, self.JM + 1, self.IM + 1, 3, device=DEV, dtype=torch.float64)
        k = torch.zeros(self.KM + 1, self.JM + 1, self.IM + 1, 1, device=DEV, dtype=torch.float64)
        for a in (0, 1):
            for b in (0, 1):
                for e in (0, 1):
                    at = (slice(a, a + self.KM), slice(b, b + self.JM), slice(e, e + self.IM))
                    s[at] += u
                    k[at] += 1
        return (s / k).reshape(-1, 3)

    def interpolate(self, corner, c, w, found):
        w = w.clamp(0, 1)
        c = torch.where(found[:, None], c, torch.zeros_like(c))
        u = torch.zeros_like(w)
        for a in (0, 1):
            for b in (0, 1):
                for e in (0, 1):
                    f = (w[:, 0] if a else 1 - w[:, 0]) * (w[:, 1] if b else 1 - w[:, 1]) * (
                        w[:, 2] if e else 1 - w[:, 2])
                    u += f[:, None] * corner[self.node(c, (a, b, e))]
        return torch.where(found[:, None], u, torch.zeros_like(u))

    def locate(self, d, p, cells):
        q = dict(pid=torch.arange(p.shape[0], device=DEV), x=p.clone())
        q["c"], q["w"], q["found"] = self.walk(p, torch.zeros_like(p, dtype=torch.int64) if cells is None else cells)
        return q

    def step(self, q, corner, dt, rk2):
        """One step of located or LOST particles; the removed ones leave."""
        start = torch.where(q["found"][:, None], q["c"], torch.zeros_like(q["c"]))
        x1 = q["x"] + q["u"] * dt
        c, w, found = self.walk(x1, start)
        if rk2:
            found &= q["found"]
            us = self.interpolate(corner, c, w, found)
            x1 = torch.where(found[:, None], q["x"] + (q["u"] + us) * (0.5 * dt), x1)
            c2, w, f2 = self.walk(x1, torch.where(found[:, None], c, torch.zeros_like(c)))
            c, found = c2, found & f2
        keep = found & (x1 >= self.lo).all(1) & (x1 <= self.hi).all(1)
        q = dict(pid=q["pid"][keep], x=x1[keep], c=c[keep], w=w[keep], found=found[keep])
        q["u"] = self.interpolate(corner, q["c"], q["w"], q["found"])
        return q

    def order(self, q):
        """The library's order of a stepped swarm: 8x8x4 tiles of cells, cell by cell, PID by PID."""
        i, j, k = q["c"].unbind(1)
        nti, ntj = -(-self.IM // 8), -(-self.JM // 8)
        key = ((k // 4 * ntj + j // 8) * nti + i // 8) * 256 + (k % 4 * 8 + j % 8) * 8 + i % 8
        at = torch.argsort(key, stable=True)  # the PIDs ascend already
        return {a: b[at] for a, b in q.items()}

    def count(self, q, value=None):
        out = torch.zeros(self.X.shape[0], device=DEV, dtype=torch.float64)
        one = torch.ones(q["x"].shape[0], device=DEV, dtype=torch.float64) if value is None else value
        return out.index_add_(0, self.node(q["c"], (0, 0, 0)), one)

    def volumes(self):
        k, j, i = torch.meshgrid(*(torch.arange(m, device=DEV) for m in (self.KM, self.JM, self.IM)), indexing="ij")
        c = torch.stack([i.reshape(-1), j.reshape(-1), k.reshape(-1)], dim=1)
        V = [self.X[self.node(c, o)] for o in VERTEX]
        v = torch.zeros(c.shape[0], device=DEV, dtype=torch.float64)
        for a, b in [(1, 2), (1, 6), (3, 2), (3, 4), (7, 6), (7, 4)]:
            v += ((V[a] - V[0]) * torch.linalg.cross(V[b] - V[0], V[5] - V[0])).sum(1).abs()
        return (v / 6).reshape(self.KM, self.JM, self.IM)

    def faces(self, q):
        """Face volume fractions of the deposited counts, directions i, j, k."""
        vol, out = self.volumes(), []
        for a in range(3):
            shape = [self.KM, self.JM, self.IM]
            shape[2 - a] += 1
            n, dual = (torch.zeros(shape, device=DEV, dtype=torch.float64) for _ in range(2))
            for up in (0, 1):
                c = q["c"].clone()
                c[:, a] += up
                wt = q["w"][:, a] if up else 1 - q["w"][:, a]
                n.reshape(-1).index_add_(0, c[:, 0] + shape[2] * (c[:, 1] + shape[1] * c[:, 2]), wt)
                at = [slice(None)] * 3
                at[2 - a] = slice(up, shape[2 - a] - 1 + up)
                dual[tuple(at)] += 0.5 * vol
            out.append((n * PARTICLE_VOLUME / dual).reshape(-1))
        return out


def _seeded_positions(d, seed):
    """Points of the reference's volume seeding: six drand48 draws each, cell and place in it."""
    mask, mul, add = (1 << 48) - 1, 0x5DEECE66D, 0xB
    m = 6 * d["n"]
    x = np.empty(m, np.uint64)
    x[0] = ((((seed << 16) + 0x330E) & mask) * mul + add) & mask
    k, A, B = 1, mul, add
    while k < m:  # x[q + k] = A x[q] + B
        e = min(k, m - k)
        x[k:k + e] = (x[:e] * np.uint64(A) + np.uint64(B)) & np.uint64(mask)
        k, A, B = 2 * k, (A * A) & mask, (A * B + B) & mask
    r = (torch.from_numpy(x.astype(np.float64) / 2.0 ** 48).to(DEV)).reshape(-1, 6)
    dims = torch.tensor([d["IM"], d["JM"], d["KM"]], device=DEV, dtype=torch.float64)
    c = torch.minimum((r[:, :3] * dims).floor(), dims - 1).long()
    e = _Exact(d)
    p = torch.zeros(d["n"], 3, device=DEV, dtype=torch.float64)
    for o in VERTEX:
        f = torch.ones(d["n"], device=DEV, dtype=torch.float64)
        for a in range(3):
            f = f * (r[:, 3 + a] if o[a] else 1 - r[:, 3 + a])
        p += f[:, None] * e.X[e.node(c, o)]
    return p


def exact(case, seed):
    kind = case["kind"]
    # the training's bf16 steps have no 64-bit value; the prepared field follows the solver's handlers;
    # the large swarms take too long here
    if kind in ("train", "fields") or case["n"] * (case["steps"] if kind == "advance" else 1) > 40_000_000:
        return None
    d = _inputs(case, seed)
    e = _Exact(d)
    corner = e.corners(d["ucat"])
    dbl = case["precision"] == "fp64"
    if kind == "locate":
        c, w, found = e.walk(d["pos"], d["cells"])
        return {"cell": None, "weight": torch.where(found[:, None], w, torch.zeros_like(w)), "status": None}
    if kind == "setup":
        q = e.locate(d, _seeded_positions(d, seed % 100_000), None)
    else:
        q = e.locate(d, d["pos"], d["cells"])
    q["u"] = e.interpolate(corner, q["c"], q["w"], q["found"])
    if kind == "setup":
        w = torch.where(q["found"][:, None], q["w"], torch.zeros_like(q["w"]))
        return {"pos": q["x"], "vel": q["u"], "cell": None, "weight": w, "status": None, "pid": None}
    if kind == "relocate":
        # from the guess, a point where two cells overlap may be given the other one: its faces change little
        return {"count": None, "faces": e.faces({k: v[q["found"]] for k, v in q.items()})}
    for k in range(case["steps"]):
        if kind == "coupled":
            corner = e.corners(d["ucat2" if k % 2 else "ucat"])
        q = e.step(q, corner, d["dt"], case["rk2"])
    f = e.order(q)

    def tail(v):  # in FP32 a particle beside a face may end in the next cell, which changes the order of all that follow
        return torch.cat([v, v.new_zeros(case["n"] - v.shape[0], 3)]) if dbl else None

    out = {"pos": tail(f["x"]), "pid": None}
    if case["n"] <= 1_000_000:
        out["vel"] = tail(f["u"])
    if kind == "stages":
        return {"count": e.count(q) if dbl else None, "P": None, "faces": e.faces(q)}
    if kind == "run":
        out.update(cell=None, status=None, weight=tail(f["w"]), count=e.count(q) if dbl else None)
        if case["faces"]:
            out["faces"] = e.faces(q)
        else:
            num = e.count(q)
            out["P"] = torch.where(num > 0, e.count(q, d["P"][q["pid"]]) / num.clamp(min=1), 0.0) if dbl else None
        return out
    if kind == "coupled":
        out["count"] = e.count(q) if dbl else None
    elif case["n"] <= 1_000_000:
        out["faces" if case["faces"] else "count"] = (e.faces(q) if case["faces"] else e.count(q) if dbl else None)
    return out
