"""The work that a user of this framework has it do, as cases that can be timed and compared.

A program using the library marches a solver through background steps and takes the density and
velocity of every level (or, for a checkpoint, the populations) when it wants them; before that it
trains the closure network the solver evaluates.  Each case is one such stretch:

  march    ``time_marching(steps)``, then ``macros`` of every level (and the marker forces where
           there is an immersed boundary): what a run does between two outputs.  Refined runs keep
           their levels on one stream (``level_streams_enable(False)``), so that a step is one
           chain of launches whichever HIP runtime the process has loaded
  restart  ``set_f`` of every level, two background steps, ``f`` of every level: resuming from a
           checkpoint and writing the next one
  train    ``mlp_train``: Adam steps on minibatches of filtered-DNS samples
  gradient ``mlp_gradient`` over all samples of a set

Outputs of the FP32 and BF16 solvers are kept in single precision, as the VTU files keep them.
"""
import math
from functools import lru_cache

import numpy as np
import torch

from zllbm_amd import closure, fields, grid as zg, hip, workloads
from zllbm_amd.hip import BF16_SHIFTED, FP32_SHIFTED, FP64

PRECISION = {"fp64": FP64, "fp32": FP32_SHIFTED, "bf16": BF16_SHIFTED}
STORED = {"fp64": 8, "fp32": 4, "bf16": 2}
LES = {"none": 0, "smagorinsky": 1, "learned": 2}


def listed():
    return [
        # a small enclosed flow watched after every step (a convergence criterion, a probe): one
        # launch-bound step and its fields
        dict(name="monitored cavity 32x32", kind="march", flow="cavity", nx=32, ny=32, precision="fp64",
             collision="srt", les="none", steps=1),
        # the lid-driven cavity of the test-suite and of the accuracy table
        dict(name="cavity 128x128 FP64", kind="march", flow="cavity", nx=128, ny=128, precision="fp64",
             collision="srt", les="none", steps=500),
        # a two-dimensional flow on nested refinement boxes, in double precision
        dict(name="refined cavity 256x192 3 levels", kind="march", flow="boxes", nx=256, ny=192, precision="fp64",
             collision="mrt", les="none", steps=200),
        # a large-eddy simulation in a periodic box whose edges are no multiples of a brick
        dict(name="TGV 97x80x66 FP32 LES", kind="march", flow="tgv", nx=97, ny=80, nz=66, precision="fp32",
             collision="mrt", les="smagorinsky", steps=500),
        # a direct simulation in double precision with the simplest operator
        dict(name="TGV 64^3 FP64 SRT", kind="march", flow="tgv", nx=64, ny=64, nz=64, precision="fp64",
             collision="srt", les="none", steps=500),
        # half the bytes for throughput studies, the largest uniform box here
        dict(name="TGV 128^3 BF16 LES", kind="march", flow="tgv", nx=128, ny=128, nz=128, precision="bf16",
             collision="mrt", les="smagorinsky", steps=500),
        # decaying turbulence with the learned closure on a few levels, a workstation-sized run
        dict(name="turbulence 24^3 3 levels learned", kind="march", flow="turbulence", base=24, levels=3, buffer=2,
             precision="fp32", collision="mrt", les="learned", steps=100),
        # the benchmark's flow and grid: four levels, 256^3-equivalent
        dict(name="turbulence 32^3 4 levels learned", kind="march", flow="turbulence", base=32, levels=4, buffer=6,
             precision="fp32", collision="mrt", les="learned", steps=60),
        # a refined channel around an immersed sphere: many small launches per background step
        dict(name="sphere 4 levels learned", kind="march", flow="sphere", levels=4, diameter=24, precision="fp32",
             collision="mrt", les="learned", steps=100),
        # resuming a run from its checkpoint
        dict(name="restart 24^3 3 levels FP64", kind="restart", flow="turbulence", base=24, levels=3, buffer=2,
             precision="fp64", collision="mrt", les="smagorinsky", steps=2),
        # training the closure as the training script does: minibatches of 4096, FP32 kernel
        dict(name="closure training 4096 FP32", kind="train", samples=262144, batch=4096, steps=60, form="fp32"),
        # a full gradient over a sample set on the matrix cores
        dict(name="closure gradient 70000 BF16", kind="gradient", samples=70000, form="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cavity", "cavity", "boxes", "tgv", "tgv", "tgv", "turbulence", "turbulence", "sphere",
                       "restart", "train", "gradient"])
    if kind == "cavity":
        return dict(kind="march", flow="cavity", nx=_log(rng, 24, 256), ny=_log(rng, 24, 256),
                    precision=rng.choice(["fp64", "fp64", "fp32"]), collision=rng.choice(["srt", "mrt"]), les="none",
                    steps=_log(rng, 1, 600))
    if kind == "boxes":
        return dict(kind="march", flow="boxes", nx=rng.randint(64, 320), ny=rng.randint(64, 256),
                    precision=rng.choice(["fp64", "fp32"]), collision=rng.choice(["srt", "mrt"]), les="none",
                    steps=_log(rng, 10, 300))
    if kind == "tgv":
        return dict(kind="march", flow="tgv", nx=_log(rng, 20, 112), ny=_log(rng, 20, 112), nz=_log(rng, 20, 112),
                    precision=rng.choice(["fp64", "fp32", "fp32", "bf16"]), collision=rng.choice(["srt", "mrt"]),
                    les=rng.choice(["none", "smagorinsky"]), steps=_log(rng, 10, 300))
    if kind == "turbulence":
        les, precision = rng.choice([("learned", "fp32"), ("learned", "fp32"), ("smagorinsky", "fp32"),
                                     ("smagorinsky", "fp64")])
        return dict(kind="march", flow="turbulence", base=rng.randint(20, 30), levels=rng.choice([2, 3]),
                    buffer=rng.choice([2, 4]), precision=precision, collision="mrt", les=les, steps=_log(rng, 5, 100))
    if kind == "sphere":
        return dict(kind="march", flow="sphere", levels=rng.choice([3, 4]), diameter=rng.choice([16, 20, 24]),
                    precision=rng.choice(["fp32", "fp64"]), collision="mrt",
                    les=rng.choice(["learned", "smagorinsky"]), steps=_log(rng, 5, 100))
    if kind == "restart":
        return dict(kind="restart", flow="turbulence", base=rng.randint(20, 28), levels=rng.choice([2, 3]), buffer=2,
                    precision=rng.choice(["fp64", "fp32"]), collision="mrt", les="smagorinsky", steps=rng.randint(1, 4))
    if kind == "train":
        return dict(kind="train", samples=_log(rng, 30000, 400000), batch=_log(rng, 512, 16384),
                    steps=rng.randint(20, 60), form=rng.choice(["fp32", "fp32", "bf16"]))
    return dict(kind="gradient", samples=_log(rng, 3000, 200000), form=rng.choice(["fp32", "bf16"]))


# ---- inputs ------------------------------------------------------------------------------------

@lru_cache(maxsize=None)
def _flow(flow, **size):
    """Grid, settings and markers of a flow (the mesh a program reads once), as a Workload."""
    if flow in ("cavity", "boxes"):
        cells = (size["nx"], size["ny"])
        bc = {d: (zg.BC_BOUNCE_BACK, (0., 0., 0.)) for d in range(1, 5)}
        bc[zg.YMAX] = (zg.BC_BOUNCE_BACK, (0.1, 0., 0.))
        mesh = zg.uniform_grid(2, cells)
        if flow == "boxes":
            # the middle half, and the middle half of that, twice as fine each
            lo, hi = [n // 4 for n in cells], [n - n // 4 for n in cells]
            inner = [(2 * a + (b - a) // 2, 2 * b - (b - a) // 2) for a, b in zip(lo, hi)]
            mesh = zg.refined_box_grid(2, cells, [(lo, hi), tuple(zip(*inner))])
        return workloads.Workload(flow, mesh, dict(nu0=0.1 * (max(cells) + 1) / 100.0, bc=bc))
    if flow == "tgv":
        cells = (size["nx"], size["ny"], size["nz"])
        nu = 0.05 * (max(cells) / (2 * math.pi)) / 1600.0
        return workloads.Workload("tgv", zg.uniform_grid(3, cells),
                                  dict(nu0=nu, bc=workloads.periodic_bc(3), les_tau_mode=1, cs=0.1))
    if flow == "turbulence":
        cells = (size["base"],) * 3
        modes = fields.fourier_modes(cells)
        threshold = workloads.vorticity_threshold(modes)
        mesh = zg.refined_mask_grid(3, cells, size["levels"], lambda k, c: np.linalg.norm(modes.vorticity(c), axis=1)
                                    > threshold, buffer=size["buffer"])
        return workloads.Workload("turbulence", mesh, dict(nu0=1e-4 * (1 << (size["levels"] - 1)), cs=0.1,
                                                           bc=workloads.periodic_bc(3), les_tau_mode=1))
    return workloads.sphere_amr(levels=size["levels"], diameter_fine=size["diameter"])


def _workload(case):
    return _flow(case["flow"], **{k: case[k] for k in ("nx", "ny", "nz", "base", "levels", "buffer", "diameter")
                                  if k in case})


@lru_cache(maxsize=None)
def _model():
    return closure.ClosureModel.load(zg.__file__.rsplit("/", 1)[0] + "/data/closure_turbulence.npz")


def _initial(case, W, seed):
    """Density and velocity of every level, numpy float64."""
    rng = np.random.default_rng(seed)
    out = []
    if case["flow"] == "cavity":
        # at rest but for the noise a program seeds to break the symmetry
        n = W.grid.levels[0].n
        return [(1.0 + rng.normal(0.0, 1e-4, n), rng.normal(0.0, 1e-3, (n, 2)))]
    if case["flow"] == "boxes":
        # a smooth solenoidal field, the same on every level
        out, box, wave = [], np.array(W.grid.cells), rng.integers(1, 5, (6, 2)) * math.pi
        amp, phase = rng.normal(0.0, 0.3, 6), rng.uniform(0.0, 2 * math.pi, 6)
        for l in range(W.grid.max_level + 1):
            x = (W.grid.coords(l).astype(np.float64) / (1 << l) - 1.0) / box
            s = np.cos(x @ wave.T + phase) * (amp * 0.003)
            out.append((np.ones(len(x)), np.stack([s @ wave[:, 1], -(s @ wave[:, 0]) * box[1] / box[0]], 1)))
        return out
    if case["flow"] == "tgv":
        cells = np.array([case["nx"], case["ny"], case["nz"]])
        at = (W.grid.coords(0).astype(np.int64) - 1) % cells   # the duplicated planes carry their twins' values
        k = 2 * math.pi / cells
        x = at * k
        u0 = 0.05
        u = np.zeros(at.shape)
        u[:, 0] = u0 * np.sin(x[:, 0]) * np.cos(x[:, 1]) * np.cos(x[:, 2])
        u[:, 1] = -u0 * min(1.0, k[0] / k[1]) * np.cos(x[:, 0]) * np.sin(x[:, 1]) * np.cos(x[:, 2])
        noise = rng.normal(0.0, 1e-3, (int(np.prod(cells)), 3))
        u += noise[(at[:, 0] * cells[1] + at[:, 1]) * cells[2] + at[:, 2]]
        rho = 1.0 + 3.0 * (u0 ** 2 / 16.0) * (np.cos(2 * x[:, 0]) + np.cos(2 * x[:, 1])) * (np.cos(2 * x[:, 2]) + 2.0)
        return [(rho, u)]
    if case["flow"] == "turbulence":
        modes = fields.fourier_modes((case["base"],) * 3, seed=seed)
        d = "cuda" if torch.cuda.is_available() else "cpu"
        wave, dirs = (torch.from_numpy(v).to(d) for v in ((modes.k / modes.box).T.copy(), modes.dirs * modes.amp[:, None]))
        phase = torch.from_numpy(modes.phase).to(d)
        for l in range(W.grid.max_level + 1):
            at = torch.from_numpy(W.grid.coords(l).astype(np.int32)).to(d).double() / (1 << l) - 1.0
            u = torch.cat([torch.cos(2 * math.pi * (part @ wave) + phase) @ dirs for part in at.split(1 << 20)])
            out.append((np.ones(len(u)), u.cpu().numpy()))
        return out
    # channels: the workload's inflow everywhere, perturbed
    return [(rho, u * (1.0 + rng.normal(0.0, 0.01, len(u)))[:, None]) for rho, u in W.init]


def _samples(case, seed):
    """Normalised inputs (heavy-tailed, correlated) and targets: an eddy viscosity in units of its
    mean, zero where the filtered stress scatters back."""
    rng = np.random.default_rng(seed)
    n = case["samples"]
    x = rng.standard_normal((n, closure.NF), dtype=np.float32)
    x[:, 0] = np.abs(x[:, 0]) - 0.8
    x[:, 7] = x[:, 0] + 0.1 * x[:, 7]
    x[:, 8] = x[:, 0] * x[:, 0] - 0.5 + 0.1 * x[:, 8]
    t = np.maximum(0.0, 1.0 + 0.9 * x[:, 0] - 0.3 * x[:, 2] * x[:, 4] + 0.5 * rng.standard_normal(n, dtype=np.float32))
    return x, t.astype(np.float32)


def _solver(case, W):
    kw = dict(W.solver, collision=(hip.MRT if case["collision"] == "mrt" else hip.SRT,), les=LES[case["les"]])
    if case["les"] == "learned":
        kw["mlp_operands"] = hip.MLP_OPERANDS_FP16
    s = hip.Solver(W.grid, precision=PRECISION[case["precision"]], **kw)
    ib = getattr(W, "ib", None)
    if ib is not None:
        s.set_ib(ib.level, ib.xyz, ib.area, np.zeros_like(ib.xyz), stencil_dis=2)
    if W.grid.max_level > 0:
        s.level_streams_enable(False)
    s.build()
    if case["les"] == "learned":
        s.mlp_set(_model())
    return s


def prepare(case, seed):
    if case["kind"] in ("train", "gradient"):
        x, t = _samples(case, seed)
        s = hip.Solver(zg.uniform_grid(2, (8, 8)), nu0=0.1, bc={d: (zg.BC_BOUNCE_BACK, (0., 0., 0.)) for d in range(1, 5)})
        return dict(case=case, solver=s, x=x, t=t, params=closure.init_params(seed),
                    form=hip.MLP_FP32 if case["form"] == "fp32" else hip.MLP_BF16_MFMA)
    W = _workload(case)
    s = _solver(case, W)
    for l, (rho, u) in enumerate(_initial(case, W, seed)):
        s.init_macro(l, rho, u)
    state = dict(case=case, solver=s, levels=W.grid.max_level + 1, ib=getattr(W, "ib", None))
    if case["kind"] == "restart":
        # the populations a checkpoint holds
        s.time_marching(4)
        state["f"] = [s.f(l) for l in range(state["levels"])]
    return state


# ---- one pass ----------------------------------------------------------------------------------

def run(state):
    case, s = state["case"], state["solver"]
    if case["kind"] == "train":
        params, losses = s.mlp_train(state["params"], state["x"], state["t"], case["steps"], case["batch"], 2e-3,
                                     form=state["form"])
        return dict(params=params, losses=losses)
    if case["kind"] == "gradient":
        loss, grad = s.mlp_gradient(state["params"], state["x"], state["t"], form=state["form"])
        return dict(grad=grad, loss=np.float32(loss))
    if case["kind"] == "restart":
        for l, f in enumerate(state["f"]):
            s.set_f(l, f)
    s.time_marching(case["steps"])
    out = {}
    for l in range(state["levels"]):
        if case["kind"] == "restart":
            out["f%d" % l] = _kept(case, s.f(l))
        else:
            rho, u = s.macros(l)
            out["rho%d" % l], out["u%d" % l] = _kept(case, rho), _kept(case, u)
    if state["ib"] is not None:
        out["force"] = s.ib_force(state["ib"].level)
        if case["precision"] != "fp64":
            out["force"] = out["force"].astype(np.float32)
    return out


def _kept(case, v):
    v = torch.from_numpy(v)
    return v if case["precision"] == "fp64" else v.float()


# ---- what a pass cannot do without ---------------------------------------------------------------

def work(case):
    if case["kind"] in ("train", "gradient"):
        forward = 2 * (9 * 32 + 32 * 32 + 32) + 65 * 6
        n = min(case["batch"], case["samples"]) * case["steps"] if case["kind"] == "train" else case["samples"]
        return {"bytes": case["samples"] * 40 + closure.NPARAM * 4 * 2, "flops": 3.0 * forward * n}
    W = _workload(case)
    dims = W.grid.dims
    q = 9 if dims == 2 else 19
    updates = W.updates_per_step * case["steps"]
    nodes = sum(W.nodes)
    # moments, equilibrium, relaxation and the way back per node; the network where there is one
    per_node = (8 if case["collision"] == "srt" else 14) * q + (60 if case["les"] != "none" else 0)
    if case["les"] == "learned":
        per_node += 2 * (9 * 32 + 32 * 32 + 32) + 65 * 4
    values = 2 * q if case["kind"] == "restart" else 1 + dims
    return {"bytes": 2.0 * q * STORED[case["precision"]] * updates + 8.0 * values * nodes, "flops": float(per_node) * updates}


# ---- the same in 64 bits, in plain torch and numpy ------------------------------------------------

def exact(case, seed):
    if case["kind"] in ("train", "gradient"):
        return _exact_closure(case, seed)
    if case["kind"] == "march" and case["flow"] in ("tgv", "cavity"):
        return _exact_uniform(case, seed)
    return None   # refined grids: no short plain form of the level coupling


def _net(p):
    at = np.cumsum([0, 288, 32, 1024, 32, 32, 1])
    W1, b1, W2, b2, w3, b3 = (p[a:b] for a, b in zip(at, at[1:]))
    return W1.reshape(32, 9), b1, W2.reshape(32, 32), b2, w3, b3


def _loss_and_grad(p, x, t):
    W1, b1, W2, b2, w3, b3 = _net(p)
    z1 = x @ W1.T + b1
    s1 = 1 / (1 + np.exp(-z1))
    h1 = z1 * s1
    z2 = h1 @ W2.T + b2
    s2 = 1 / (1 + np.exp(-z2))
    h2 = z2 * s2
    z3 = h2 @ w3 + b3
    y = np.logaddexp(0.0, z3)
    d3 = 2 * (y - t) / len(t) / (1 + np.exp(-z3))
    d2 = d3[:, None] * w3 * s2 * (1 + z2 * (1 - s2))
    d1 = (d2 @ W2) * s1 * (1 + z1 * (1 - s1))
    g = np.concatenate([(d1.T @ x).ravel(), d1.sum(0), (d2.T @ h1).ravel(), d2.sum(0), h2.T @ d3, [d3.sum()]])
    return np.mean((y - t) ** 2), g


def _batch(seed, it, batch, n):
    """Sample indices of minibatch `it` (the seeded hash that mlp_train documents)."""
    u32 = np.uint32
    with np.errstate(over="ignore"):
        h = u32((seed * 1000003 + it) & 0xFFFFFFFF) * u32(2654435761) + np.arange(batch, dtype=u32)
        h ^= h >> u32(16)
        h *= u32(0x7FEB352D)
        h ^= h >> u32(15)
        h *= u32(0x846CA68B)
        h ^= h >> u32(16)
    return h.astype(np.int64) % n


def _exact_closure(case, seed):
    x, t = (v.astype(np.float64) for v in _samples(case, seed))
    p = closure.init_params(seed).astype(np.float64)
    if case["kind"] == "gradient":
        loss, g = _loss_and_grad(p, x, t)
        return dict(grad=g, loss=np.float64(loss))
    m, v, losses = np.zeros_like(p), np.zeros_like(p), []
    for it in range(1, case["steps"] + 1):
        at = slice(None) if case["batch"] >= len(t) else _batch(20261202, it, case["batch"], len(t))
        loss, g = _loss_and_grad(p, x[at], t[at])
        losses.append(loss)
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        p = p - 2e-3 * (m / (1 - 0.9 ** it)) / (np.sqrt(v / (1 - 0.999 ** it)) + 1e-8)
    return dict(params=p, losses=np.array(losses))


def _lattice(dims):
    if dims == 2:
        c = [(0, 0), (1, 0), (0, 1), (-1, 0), (0, -1), (1, 1), (-1, 1), (-1, -1), (1, -1)]
    else:
        c = [(0, 0, 0)] + [tuple(s if a == b else 0 for b in range(3)) for a in range(3) for s in (1, -1)]
        for a, b in ((0, 1), (0, 2), (1, 2)):
            for sb in (1, -1):
                for sa in (1, -1):
                    c.append(tuple(sa if k == a else sb if k == b else 0 for k in range(3)))
    c = np.array(c)
    w = {2: {0: 4 / 9, 1: 1 / 9, 2: 1 / 36}, 3: {0: 1 / 3, 1: 1 / 18, 2: 1 / 36}}[dims]
    return c, np.array([w[int(k)] for k in (c * c).sum(1)])


def _moments(c):
    """Rows of the orthogonal moment basis, their fixed rates (None: the viscous rate)."""
    c2 = (c * c).sum(1)
    if c.shape[1] == 2:
        x, y = c.T
        rows = [1 + 0 * x, 3 * c2 - 4, (9 * c2 ** 2 - 21 * c2) // 2 + 4, x, (3 * c2 - 5) * x, y, (3 * c2 - 5) * y,
                x * x - y * y, x * y]
        return np.array(rows, float), [0, 1.4, 1.4, 0, 1.2, 0, 1.2, None, None]
    x, y, z = c.T
    rows = [1 + 0 * x, 19 * c2 - 30, (21 * c2 ** 2 - 53 * c2 + 24) // 2, x, (5 * c2 - 9) * x, y, (5 * c2 - 9) * y, z,
            (5 * c2 - 9) * z, 3 * x * x - c2, (3 * c2 - 5) * (3 * x * x - c2), y * y - z * z,
            (3 * c2 - 5) * (y * y - z * z), x * y, y * z, x * z, (y * y - z * z) * x, (z * z - x * x) * y,
            (x * x - y * y) * z]
    return np.array(rows, float), [0, 1.5, 1.4, 0, 1.2, 0, 1.2, 0, 1.2, None, 1.4, None, 1.4, None, None, None, 1.98,
                                   1.98, 1.98]


def _exact_uniform(case, seed):
    W = _workload(case)
    rho0, u0 = _initial(case, W, seed)[0]
    cells = W.grid.cells
    dims, wall = len(cells), case["flow"] == "cavity"
    shape = tuple(n + 1 for n in cells) if wall else cells   # a periodic box keeps one of each duplicated plane
    at = W.grid.coords(0).astype(np.int64) - 1
    at = at if wall else at % np.array(cells)
    flat = torch.from_numpy(np.ravel_multi_index(tuple(at.T), shape))
    d = "cuda" if torch.cuda.is_available() else "cpu"
    rho, u = torch.ones(math.prod(shape), dtype=torch.float64), torch.zeros(math.prod(shape), dims, dtype=torch.float64)
    rho[flat], u[flat] = torch.from_numpy(rho0), torch.from_numpy(u0)
    rho, u = rho.to(d), u.to(d)
    c, w = _lattice(dims)
    C, w_ = torch.from_numpy(c.astype(float)).to(d), torch.from_numpy(w).to(d)

    def equilibrium(rho, u):
        cu = C @ u.T
        return w_[:, None] * rho * (1 + 3 * cu + 4.5 * cu * cu - 1.5 * (u * u).sum(1))

    M, rates = _moments(c)
    M = torch.from_numpy(M).to(d)
    back = M.T / (M * M).sum(1)
    viscous = [k for k, s in enumerate(rates) if s is None]
    fixed = torch.tensor([0.0 if s is None else s for s in rates], dtype=torch.float64, device=d)[:, None]
    tau0 = 3 * W.solver["nu0"] + 0.5
    opposite = [int(np.nonzero((c == -e).all(1))[0][0]) for e in c]
    f = equilibrium(rho, u)
    for _ in range(case["steps"]):
        rho = f.sum(0)
        u = (C.T @ f / rho).T
        neq = f - equilibrium(rho, u)
        tau = torch.full_like(rho, tau0)
        if case["les"] == "smagorinsky":
            pi = torch.einsum("qa,qb,qn->abn", C, C, neq)
            tau = tau0 + 0.5 * (torch.sqrt(tau0 ** 2 + 18 * 0.1 ** 2 * torch.sqrt(2 * (pi * pi).sum((0, 1)))) - tau0)
        if case["collision"] == "srt":
            post = f - neq / tau
        else:
            m = M @ neq
            relaxed = fixed * m
            relaxed[viscous] = m[viscous] / tau
            post = f - back @ relaxed
        post = post.reshape(-1, *shape)
        f = torch.stack([torch.roll(post[q], tuple(int(k) for k in c[q]), tuple(range(dims))) for q in range(len(c))])
        if wall:
            # bounce-back of the wall nodes, minimum faces first; the lid moves along x
            for axis, end in ((0, 0), (1, 0), (0, -1), (1, -1)):
                face = tuple(end if a == axis else slice(None) for a in range(dims))
                lid = 0.1 if (axis, end) == (1, -1) else 0.0
                for q in range(len(c)):
                    if c[q][axis] == (1 if end == 0 else -1):
                        o = opposite[q]
                        f[q][face] = post[o][face] - 6 * w[o] * c[o][0] * lid
        f = f.reshape(len(c), -1)
    rho = f.sum(0)
    u = (C.T @ f / rho).T
    flat = flat.to(d)
    return dict(rho0=rho[flat].cpu(), u0=u[flat].cpu())
