"""The work that users have this framework do, as measurable cases.

A case is one stretch of a program's time loop: ``calls`` calls of one kernel on
grids that live on the GPU, one step of a batch of solves, or one convergence
norm.  The sizes are those of the configured workloads (diffusion 1-D 4096, the
2049^2 cavity in both precisions, heat 512^3), of the tests (65^2, 300^2), and
odd and ragged ones between them, in FP64 and in FP32 fields.

``draw`` gives more cases of the same kinds, sizes spread over the same ranges.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import xgrid_amd as xgrid
from xgrid_amd import _lib, norms
from xgrid_amd import workloads as W
from xgrid_amd.multi import MultiSolver

DEV = "cuda" if torch.cuda.is_available() else "cpu"


def listed() -> list:
    return [
        # the smallest calls: 1-D diffusion, 4096 cells, a stretch of its 500-step time
        # loop; one call is a few microseconds, all of it launch and host latency
        {"name": "diffusion1d_4096_f64", "kind": "diffusion_1d", "n0": 4096, "precision": "double", "calls": 50},
        # a small 2-D run as tutorials and tests make it, FP32 (the default precision)
        {"name": "diffusion2d_97_f32", "kind": "diffusion_2d", "n0": 97, "n1": 97, "precision": "float", "calls": 20},
        # an ordinary 2-D run on a ragged, non-square grid
        {"name": "diffusion2d_1100x1537_f64", "kind": "diffusion_2d", "n0": 1100, "n1": 1537,
         "precision": "double", "calls": 10},
        # the lid-driven cavity (1 + 50 pressure sweeps a call): a test-sized grid, where
        # latency counts; FP32 and odd mid sizes; and the headline size in both precisions
        {"name": "cavity_65_f64", "kind": "cavity", "n0": 65, "precision": "double", "calls": 4},
        {"name": "cavity_300_f32", "kind": "cavity", "n0": 300, "precision": "float", "calls": 2},
        {"name": "cavity_1000_f64", "kind": "cavity", "n0": 1000, "precision": "double", "calls": 1},
        {"name": "cavity_2049_f64", "kind": "cavity", "n0": 2049, "precision": "double", "calls": 1},
        {"name": "cavity_2049_f32", "kind": "cavity", "n0": 2049, "precision": "float", "calls": 1},
        # 3-D heat: the configured 512^3 FP32 grid, and a ragged FP64 one whose rows are
        # not a whole number of cache lines
        {"name": "heat3d_512_f32", "kind": "heat_3d", "n0": 512, "n1": 512, "n2": 512, "precision": "float", "calls": 4},
        {"name": "heat3d_250x333x301_f64", "kind": "heat_3d", "n0": 250, "n1": 333, "n2": 301,
         "precision": "double", "calls": 4},
        # many independent cavity and 2-D diffusion solves of sides 64 to 1024, one step of all
        {"name": "batch_16_f64", "kind": "batch", "count": 16, "mix": 1, "lo": 64, "hi": 1024, "precision": "double"},
        # an error report: L2 and Linf of an FP32 field against its FP64 twin
        {"name": "diff_norm_256_f32", "kind": "diff_norm", "n0": 256, "n1": 256, "n2": 256, "precision": "float"},
    ]


def _log(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["diffusion_1d", "diffusion_2d", "diffusion_2d", "cavity", "cavity", "cavity", "heat_3d", "heat_3d",
                       "batch", "diff_norm"])
    c = {"kind": kind, "precision": rng.choice(["double", "float"])}
    if kind == "diffusion_1d":
        return {**c, "n0": _log(rng, 64, 65536), "calls": rng.randint(10, 50)}
    if kind == "diffusion_2d":
        return {**c, "n0": _log(rng, 64, 2048), "n1": _log(rng, 64, 2048), "calls": rng.randint(4, 20)}
    if kind == "cavity":
        n = _log(rng, 33, 2049)
        return {**c, "n0": n, "calls": rng.randint(1, 4) if n <= 512 else 1}
    if kind == "batch":
        return {**c, "count": rng.randint(4, 16), "mix": rng.randint(1, 10 ** 6), "lo": 64, "hi": 1024}
    n0, n1, n2 = (_log(rng, 33, 400) for _ in range(3))
    if kind == "heat_3d":
        return {**c, "n0": n0, "n1": n1, "n2": n2, "calls": rng.randint(1, 4)}
    return {**c, "n0": n0, "n1": n1, "n2": n2}


# ------------------------------------------------------------------ inputs
def _gen(seed: int):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _waves(n: int, gen, modes: int = 4):
    """A smooth field: a few sine products with random weights, largest magnitude 1."""
    x = torch.linspace(0, math.pi, n, dtype=torch.float64, device=DEV)
    k = torch.arange(1, modes + 1, dtype=torch.float64, device=DEV)
    s = torch.sin(k[:, None] * x[None, :])
    w = torch.rand((modes, modes), generator=gen, dtype=torch.float64, device=DEV) - 0.5
    f = s.T @ w @ s
    return f / f.abs().max()


def _cavity_fields(n: int, gen):
    """A flow in progress: velocities of a smooth stream function (no net divergence),
    at rest on the walls, the lid moving; a smooth pressure."""
    psi = _waves(n, gen) * _waves(n, gen, 1)
    u, v = torch.gradient(psi)[0], -torch.gradient(psi)[1]
    s = 0.5 / torch.maximum(u.abs().max(), v.abs().max())
    u, v = u * s, v * s
    for a in (u, v):
        a[0], a[-1], a[:, 0], a[:, -1] = 0, 0, 0, 0
    u[-1] = 1.0
    p = 0.1 * _waves(n, gen)
    return [torch.zeros_like(p), p, u, v]


def _viscosity(seed: int) -> float:
    return 0.02 + 0.08 * ((int(seed) * 2654435761) % 1000) / 1000.0


def _fields(case: dict, seed: int) -> list:
    """Initial fields, as FP64 tensors (a grid of FP32 holds their rounded values)."""
    gen = _gen(seed)
    kind = case["kind"]
    if kind == "cavity":
        return _cavity_fields(case["n0"], gen)
    if kind == "batch":
        out = []
        for spec in _specs(case, seed):
            if spec.kind == "cavity":
                out += _cavity_fields(spec.n, gen)
            else:
                out.append(1.0 + 0.5 * _waves(spec.n, gen))
        return out
    shape = tuple(case[k] for k in ("n0", "n1", "n2") if k in case)
    u = torch.rand(shape, generator=gen, dtype=torch.float32, device=DEV).double()
    if kind == "diff_norm":      # a field and its rounded, slightly drifted twin
        return [u, u + 1e-6 * torch.rand(shape, generator=gen, dtype=torch.float32, device=DEV)]
    if kind != "heat_3d":
        u = u + 1.0
    return [u]


def _mask(case: dict) -> np.ndarray:
    return W.box_walls(tuple(case[k] for k in ("n0", "n1", "n2") if k in case))


def _scalars(case: dict, seed: int) -> tuple:
    nu, kind = _viscosity(seed), case["kind"]
    n = case["n0"]
    if kind == "cavity":
        return (W.cavity_config(n, dt=W.stable_dt("cavity", n, nu), nu=nu),)
    dx = 2 / (n - 1)
    return (nu, 0.1 * dx * dx / nu, dx)


def _specs(case: dict, seed: int) -> list:
    """The instances of a batch: sides and kinds from its mix, viscosities from the seed."""
    out = []
    for i, s in enumerate(W.batch_specs(case["count"], case["mix"], case["lo"], case["hi"])):
        nu = _viscosity(seed * 64 + i)
        out.append(W.InstanceSpec(s.kind, s.n, nu, W.stable_dt(s.kind, s.n, nu), rid=i))
    return out


# ------------------------------------------------------------------ programs
_OPS: dict = {}
_MAKE = {"diffusion_1d": W.make_diffusion_1d, "diffusion_2d": W.make_diffusion_2d,
         "cavity": W.make_cavity, "heat_3d": W.make_heat_3d}


class _Level:
    """A grid's current level as an array on the GPU (keeps the grid alive)."""

    def __init__(self, grid, ptr: int):
        self.grid = grid
        self.__cuda_array_interface__ = {"shape": grid.shape, "typestr": grid.numpy_dtype.str, "data": (ptr, False),
                                         "version": 2, "strides": None}


def _now(state: dict, grids: list) -> list:
    """The grids' current levels, as tensors on the GPU over the grids' own memory."""
    lib, seen, out = _lib.load(), state["views"], []
    for g in grids:
        ptr = lib.xg_grid_level_ptr(g._handle, 0)
        t = seen.get(ptr)
        if t is None:
            t = seen[ptr] = torch.as_tensor(_Level(g, ptr), device=DEV)
        out.append(t)
    return out


def _set(grid, field, mask=None) -> None:
    """A grid's field and boundary mask, current on the GPU."""
    now = grid.now
    now[...] = field.to(torch.float32 if now.dtype == np.float32 else torch.float64).cpu().numpy()
    if mask is not None:
        grid.boundary[...] = mask
    grid.class_info(0)


def prepare(case: dict, seed: int) -> dict:
    kind, precision = case["kind"], case["precision"]
    xgrid.init(precision=precision)
    fields = _fields(case, seed)
    state = {"kind": kind, "views": {}, "calls": case.get("calls", 1)}
    if kind == "batch":
        ms = MultiSolver(precision)
        state["solver"], state["grids"] = ms, []
        for spec in _specs(case, seed):
            state["grids"] += ms.grids(ms.add(spec))
        for g, f in zip(state["grids"], fields):
            _set(g, f)
        return state
    if kind == "diff_norm":
        a = xgrid.Grid(tuple(fields[0].shape), float)
        xgrid.init(precision="double")
        b = xgrid.Grid(tuple(fields[0].shape), float)
        _set(a, fields[0], _mask(case))
        _set(b, fields[1])
        state["grids"] = [a, b]
        return state
    if (kind, precision) not in _OPS:
        _OPS[kind, precision] = _MAKE[kind]()
    state["op"] = _OPS[kind, precision]
    if kind == "cavity":
        masks = [W.cavity_masks(case["n0"])[c] for c in "bpuv"]
    else:
        masks = [_mask(case)]
    state["grids"] = [xgrid.Grid(tuple(f.shape), float) for f in fields]
    for g, f, m in zip(state["grids"], fields, masks):
        _set(g, f, m)
    state["args"] = (*state["grids"], *_scalars(case, seed))
    return state


def run(state: dict):
    if state["kind"] == "diff_norm":
        r = norms.diff_norm(*state["grids"])
        return [r["l2"], r["linf"], r["cells"]]
    if state["kind"] == "batch":
        state["solver"].step(1)
        return _now(state, state["grids"])
    op, args = state["op"], state["args"]
    for _ in range(state["calls"]):
        op(*args)
    return _now(state, state["grids"])


# ------------------------------------------------------------------ counts and exact values
def _cells(case: dict) -> int:
    return case["n0"] * case.get("n1", case["n0"] if case["kind"] == "cavity" else 1) * case.get("n2", 1)


def _cavity_work(n: int, elem: int) -> tuple:
    # reads p, u, v; writes b, p, u, v; 51 sweeps of 8 operations, and the three other updates
    return 7 * n * n * elem, (51 * 8 + 80) * n * n


def work(case: dict) -> dict:
    elem = 4 if case["precision"] == "float" else 8
    kind, calls = case["kind"], case.get("calls", 1)
    if kind == "batch":
        b = f = 0
        for s in _specs(case, 0):
            x, y = _cavity_work(s.n, elem) if s.kind == "cavity" else (2 * s.n * s.n * elem, 7 * s.n * s.n)
            b, f = b + x, f + y
        return {"bytes": b, "flops": f}
    n = _cells(case)
    if kind == "cavity":
        b, f = _cavity_work(case["n0"], elem)
        return {"bytes": b * calls, "flops": f * calls}
    if kind == "diff_norm":
        return {"bytes": n * (elem + 8), "flops": 4 * n}
    per = {"diffusion_1d": 6, "diffusion_2d": 7, "heat_3d": 9}[kind]
    return {"bytes": 2 * n * elem * calls, "flops": per * n * calls}


def _held(fields: list, precision: str) -> list:
    return [f.float().double() for f in fields] if precision == "float" else fields


def _cavity_step(b, p, u, v, cfg):
    dx, dy, dt, rho, nu = cfg.dx, cfg.dy, cfg.dt, cfg.rho, cfg.nu
    i = slice(1, -1)
    un, us, ue, uw, uc = u[2:, i], u[:-2, i], u[i, 2:], u[i, :-2], u[i, i]
    vn, vs, ve, vw, vc = v[2:, i], v[:-2, i], v[i, 2:], v[i, :-2], v[i, i]
    ux, uy, vx, vy = (ue - uw) / (2 * dx), (un - us) / (2 * dy), (ve - vw) / (2 * dx), (vn - vs) / (2 * dy)
    b = torch.zeros_like(p)
    b[i, i] = rho * ((ux + vy) / dt - ux ** 2 - 2 * uy * vx - vy ** 2)
    d = 2 * (dx ** 2 + dy ** 2)
    src = dx ** 2 * dy ** 2 / d * b[i, i]
    for _ in range(51):
        q = torch.zeros_like(p)
        q[i, i] = ((p[i, 2:] + p[i, :-2]) * dy ** 2 + (p[2:, i] + p[:-2, i]) * dx ** 2) / d - src
        q[i, -1] = q[i, -2]
        q[0, 1:] = q[1, 1:]
        q[:-1, 0] = q[:-1, 1]
        q[-1] = 0
        p = q
    pe, pw, pn, ps = p[i, 2:], p[i, :-2], p[2:, i], p[:-2, i]
    U, V = torch.zeros_like(u), torch.zeros_like(v)
    U[i, i] = uc - uc * dt / dx * (uc - uw) - vc * dt / dy * (uc - us) - dt / (2 * rho * dx) * (pe - pw) + \
        nu * (dt / dx ** 2 * (ue - 2 * uc + uw) + dt / dy ** 2 * (un - 2 * uc + us))
    V[i, i] = vc - uc * dt / dx * (vc - vw) - vc * dt / dy * (vc - vs) - dt / (2 * rho * dy) * (pn - ps) + \
        nu * (dt / dx ** 2 * (ve - 2 * vc + vw) + dt / dy ** 2 * (vn - 2 * vc + vs))
    U[-1] = 1.0
    return b, p, U, V


def _diffuse(u, nu, dt, dx, wall: float):
    """One explicit diffusion step in any number of dimensions; the frame is `wall`."""
    D = u.dim()
    c = u[(slice(1, -1),) * D]
    lap = -2.0 * D * c
    for a in range(D):
        for s in (slice(2, None), slice(None, -2)):
            lap = lap + u[tuple(s if d == a else slice(1, -1) for d in range(D))]
    out = torch.full_like(u, wall)
    out[(slice(1, -1),) * D] = c + nu * dt / dx ** 2 * lap
    return out


def exact(case: dict, seed: int):
    kind, precision = case["kind"], case["precision"]
    f = _fields(case, seed)
    if kind == "diff_norm":
        d = (f[0].float().double() if precision == "float" else f[0]) - f[1]
        d = d[1:-1, 1:-1, 1:-1]
        return [float(d.square().sum().sqrt()), float(d.abs().max()), d.numel()]
    f = _held(f, precision)
    if kind == "batch":
        out, k = [], 0
        for s in _specs(case, seed):
            if s.kind == "cavity":
                out += _cavity_step(*f[k:k + 4], W.cavity_config(s.n, dt=s.dt, nu=s.nu))
                k += 4
            else:
                out.append(_diffuse(f[k], s.nu, s.dt, 2 / (s.n - 1), 1.0))
                k += 1
        return out
    args = _scalars(case, seed)
    for _ in range(case["calls"]):
        if kind == "cavity":
            f = list(_cavity_step(*f, *args))
        else:
            f = [_diffuse(f[0], *args, 0.0 if kind == "heat_3d" else 1.0)]
    return f
