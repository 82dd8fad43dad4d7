"""What a user of the direct-sum library has it do, as cases that can be timed.

The library replaces the O(T*S) particle sums of a vortex / PSE code and the RK4
steps around them, so the cases are those calls at the sizes of the library's
own workloads (lpmgpu.workloads, lpmgpu.configs): icosahedral and cubed-sphere
meshes, planar grids, one rank's block of targets, many problems at once, the
learned far field and the training of its network.  Calls on host arrays get
host arrays, as from the Fortran solvers; solvers keep their state on the GPU.

Results come in the type of the precision asked for: `fp64` calls as the
library's float64 arrays, `fp32` calls (FP32 pairs, results defined up to FP32
rounding) as the float32 arrays that a single-precision program keeps.
"""
from __future__ import annotations

import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "lpm-v2_amd"))

from lpmgpu import BVEBatch, BVESolver, Context, ic, mesh  # noqa: E402
from lpmgpu.farfield import EXPANSION, LEARNED, N_PARAMS, FarFieldBVE  # noqa: E402
from lpmgpu.mlp import ACT_ISRU, Mlp  # noqa: E402

OMEGA = 2.0 * math.pi


def listed():
    return [
        # the smallest drop-in call: one evaluation of a coarse run (icosahedral
        # level 4, 7,682 particles) from the reference's own FP64 loop; call
        # overhead and latency count
        {"name": "velocity_icos4_fp64", "op": "velocity", "mesh": "icos", "level": 4, "precision": "fp64",
         "i0": 0, "i1": 7682},
        # a whole RK4 step of the same run by the device-resident solver, replayed as a graph
        {"name": "step_icos4_fp64", "op": "step", "mesh": "icos", "level": 4, "precision": "fp64"},
        # the precision workload: cubed sphere, level 7 (196,610 particles), FP32 pairs
        {"name": "velocity_cubed7_fp32", "op": "velocity", "mesh": "cubed", "level": 7, "precision": "fp32",
         "i0": 0, "i1": 196610},
        # one of 8 MPI ranks at the headline size (icosahedral level 8, 1,966,082 particles)
        {"name": "velocity_icos8_rank_fp32", "op": "velocity", "mesh": "icos", "level": 8, "precision": "fp32",
         "i0": 491520, "i1": 737280},
        # stream functions at the reference's precision, an odd block of a mid-size run
        {"name": "stream_icos6_fp64", "op": "stream", "mesh": "icos", "level": 6, "precision": "fp64",
         "i0": 10007, "i1": 104003},
        # planar vortex sums on the 512^2 grid
        {"name": "plane_velocity_512_fp32", "op": "plane_velocity", "side": 512, "active_per_mille": 1000,
         "precision": "fp32"},
        # the PSE workload: Laplacian on the jittered 512^2 grid, eps = 2h
        {"name": "pse8_laplacian_512_fp32", "op": "pse_laplacian", "side": 512, "order": 8, "precision": "fp32"},
        # a first-derivative PSE operator on the sphere at the reference's precision
        {"name": "sphere_gradient_icos6_fp64", "op": "sphere_gradient", "mesh": "icos", "level": 6,
         "precision": "fp64", "i0": 0, "i1": 122882},
        # one right-hand side of a planar shallow-water run, ragged grid
        {"name": "swe_rhs_301_fp32", "op": "swe", "side": 301, "precision": "fp32"},
        # an ensemble of uneven problems, one RK4 step of all of them
        {"name": "batch_20_fp32", "op": "batch", "problems": 20, "max_level": 6, "precision": "fp32"},
        # one evaluation with the learned far field (near sums, expansions, network)
        {"name": "far_field_icos7", "op": "far_field", "level": 7, "mode": LEARNED, "near": 0.1, "band": 0.2,
         "parents": 0.6},
        # forward and backward of the far field's network on a training batch
        {"name": "network_grad_32768", "op": "network_grad", "samples": 32768},
    ]


def draw(rng):
    op = rng.choice(["velocity", "velocity", "stream", "step", "plane_velocity", "pse_laplacian", "sphere_gradient",
                     "sphere_interpolate", "swe", "batch", "far_field", "network_grad"])
    prec = rng.choice(["fp64", "fp32"])
    if op in ("velocity", "stream", "sphere_gradient"):
        kind = rng.choice(["icos", "cubed"])
        level = rng.randint(3, 7)
        n = _particles(kind, level)
        share = 1.0 if n < 30000 else rng.choice([1.0, 0.5, 0.25]) if n < 200000 else rng.uniform(0.1, 0.3)
        size = min(n, max(1, int(n * share * rng.uniform(0.9, 1.0))))
        i0 = rng.randint(0, n - size)
        return {"op": op, "mesh": kind, "level": level, "precision": prec, "i0": i0, "i1": i0 + size}
    if op == "step":
        return {"op": op, "mesh": rng.choice(["icos", "cubed"]), "level": rng.randint(3, 6), "precision": prec}
    if op in ("plane_velocity", "pse_laplacian", "swe"):
        side = int(round(math.exp(rng.uniform(math.log(40), math.log(360 if prec == "fp64" else 512)))))
        case = {"op": op, "side": side, "precision": prec}
        if op == "pse_laplacian":
            case["order"] = rng.choice([2, 8])
        if op == "plane_velocity":
            case["active_per_mille"] = rng.choice([1000, rng.randint(300, 999)])
        return case
    if op == "sphere_interpolate":
        return {"op": op, "level": rng.randint(4, 7), "lats": rng.randint(30, 181), "precision": prec}
    if op == "batch":
        return {"op": op, "problems": rng.randint(2, 20 if prec == "fp32" else 6), "max_level": rng.randint(4, 6),
                "precision": prec}
    if op == "far_field":
        return {"op": op, "level": rng.randint(5, 7), "mode": rng.choice([EXPANSION, LEARNED]),
                "near": rng.choice([0.1, 0.12, 0.15]), "band": rng.choice([0.2, 0.25]),
                "parents": rng.choice([0.0, 0.6])}
    return {"op": op, "samples": int(round(math.exp(rng.uniform(math.log(1000), math.log(130000)))))}


# ------------------------------------------------------------------- inputs


def _particles(kind, level):
    return 30 * 4**level + 2 if kind == "icos" else 12 * 4**level + 2


def _sources(kind, level):
    return 20 * 4**level if kind == "icos" else 6 * 4**level


@functools.lru_cache(maxsize=8)
def _mesh(kind, level, cell_level=-1):
    make = mesh.icosahedral_mesh if kind == "icos" else mesh.cubed_sphere_mesh
    return make(level, cell_level=cell_level)


@functools.lru_cache(maxsize=1)
def _context():
    return Context(0)


def _sphere(case, seed):
    """The mesh turned by a random rotation, and vorticity of 1-4 random vortices on a wave."""
    m = _mesh(case.get("mesh", "icos"), case["level"])
    rng = np.random.default_rng(seed)
    rot, _ = np.linalg.qr(rng.normal(size=(3, 3)))
    x, y, z = (np.ascontiguousarray(a) for a in (m.xyz() @ rot).T)
    zeta = ic.random_gaussian_vortices(rng, int(rng.integers(1, 5)), x, y, z) + ic.rh4_vorticity(x, y, z)
    return dict(x=x, y=y, z=z, relvort=zeta, absvort=zeta + 2 * OMEGA * z, area=m.area, active=m.active,
                eps=float(m.max_edge_length**0.75))


def _plane(case, seed):
    """A jittered grid, as particles are after a few steps, with smooth fields on it."""
    side = case["side"]
    rng = np.random.default_rng(seed)
    x, y, area, h = mesh.grid_centres(side, 1.0, jitter=0.5 / side, seed=seed)
    cx, cy = rng.uniform(-0.4, 0.4, 2)
    r2 = (x - cx) ** 2 + (y - cy) ** 2
    active = np.ones(x.size, np.int32)
    if case.get("active_per_mille", 1000) < 1000:
        active = (rng.uniform(size=x.size) * 1000 < case["active_per_mille"]).astype(np.int32)
    return dict(x=x, y=y, area=area, active=active, eps=2.0 * h, f=np.exp(-8.0 * r2), vort=3.0 * np.exp(-4 * r2),
                div=0.5 * np.sin(2 * x) * np.cos(y + cx), h=1.0 + 0.1 * np.exp(-6 * r2), bottom=0.05 * x - 0.02 * y * y)


def _batch(case, seed):
    """Uneven problems: the levels belong to the case, the vortices to the seed."""
    levels = np.random.default_rng(case["problems"]).integers(3, case["max_level"] + 1, case["problems"])
    out = []
    for k, level in enumerate(levels):
        p = _sphere({"level": int(level)}, seed * 1000 + k)
        out.append(dict(x=p["x"], y=p["y"], z=p["z"], relvort=p["relvort"], area=p["area"], active=p["active"],
                        radius=1.0, rotation_rate=OMEGA))
    return out


def _latlon(lats):
    la = np.linspace(-0.5 * np.pi, 0.5 * np.pi, lats)
    lo = np.arange(2 * lats - 2) * (np.pi / (lats - 1))
    la, lo = (a.ravel() for a in np.meshgrid(la, lo, indexing="ij"))
    return np.cos(lo) * np.cos(la), np.sin(lo) * np.cos(la), np.sin(la)


def _network(seed):
    """Weights of a trained network's size: fan-in scaled, a small last layer."""
    rng = np.random.default_rng(seed)
    parts = []
    for nin, nout, gain in ((13, 128, 1.0), (128, 128, 1.0), (128, 128, 1.0), (128, 3, 0.3)):
        parts += [rng.normal(size=nout * nin) * gain / math.sqrt(nin), rng.normal(size=nout) * 0.05]
    return np.concatenate(parts).astype(np.float32)


def _samples(case, seed):
    rng = np.random.default_rng(seed + 1)
    x = rng.normal(size=(case["samples"], 13)).astype(np.float32)
    t = np.tanh(x[:, :3] * x[:, 3:6]).astype(np.float32)
    return x, t


def prepare(case, seed):
    ctx = _context()
    op = case["op"]
    if op in ("velocity", "stream", "sphere_gradient", "sphere_interpolate"):
        s = _sphere(case, seed)
        if op == "sphere_interpolate":
            s["points"] = _latlon(case["lats"])
    elif op in ("plane_velocity", "pse_laplacian", "swe"):
        s = _plane(case, seed)
    elif op == "step":
        p = _sphere(case, seed)
        s = {"solver": BVESolver(ctx, p["x"], p["y"], p["z"], p["relvort"], p["area"], p["active"],
                                 rotation_rate=OMEGA, precision=case["precision"], use_graph=True, project=True)}
    elif op == "batch":
        s = {"batch": BVEBatch(ctx, _batch(case, seed), precision=case["precision"], use_graph=True, project=True)}
    elif op == "far_field":
        m = _mesh("icos", case["level"], 3)
        rng = np.random.default_rng(seed)
        zeta = ic.random_gaussian_vortices(rng, int(rng.integers(1, 5)), m.x, m.y, m.z) + ic.rh4_vorticity(m.x, m.y, m.z)
        ff = FarFieldBVE(ctx, m, zeta, rotation_rate=OMEGA, near_radius=case["near"], band_radius=case["band"],
                         parent_radius=case["parents"])
        ff.set_params(_network(seed))
        s = {"ff": ff}
    else:
        net = Mlp(ctx, act=ACT_ISRU)
        net.set_params(_network(seed))
        x, t = _samples(case, seed)
        s = {"net": net, "x": x, "t": t}
    return {"case": dict(case), "ctx": ctx, **s}


# ---------------------------------------------------------------- one pass


def run(s):
    c, ctx = s["case"], s["ctx"]
    op, prec = c["op"], c.get("precision", "fp32")
    if op == "velocity":
        out = ctx.bve_sphere_velocity(s["x"], s["y"], s["z"], s["relvort"], s["area"], s["active"],
                                      i0=c["i0"], i1=c["i1"], precision=prec)
    elif op == "stream":
        out = ctx.bve_sphere_stream(s["x"], s["y"], s["z"], s["relvort"], s["absvort"], s["area"], s["active"],
                                    i0=c["i0"], i1=c["i1"], precision=prec)
    elif op == "sphere_gradient":
        out = ctx.pse_sphere_gradient(s["x"], s["y"], s["z"], s["relvort"], s["area"], s["active"], s["eps"],
                                      i0=c["i0"], i1=c["i1"], precision=prec)
    elif op == "sphere_interpolate":
        out = (ctx.pse_sphere_interpolate(s["x"], s["y"], s["z"], s["relvort"], s["area"], s["active"], s["eps"],
                                          *s["points"], precision=prec),)
    elif op == "plane_velocity":
        out = ctx.plane_velocity(s["x"], s["y"], s["vort"], s["area"], s["active"], precision=prec)
    elif op == "pse_laplacian":
        out = (ctx.pse_plane_laplacian(s["x"], s["y"], s["f"], s["area"], s["active"], s["eps"], order=c["order"],
                                       precision=prec),)
    elif op == "swe":
        out = ctx.swe_plane_rhs(s["x"], s["y"], s["vort"], s["div"], s["h"], s["bottom"], s["area"], s["active"],
                                s["eps"], precision=prec)
    elif op == "step":
        s["solver"].timestep(0.01)
        out = tuple(s["solver"].state().values())
    elif op == "batch":
        s["batch"].timestep(0.01)
        out = tuple(s["batch"].state().values())
    elif op == "far_field":
        out = s["ff"].velocity(c["mode"])
    else:
        loss, grad = s["net"].loss_grad(s["x"], s["t"])
        return {"loss": loss, "grad": grad}
    return tuple(a.astype(np.float32) for a in out) if prec == "fp32" else tuple(out)


# ------------------------------------------------- what a pass cannot do without

# flops per pair (+, -, * = 1, fma = 2, rcp / exp / log = 1)
_FLOPS = {"velocity": 23, "stream": 11, "sphere_gradient": 43, "sphere_interpolate": 32, "plane_velocity": 11}


def _reach(precision):
    """Separation, in eps, beyond which exp(-rho^2) is zero in the precision."""
    return math.sqrt(126 * math.log(2)) if precision == "fp32" else math.sqrt(745.0)


def work(case):
    op, prec = case["op"], case.get("precision", "fp32")
    if op in ("velocity", "stream", "sphere_gradient", "sphere_interpolate"):
        kind, level = case.get("mesh", "icos"), case["level"]
        n, ns = _particles(kind, level), _sources(kind, level)
        nt = case["i1"] - case["i0"] if "i0" in case else case["lats"] * (2 * case["lats"] - 2)
        fields, outs = {"velocity": (5, 3), "stream": (6, 2), "sphere_gradient": (5, 3)}.get(op, (5, 1))
        pairs = nt * ns
        if op.startswith("sphere_"):
            edge = math.sqrt(4 * math.pi / ns) * (1.7 if kind == "icos" else 1.25)
            cap = min(2.0, _reach(prec) * edge**0.75)
            pairs *= min(1.0, cap * cap / 4.0)  # share of the sphere within the chord
        return {"bytes": 8 * fields * n + 4 * n + 8 * outs * nt, "flops": _FLOPS[op] * pairs}
    if op in ("plane_velocity", "pse_laplacian", "swe"):
        n = case["side"] ** 2
        near = n * min(1.0, math.pi * (_reach(prec) * 2.0 / case["side"] * 2.0) ** 2 / 4.0)
        ns = n * case.get("active_per_mille", 1000) / 1000
        if op == "plane_velocity":
            return {"bytes": n * (8 * 4 + 4 + 16), "flops": 11 * n * ns}
        if op == "pse_laplacian":
            return {"bytes": n * (8 * 4 + 4 + 8), "flops": (18 if case["order"] == 8 else 11) * n * near}
        return {"bytes": n * (8 * 7 + 4 + 32), "flops": n * (37 * n + 14 * near)}
    if op == "step":
        n, ns = _particles(case["mesh"], case["level"]), _sources(case["mesh"], case["level"])
        return {"bytes": 8 * 15 * n, "flops": 4 * 23 * n * ns}
    if op == "batch":
        levels = np.random.default_rng(case["problems"]).integers(3, case["max_level"] + 1, case["problems"])
        n = [(_particles("icos", int(k)), _sources("icos", int(k))) for k in levels]
        return {"bytes": 8 * 15 * sum(a for a, _ in n), "flops": 4 * 23 * sum(a * b for a, b in n)}
    net = 2 * (13 * 128 + 2 * 128 * 128 + 128 * 3)
    if op == "far_field":
        # of 1,280 cells: those within the near radius summed directly, one expansion for each other
        n, ns = _particles("icos", case["level"]), _sources("icos", case["level"])
        near = 1280 * ((case["near"] + 0.16) / 2.0) ** 2
        band = 1280 * ((case["band"] + 0.16) / 2.0) ** 2 - near
        far = 462 if case["parents"] else 1258
        return {"bytes": n * (8 * 5 + 4 + 24),
                "flops": n * (23 * near * ns / 1280 + 150 * far + (net * band if case["mode"] == LEARNED else 0))}
    return {"bytes": case["samples"] * 16 * 4 + 2 * 4 * N_PARAMS, "flops": 3 * net * case["samples"]}


# ------------------------------------------------------- the same in 64 bits


def _gpu(*arrays):
    return [torch.from_numpy(np.asarray(a, dtype=np.float64)).cuda() for a in arrays]


def _pair_sums(term, targets, sources, tgt_index, src_index, nout):
    """sum_j term(target block, sources) with the pairs of equal index left out."""
    nt, ns = targets[0].numel(), max(1, sources[0].numel())
    out = torch.zeros(nout, nt, dtype=torch.float64, device="cuda")
    step = max(1, min(nt, (1 << 26) // ns))
    for a in range(0, nt, step):
        b = min(nt, a + step)
        skip = None if tgt_index is None else tgt_index[a:b, None] == src_index[None, :]
        for k, v in enumerate(term([t[a:b, None] for t in targets], [q[None, :] for q in sources], skip)):
            out[k, a:b] = v
    return out


def _velocity64(x, y, z, q, area, active, i0=0, i1=None):
    """Sphere Biot-Savart sum, radius 1: denominator 1 - x.y as (|x - y|^2 + e_i + e_j) / 2."""
    idx = torch.nonzero(active).reshape(-1)
    i1 = x.numel() if i1 is None else i1
    e = 1.0 - (x * x + y * y + z * z)
    w = -q * area / (2 * math.pi)

    def term(t, s, skip):
        d = [t[k] - s[k] for k in range(3)]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2] + t[3] + s[3]
        f = (s[4] / r2).masked_fill_(skip, 0.0)
        return [(f * dk).sum(1) for dk in d]

    tg = [a[i0:i1] for a in (x, y, z, e)]
    if (i1 - i0) * idx.numel() > 5e10:
        A = _velocity64_products(torch.stack(tg[:3], 1), torch.stack([x, y, z], 1)[idx], w[idx], idx - i0)
    else:
        A = _pair_sums(term, tg, [a[idx] for a in (x, y, z, e, w)], torch.arange(i0, i1, device="cuda"), idx, 3)
    tx, ty, tz = tg[:3]
    return torch.stack([A[1] * tz - A[2] * ty, A[2] * tx - A[0] * tz, A[0] * ty - A[1] * tx])


def _velocity64_products(X, Y, w, self_row):
    """The same sums by matrix products, for the largest blocks: the denominator
    2 - 2 x.y is good to about 1e-10 of its value at these spacings."""
    nt, ns = X.shape[0], Y.shape[0]
    left = torch.cat([-2 * X, torch.full((nt, 1), 2.0, dtype=X.dtype, device="cuda")], 1)
    right = torch.cat([Y, torch.ones(ns, 1, dtype=X.dtype, device="cuda")], 1)
    weighted = right * w[:, None]
    acc = torch.zeros(nt, 4, dtype=X.dtype, device="cuda")
    for b in range(0, ns, 16384):
        cols = slice(b, min(ns, b + 16384))
        rt, wt, row = right[cols].T.contiguous(), weighted[cols].contiguous(), self_row[cols]
        for a in range(0, nt, 8192):
            f = (left[a:a + 8192] @ rt).reciprocal_()
            here = torch.nonzero((row >= a) & (row < a + f.shape[0])).reshape(-1)
            f[row[here] - a, here] = 0.0
            acc[a:a + 8192] += f @ wt
    return (X * acc[:, 3:] - acc[:, :3]).T


def _step64(p, dt):
    """One RK4 step with every stage point put back on the unit sphere."""
    X = torch.stack(_gpu(p["x"], p["y"], p["z"]))
    zeta, area = _gpu(p["relvort"], p["area"])
    active = torch.from_numpy(np.asarray(p["active"]) != 0).cuda()

    def on(v):
        return v / v.square().sum(0).sqrt()

    def rate(v, q):
        u = _velocity64(v[0], v[1], v[2], q, area, active)
        return dt * u, -dt * 2.0 * OMEGA * u[2]

    X = on(X)
    ks = [rate(X, zeta)]
    for h in (0.5, 0.5, 1.0):
        ks.append(rate(on(X + h * ks[-1][0]), zeta + h * ks[-1][1]))
    new = [a + (k[0] + 2 * k[1] + 2 * k[2] + k[3]) / 6.0 for a, k in ((X, [k[0] for k in ks]), (zeta, [k[1] for k in ks]))]
    X, zeta = on(new[0]), new[1]
    u = _velocity64(X[0], X[1], X[2], zeta, area, active)
    return [X[0], X[1], X[2], zeta, u[0], u[1], u[2]]


def _back(outs, n=None, i0=0):
    """Host arrays of length n with the block's values at i0 (the rest zero)."""
    got = []
    for o in outs:
        a = o.cpu().numpy()
        if n is not None and a.size < n:
            b = np.zeros(n)
            b[i0:i0 + a.size] = a
            a = b
        got.append(a)
    return tuple(got)


def exact(case, seed):
    op = case["op"]
    if op == "far_field":
        return None  # an approximation: its value is not a sum in 64 bits
    if op == "network_grad":
        params = torch.from_numpy(_network(seed)).cuda().double().requires_grad_(True)
        x, t = (torch.from_numpy(a).cuda().double() for a in _samples(case, seed))
        at = 0
        for k, (nin, nout) in enumerate(((13, 128), (128, 128), (128, 128), (128, 3))):
            wt = params[at:at + nin * nout].reshape(nout, nin)
            at += nin * nout
            x = x @ wt.T + params[at:at + nout]
            at += nout
            x = x / (1 + x * x).sqrt() if k < 3 else x
        loss = (x - t).square().mean()
        (grad,) = torch.autograd.grad(loss, params)
        return {"loss": float(loss), "grad": grad.cpu().numpy()}
    if op == "step":
        return _back(_step64(_sphere(case, seed), 0.01))
    if op == "batch":
        steps = [_step64(p, 0.01) for p in _batch(case, seed)]
        return _back([torch.cat([s[k] for s in steps]) for k in range(7)])
    if op in ("plane_velocity", "pse_laplacian", "swe"):
        return _exact_plane(case, seed)
    return _exact_sphere(case, seed)


def _exact_sphere(case, seed):
    op = case["op"]
    p = _sphere(case, seed)
    n = p["x"].size
    i0, i1 = case.get("i0", 0), case.get("i1", n)
    x, y, z, q, area = _gpu(p["x"], p["y"], p["z"], p["relvort"], p["area"])
    active = torch.from_numpy(np.asarray(p["active"]) != 0).cuda()
    idx = torch.nonzero(active).reshape(-1)
    if op == "velocity":
        return _back(_velocity64(x, y, z, q, area, active, i0, i1), n, i0)
    if op == "stream":
        (qa,) = _gpu(p["absvort"])
        e = 1.0 - (x * x + y * y + z * z)

        def term(t, s, skip):
            r2 = (t[0] - s[0]).square() + (t[1] - s[1]).square() + (t[2] - s[2]).square() + t[3] + s[3]
            lg = (0.5 * r2).masked_fill_(skip, 1.0).log_()
            return [(lg * s[4]).sum(1), (lg * s[5]).sum(1)]

        w = [-a * area / (4 * math.pi) for a in (q, qa)]
        return _back(_pair_sums(term, [a[i0:i1] for a in (x, y, z, e)], [a[idx] for a in (x, y, z, e, *w)],
                                torch.arange(i0, i1, device="cuda"), idx, 2), n, i0)
    eps = p["eps"]

    def rho2(d):
        chord = (d[0].square() + d[1].square() + d[2].square()).sqrt_()
        return (2.0 / eps * torch.asin((0.5 * chord).clamp_(max=1.0))).square_()

    if op == "sphere_interpolate":
        pts = _gpu(*_latlon(case["lats"]))

        def term(t, s, skip):
            r2 = rho2([t[k] - s[k] for k in range(3)])
            ker = (4 - 6 * r2 + 2 * r2.square() - r2**3 / 6) * torch.exp(-r2) / math.pi
            return [(ker * s[3]).sum(1) / eps**2]

        return _back(_pair_sums(term, pts, [a[idx] for a in (x, y, z, q * area)], None, None, 1))

    def term(t, s, skip):
        d = [t[k] - s[k] for k in range(3)]
        r2 = rho2(d)
        ker = (-20 + 20 * r2 - 5 * r2.square() + r2**3 / 3) * torch.exp(-r2) / (math.pi * eps**4)
        f = (ker * (t[3] + s[3]) * s[4]).masked_fill_(skip, 0.0)
        return [(f * dk).sum(1) for dk in d]

    tg = [a[i0:i1] for a in (x, y, z, q)]
    g = _pair_sums(term, tg, [a[idx] for a in (x, y, z, q, area)], torch.arange(i0, i1, device="cuda"), idx, 3)
    dot = g[0] * tg[0] + g[1] * tg[1] + g[2] * tg[2]
    return _back([g[k] - dot * tg[k] for k in range(3)], n, i0)


def _exact_plane(case, seed):
    op = case["op"]
    p = _plane(case, seed)
    x, y, area = _gpu(p["x"], p["y"], p["area"])
    idx = torch.nonzero(torch.from_numpy(p["active"]).cuda()).reshape(-1)
    me = torch.arange(x.numel(), device="cuda")
    eps = p["eps"]
    if op == "plane_velocity":
        (w,) = _gpu(p["vort"] * p["area"] / (2 * math.pi))

        def term(t, s, skip):
            dx, dy = t[0] - s[0], t[1] - s[1]
            f = (s[2] / (dx * dx + dy * dy)).masked_fill_(skip, 0.0)
            return [-(f * dy).sum(1), (f * dx).sum(1)]

        return _back(_pair_sums(term, [x, y], [a[idx] for a in (x, y, w)], me, idx, 2))

    def laplacian(r2, f):
        ker = (40 - 40 * r2 + 10 * r2.square() - 2 * r2**3 / 3) / math.pi
        return ((ker if case.get("order", 8) == 8 else 4 / math.pi) * torch.exp(-r2) * f).sum(1) / eps**4

    if op == "pse_laplacian":
        (f,) = _gpu(p["f"])

        def term(t, s, skip):
            r2 = ((t[0] - s[0]).square() + (t[1] - s[1]).square()) / eps**2
            return [laplacian(r2, (s[2] - t[2]) * s[3])]

        return _back(_pair_sums(term, [x, y, f], [a[idx] for a in (x, y, f, area)], me, idx, 1))
    vort, div, surf = _gpu(p["vort"], p["div"], p["h"] + p["bottom"])

    def term(t, s, skip):
        X, Y = t[0] - s[0], t[1] - s[1]
        r2 = X * X + Y * Y
        f = (1.0 / r2).masked_fill_(skip, 0.0)
        a, b = s[2] * f, s[3] * f
        f2 = 2 * f
        p1, p2 = (X * b - Y * a) * f2, (Y * b + X * a) * f2
        return [(-Y * a + X * b).sum(1), (X * a + Y * b).sum(1), (b - X * p1).sum(1), (-a - Y * p1).sum(1),
                (a - X * p2).sum(1), (b - Y * p2).sum(1), laplacian(r2 / eps**2, (s[4] - t[2]) * s[5])]

    S = _pair_sums(term, [x, y, surf],
                   [a[idx] for a in (x, y, vort * area / (2 * math.pi), div * area / (2 * math.pi), surf, area)],
                   me, idx, 7)
    return _back([S[0], S[1], S[2] ** 2 + 2 * S[3] * S[4] + S[5] ** 2, S[6]])
