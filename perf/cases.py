"""The work a user of numbacs_amd has it do, as measurable cases.

Each case runs one pass through the public entry points over inputs made from
a seed: flow maps of analytic and gridded flows with their FTLE fields and
ridges, batched time series, auxiliary grids, sliding composition windows,
the set-up of a gridded flow, the analysis of a large stored flow map, and
the surrogate's inference and gradients.  Fields are sums of drifting Fourier
modes on a 0.5 degree, hourly lon/lat grid (RMS speed 30 km/h) and particle
grids cover the whole box, as in the benchmark workloads.
"""
import math

import numpy as np
import torch

from numbacs_amd import _lib
from numbacs_amd.batch import FTLEBatch
from numbacs_amd.diagnostics import (C_eig_aux_2D, ftle_eig_2d_device, ftle_grid_2D,
                                     ftle_grid_2d_device)
from numbacs_amd.extraction.ridges import ftle_ridges_device_async
from numbacs_amd.flows import (get_flow_2D, get_flow_linear_2D, get_predefined_flow, ingest_xy,
                               prefilter3_device)
from numbacs_amd.integration import (FlowmapComposer, flowmap_aux_grid_2d_device,
                                     flowmap_grid_2D, flowmap_grid_2d_device)
from numbacs_amd.surrogate import MLPSurrogate, grid_inputs

PRECISION = {"fp64": _lib.NBX_FP64, "fp32": _lib.NBX_FP32_DISP}
BOX = ((-100.0, 35.0), (-5.0, 45.0))


def listed():
    return [
        # one interactive call on a coarse double-gyre grid, numpy in and out
        dict(name="gyre_host", kind="analytic", flow="double_gyre", api="host", nx=81, ny=41,
             T=-10.0, precision="fp64"),
        # the double-gyre FTLE example at its own size, device to device
        dict(name="gyre", kind="analytic", flow="double_gyre", api="device", nx=401, ny=201,
             T=-10.0, precision="fp64"),
        # the Bickley jet over 40 days: long chaotic trajectories
        dict(name="bickley", kind="analytic", flow="bickley_jet", api="device", nx=1001, ny=401,
             T=-40.0, precision="fp64"),
        # one step of the gridded-velocity workload: flow map, FTLE with
        # eigenvectors, ridges above the 90th percentile
        dict(name="step", kind="step", nx=676, ny=251, T=-72.0, precision="fp64"),
        # an FTLE time series: uneven requests and windows in one batch
        dict(name="series_fp32", kind="series", requests=8, nx=901, ny=333, precision="fp32"),
        # auxiliary-grid flow map (five particles a point) and its eigenpairs
        dict(name="aux", kind="aux", nx=338, ny=126, T=-72.0),
        # flow map over the trilinear interpolant of the same samples
        dict(name="trilinear", kind="trilinear", nx=676, ny=251, T=-72.0),
        # one slide of a 72 h composition window: a 6 h map and the composed map
        dict(name="window", kind="window", nx=676, ny=251, h=6.0, maps=12),
        # set-up of a gridded flow from raw samples: ingest, prefilter, handle
        dict(name="setup", kind="setup", frames=96),
        # FTLE with eigenvectors and ridges of a large stored flow map
        dict(name="field", kind="field", nx=4001, ny=2001),
        # surrogate displacements of a 0.05 degree particle grid
        dict(name="infer", kind="infer", nx=2701, ny=1001),
        # loss and gradients of one surrogate training batch
        dict(name="train", kind="train", batch=8192),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["analytic", "step", "series", "aux", "trilinear", "window", "setup",
                       "field", "infer", "train"])
    precision = rng.choice(["fp64", "fp64", "fp32"])
    if kind == "analytic":
        if rng.random() < 0.6:
            nx = _log_int(rng, 21, 1601)
            return dict(kind=kind, flow="double_gyre", api=rng.choice(["host", "device"]), nx=nx,
                        ny=max(5, int(nx * rng.uniform(0.4, 0.6))), T=rng.uniform(-10.0, -4.0),
                        precision="fp64")
        nx = _log_int(rng, 41, 801)
        return dict(kind=kind, flow="bickley_jet", api="device", nx=nx,
                    ny=max(5, int(nx * rng.uniform(0.3, 0.5))), T=rng.uniform(-40.0, -10.0),
                    precision=precision)
    if kind in ("step", "trilinear", "aux"):
        nx = _log_int(rng, 34, 338 if kind == "aux" else 700)
        c = dict(kind=kind, nx=nx, ny=max(9, int(nx * rng.uniform(0.3, 0.45))),
                 T=-rng.uniform(24.0, 72.0))
        return dict(c, precision=precision) if kind == "step" else c
    if kind == "series":
        nx = _log_int(rng, 101, 901)
        return dict(kind=kind, requests=rng.randint(2, 8), nx=nx, ny=int(nx * 0.37),
                    precision=rng.choice(["fp64", "fp32"]) if nx < 451 else "fp32")
    if kind == "window":
        nx = _log_int(rng, 68, 676)
        return dict(kind=kind, nx=nx, ny=max(25, int(nx * rng.uniform(0.3, 0.4))),
                    h=rng.choice([3.0, 6.0]), maps=rng.randint(4, 12))
    if kind == "setup":
        return dict(kind=kind, frames=_log_int(rng, 12, 128))
    if kind == "field":
        nx = _log_int(rng, 201, 4001)
        return dict(kind=kind, nx=nx, ny=max(51, int(nx * rng.uniform(0.4, 0.5))))
    if kind == "infer":
        nx = _log_int(rng, 34, 2701)
        return dict(kind=kind, nx=nx, ny=max(13, int(nx * 0.37)))
    return dict(kind=kind, batch=64 * _log_int(rng, 8, 256))


# ---------------------------------------------------------------------------
# Inputs.

def _dev(a):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda")


def _axes(case):
    return np.linspace(*BOX[0], case["nx"]), np.linspace(*BOX[1], case["ny"])


def _velocity(seed, frames):
    """(grid tuple, U, V): (frames, 271, 101) km/h on the device."""
    rng = np.random.default_rng(seed)
    X = torch.linspace(0, 1, 271, dtype=torch.float64, device="cuda")[:, None]
    Y = torch.linspace(0, 1, 101, dtype=torch.float64, device="cuda")[None, :]
    t = torch.arange(frames, dtype=torch.float64, device="cuda")[:, None, None]
    U = torch.zeros((frames, 271, 101), dtype=torch.float64, device="cuda")
    V = torch.zeros_like(U)
    power, count = 0.0, 0
    while count < 64:
        kx, ky = int(rng.integers(-12, 13)), int(rng.integers(0, 13))
        k = math.hypot(kx, ky)
        if not 1 <= k <= 12:
            continue
        count += 1
        cu, cv = ky / 50.0 / k ** 2, -kx / 135.0 / k ** 2
        phase, omega = rng.uniform(0, 2 * math.pi), 2 * math.pi * rng.uniform(-1, 1) / 24.0
        wave = torch.sin((2 * math.pi * (kx * X + ky * Y) + phase) - omega * t)
        U.add_(wave, alpha=cu)
        V.add_(wave, alpha=cv)
        power += 0.5 * (cu * cu + cv * cv)
    grid = ((0.0, frames - 1.0, frames), (*BOX[0], 271), (*BOX[1], 101))
    return grid, U.mul_(30.0 / math.sqrt(power)), V.mul_(30.0 / math.sqrt(power))


def _spline_flow(seed, frames=96):
    grid, U, V = _velocity(seed, frames)
    return get_flow_2D(grid, prefilter3_device(U), prefilter3_device(V), spherical=1)


def _gyre_rhs(t, x, y, p):
    a = p[2] * math.sin(p[4] * t + p[5])
    f = a * x * x + (1 - 2 * a) * x
    df = 2 * a * x + (1 - 2 * a)
    return (-math.pi * p[1] * torch.sin(math.pi * f) * torch.cos(math.pi * y),
            math.pi * p[1] * torch.cos(math.pi * f) * torch.sin(math.pi * y) * df)


def _gyre_map(x, y, p, t0, T, steps):
    """Double-gyre flow map (nx, ny, 2) by the classic fourth-order method."""
    X, Y = (a.clone() for a in torch.meshgrid(_dev(x), _dev(y), indexing="ij"))
    h = T / steps
    for k in range(steps):
        t = t0 + k * h
        a0, b0 = _gyre_rhs(t, X, Y, p)
        a1, b1 = _gyre_rhs(t + h / 2, X + h / 2 * a0, Y + h / 2 * b0, p)
        a2, b2 = _gyre_rhs(t + h / 2, X + h / 2 * a1, Y + h / 2 * b1, p)
        a3, b3 = _gyre_rhs(t + h, X + h * a2, Y + h * b2, p)
        X = X + h / 6 * (a0 + 2 * a1 + 2 * a2 + a3)
        Y = Y + h / 6 * (b0 + 2 * b1 + 2 * b2 + b3)
    return torch.stack([X, Y], -1)


def _gyre_params(rng):
    return np.array([-1.0, rng.uniform(0.09, 0.11), rng.uniform(0.2, 0.3), 0.0, 0.2 * math.pi,
                     rng.uniform(0, 1)])


def _network(rng):
    return MLPSurrogate(shift=[-32.5, 20.0, 72.0, -48.0], scale=[67.5, 25.0, 24.0, 24.0],
                        out_scale=[12.0, 6.0], seed=int(rng.integers(1 << 30)))


def prepare(case, seed):
    rng = np.random.default_rng(seed + 1)
    kind = case["kind"]
    s = dict(case)
    if kind == "analytic":
        s["flow"], p, dom = get_predefined_flow(case["flow"], int_direction=-1.0)
        s["params"] = _gyre_params(rng) if case["flow"] == "double_gyre" else p
        s["params"][0] = -1.0
        s["t0"] = rng.uniform(0.0, 5.0)
        s["x"], s["y"] = np.linspace(*dom[0], case["nx"]), np.linspace(*dom[1], case["ny"])
        s["dx"], s["dy"] = s["x"][1] - s["x"][0], s["y"][1] - s["y"][0]
    elif kind in ("step", "aux", "trilinear", "window"):
        if kind == "trilinear":
            s["flow"] = get_flow_linear_2D(*_velocity(seed, 96), spherical=1)
        else:
            s["flow"] = _spline_flow(seed)
        s["params"] = np.array([-1.0])
        s["t0"] = 72.0 + rng.uniform(0.0, 20.0)
        s["x"], s["y"] = _axes(case)
        s["dx"], s["dy"] = s["x"][1] - s["x"][0], s["y"][1] - s["y"][0]
        if kind == "window":
            s["params"] = np.array([1.0])
            s["composer"] = FlowmapComposer(s["flow"], s["x"], s["y"], case["h"], case["maps"],
                                            s["params"]).initial(0.0)
            s["slides"] = 0
    elif kind == "series":
        s["flow"] = _spline_flow(seed)
        reqs = []
        for k in range(case["requests"]):
            # uneven grids: golden-ratio fractions of the largest, 0.3 to 1
            nx = int(case["nx"] * (0.3 + 0.7 * ((k + 1) * 0.618 % 1))) + 2
            ny = int(case["ny"] * (0.3 + 0.7 * ((k + 4) * 0.618 % 1))) + 2
            reqs.append(dict(t0=72.0 + k, T=(-24.0, -48.0, -72.0)[k % 3],
                             x=np.linspace(*BOX[0], nx), y=np.linspace(*BOX[1], ny)))
        s["batch"] = FTLEBatch(s["flow"], reqs, [-1.0], precision=case["precision"])
    elif kind == "setup":
        s["grid"], U, V = _velocity(seed, case["frames"])
        s["u"] = (U / 3.6).transpose(1, 2).contiguous()
        s["v"] = (V / 3.6).transpose(1, 2).contiguous()
    elif kind == "field":
        s["x"], s["y"] = np.linspace(0, 2, case["nx"]), np.linspace(0, 1, case["ny"])
        s["fm"] = _gyre_map(s["x"], s["y"], _gyre_params(rng), rng.uniform(0, 5), -10.0, 40)
        s["dx"], s["dy"] = s["x"][1] - s["x"][0], s["y"][1] - s["y"][0]
    elif kind == "infer":
        s["net"] = _network(rng)
        s["inp"] = grid_inputs(*_axes(case), 72.0 + rng.uniform(0.0, 24.0), -72.0)
    else:
        s["net"] = _network(rng)
        gen = torch.Generator(device="cuda").manual_seed(seed)
        u = torch.rand((case["batch"], 4), generator=gen, device="cuda")
        s["inp"] = ((2 * u - 1) * s["net"].scale + s["net"].shift).contiguous()
        s["target"] = torch.randn((case["batch"], 2), generator=gen, device="cuda")
    if "x" in s:
        s["xd"], s["yd"] = _dev(s["x"]), _dev(s["y"])
    if kind in ("step", "field"):
        # ridge outputs a serving loop keeps, as large as the grid
        n = case["nx"] * case["ny"]
        s["pts"] = torch.zeros((n, 2), dtype=torch.float64, device="cuda")
        s["offsets"] = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
        s["counts"] = torch.zeros(3, dtype=torch.int64, device="cuda")
    return s


# ---------------------------------------------------------------------------
# One pass.

def run(s):
    kind = s["kind"]
    if kind == "analytic" and s["api"] == "host":
        fm = flowmap_grid_2D(s["flow"], s["t0"], s["T"], s["x"], s["y"], s["params"])
        return dict(flowmap=fm, ftle=ftle_grid_2D(fm, s["T"], s["dx"], s["dy"]))
    if kind in ("analytic", "trilinear", "step"):
        fm = flowmap_grid_2d_device(s["flow"], s["t0"], s["T"], s["xd"], s["yd"], s["params"],
                                    precision=PRECISION[s.get("precision", "fp64")])
        if kind != "step":
            return dict(flowmap=fm, ftle=ftle_grid_2d_device(fm, s["T"], s["dx"], s["dy"]))
        ftle, evec = ftle_eig_2d_device(fm, s["T"], s["dx"], s["dy"])
        return dict(flowmap=fm, ftle=ftle, evec=evec, **_ridges(s, ftle, evec))
    if kind == "series":
        s["batch"].run()
        return [dict(flowmap=r["flowmap"], ftle=r["ftle"]) for r in s["batch"].requests]
    if kind == "aux":
        fm = flowmap_aux_grid_2d_device(s["flow"], s["t0"], s["T"], s["xd"], s["yd"], s["params"])
        evals, evecs = C_eig_aux_2D(fm, s["dx"], s["dy"])
        return dict(flowmap=fm, evals=evals, evecs=evecs)
    if kind == "window":
        c = s["composer"]
        c.step(s["h"] * s["maps"] + s["slides"] % 12)
        s["slides"] += 1
        return dict(composed=c.compose())
    if kind == "setup":
        Cu = prefilter3_device(ingest_xy(s["u"], 3.6))
        Cv = prefilter3_device(ingest_xy(s["v"], 3.6))
        s["flow"] = get_flow_2D(s["grid"], Cu, Cv, spherical=1)
        return dict(Cu=Cu, Cv=Cv)
    if kind == "field":
        ftle, evec = ftle_eig_2d_device(s["fm"], -10.0, s["dx"], s["dy"])
        return dict(ftle=ftle, evec=evec, **_ridges(s, ftle, evec))
    if kind == "infer":
        return dict(displacement=s["net"].predict_device(s["inp"]))
    loss, gW, gb = s["net"].gradients(s["inp"], s["target"])
    return dict(loss=loss, gW=gW, gb=gb)


def _ridges(s, ftle, evec):
    pts, offsets, counts = ftle_ridges_device_async(
        ftle, evec, s["xd"], s["yd"], s["nx"], s["ny"], s["dx"], s["dy"], percentile=90,
        pts=s["pts"], offsets=s["offsets"], counts=s["counts"])
    return dict(ridge_pts=pts, ridge_offsets=offsets, ridge_counts=counts)


# ---------------------------------------------------------------------------
# What one pass cannot do without.

def _grid_work(particles, steps, rhs_flops, out_bytes=24):
    """steps attempted per particle, 12 right-hand sides of rhs_flops and 350
    solver operations each; a particle's outputs are written once."""
    return dict(bytes=particles * out_bytes, flops=particles * steps * (350 + 12 * rhs_flops))


def work(case):
    kind = case["kind"]
    n = case.get("nx", 1) * case.get("ny", 1)
    if kind == "analytic":
        if case["flow"] == "double_gyre":
            return _grid_work(n, 2.2 * abs(case["T"]), 35)
        return _grid_work(n, 3.0 * abs(case["T"]), 60)
    if kind in ("step", "aux", "trilinear"):
        rhs = 60 if kind == "trilinear" else 400
        w = _grid_work(n * (5 if kind == "aux" else 1), abs(case["T"]) / 3.0, rhs)
        w["bytes"] += 96 * 273 * 103 * 16 + n * (48 if kind == "aux" else 32)
        return w
    if kind == "series":
        w = _grid_work(0.42 * n * case["requests"], 16, 400)
        w["bytes"] += 96 * 273 * 103 * 16
        return w
    if kind == "window":
        w = _grid_work(n, 4, 400, out_bytes=16)
        w["bytes"] += n * 16 * (case["maps"] + 1)
        return w
    if kind == "setup":
        samples, coefs = case["frames"] * 271 * 101, (case["frames"] + 2) * 273 * 103
        # raw samples read, coefficients written, both handle copies written
        return dict(bytes=2 * 8 * samples + 2 * 8 * coefs + 32 * coefs, flops=2 * 24 * coefs)
    if kind == "field":
        # flow map read, FTLE and eigenvector written, both read for the ridges
        return dict(bytes=n * (16 + 24 + 24), flops=n * 60)
    mlp = 2 * (128 * 256 + 3 * 256 * 256 + 256 * 2)
    if kind == "infer":
        return dict(bytes=n * 24, flops=n * mlp)
    return dict(bytes=case["batch"] * 24 + 4 * mlp, flops=case["batch"] * 3 * mlp)


# ---------------------------------------------------------------------------
# The same outputs in plain 64-bit arithmetic.  None for trajectories through
# gridded fields (their right-hand sides jump at the box edge and kink at
# cell faces) and for the chaotic jet: a plain solution of those to rounding
# accuracy is not a matter of seconds.

def _stencil(fm, T, dx, dy):
    """FTLE of a flow map by central differences, zero on the border."""
    gx = (fm[2:, 1:-1] - fm[:-2, 1:-1]) / (2 * dx)
    gy = (fm[1:-1, 2:] - fm[1:-1, :-2]) / (2 * dy)
    a, b, d = (gx * gx).sum(-1), (gx * gy).sum(-1), (gy * gy).sum(-1)
    lam = 0.5 * (a + d) + torch.sqrt((0.5 * (a - d)) ** 2 + b * b)
    ftle = torch.zeros(fm.shape[:2], dtype=fm.dtype, device=fm.device)
    ftle[1:-1, 1:-1] = torch.where(lam > 1, torch.log(lam) / (2 * abs(T)), 0.0)
    return ftle


def _spline_axis(c, axis):
    """Natural cubic B-spline coefficients of samples along one axis."""
    n = c.shape[axis]
    M = torch.zeros((n + 2, n + 2), dtype=c.dtype, device=c.device)
    k = torch.arange(n, device=c.device)
    for d, w in ((0, 1 / 6), (1, 4 / 6), (2, 1 / 6)):
        M[k + 1, k + d] = w
    M[0, :3] = torch.tensor([1.0, -2.0, 1.0])
    M[n + 1, n - 1:] = torch.tensor([1.0, -2.0, 1.0])
    inv = torch.linalg.inv(M)[:, 1:n + 1]
    return torch.tensordot(inv, c, dims=([1], [axis])).movedim(0, axis)


def exact(case, seed):
    kind = case["kind"]
    if kind == "analytic" and case["flow"] == "double_gyre":
        s = prepare(case, seed)
        fm = _gyre_map(s["x"], s["y"], s["params"], s["t0"], s["T"], 800)
        return dict(flowmap=fm, ftle=_stencil(fm, s["T"], s["dx"], s["dy"]))
    if kind == "setup":
        s = prepare(case, seed)
        out = {}
        for name, raw in (("Cu", s["u"]), ("Cv", s["v"])):
            c = raw.transpose(1, 2) * 3.6
            for axis in range(3):
                c = _spline_axis(c, axis)
            out[name] = c
        return out
    if kind == "field":
        s = prepare(case, seed)
        return dict(ftle=_stencil(s["fm"], -10.0, s["dx"], s["dy"]), evec=None, ridge_pts=None,
                    ridge_offsets=None, ridge_counts=None)
    if kind not in ("infer", "train"):
        return None
    s = prepare(case, seed)
    net = {k: [_dev(a).double() for a in v] if isinstance(v, list) else _dev(v).double()
           for k, v in s["net"].state().items()}
    for p in net["W"] + net["b"]:
        p.requires_grad_(kind == "train")

    def forward(inp):
        z = 2 * math.pi * (((inp.double() - net["shift"]) / net["scale"]) @ net["B"])
        h = torch.cat([torch.sin(z), torch.cos(z)], 1)
        for W, b in zip(net["W"][:-1], net["b"][:-1]):
            h = torch.nn.functional.gelu(h @ W + b, approximate="tanh")
        return h @ net["W"][-1] + net["b"][-1]

    if kind == "infer":
        parts = [forward(part) for part in s["inp"].split(1 << 18)]
        return dict(displacement=torch.cat(parts) * s["net"].out_scale.double())
    loss = 0.5 * (forward(s["inp"]) - s["target"].double()).square().sum() / case["batch"]
    loss.backward()
    return dict(loss=loss.detach().reshape(1), gW=[W.grad for W in net["W"]],
                gb=[b.grad for b in net["b"]])
