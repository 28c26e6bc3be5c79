"""The calls that a user of this framework waits for, as measurable cases.

A case is a dict of plain values.  Three kinds:

* ``lattice``  one channel advanced by ``steps`` time steps through
  ``Lattice.run`` (or ``Lattice.run_frames`` with ``frames`` > 0, the output
  interval of a settings file), then read with ``Lattice.macros``;
* ``batch``    many uneven channels advanced together with ``Batch.run``,
  their residuals over the last 100 steps, and every domain's fields: the
  dataset generation and the steady solves of the learned warm start;
* ``predict`` / ``gradient``  the warm-start network, forward on host arrays
  and loss with the gradient of every parameter.

``prepare`` builds what such a program holds between calls (the lattice with
its geometry, the batch, the network and its host arrays); ``run`` is one call.
A lattice keeps its state from call to call, as a solver's loop does.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import portlbm_amd as pa
from portlbm_amd import surrogate

# Arithmetic of one fluid-node update as the reference writes it: 33 for the
# moments, 59 for the equilibria, 27 for the relaxation, rounded up for the
# few terms of boundary nodes.
FLOPS_PER_UPDATE = 120


def _lattice(name, algorithm, layout, storage, scenario, h, v, steps, group, rounding="nearest", frames=0):
    return {"name": name, "kind": "lattice", "algorithm": algorithm, "layout": layout, "storage": storage,
            "rounding": rounding, "scenario": scenario, "h": h, "v": v, "steps": steps, "group": group,
            "frames": frames}


def listed():
    return [
        # the smallest lattice of the parity tests, in short calls: launches and latency
        _lattice("channel 256x64 f64", "nptl", "stream", "f64", "Hagen-Poiseuille", 256, 64, 100, 256),
        # the default settings file: lptl, bundle, 512 x 128, a frame every 10 steps
        _lattice("circle 512x128 f64 frames", "lptl", "bundle", "f64", "circle", 512, 128, 500, 1024, frames=10),
        # the lattice of the benchmark driver and of the steady-state study
        _lattice("porous 1024x256 f64", "nptl", "collision", "f64", "porous-circles", 1024, 256, 1000, 256),
        # the benchmark's default line
        _lattice("porous 8192x2048 f64", "nptl", "collision", "f64", "porous-circles", 8192, 2048, 2000, 256),
        # the reference's float build on the same channel
        _lattice("porous 8192x2048 f32", "lptl", "stream", "f32", "porous-circles", 8192, 2048, 2000, 256),
        # the precision workload: 16-bit storage with stochastic rounding
        _lattice("cylinder 8192x2048 f16", "nptl", "stream", "f16-shifted", "cylinder", 8192, 2048, 2000, 256,
                 rounding="stochastic"),
        # the one-lattice schemes, a size between, and a ragged one
        _lattice("porous 4096x1024 npol f64", "npol", "stream", "f64", "porous-circles", 4096, 1024, 1000, 1024),
        _lattice("porous 3001x997 nsol f32", "nsol", "bundle", "f32", "porous-circles", 3001, 997, 1000, 1024),
        # 16-bit storage rounded to nearest, odd extents
        _lattice("plate 1999x501 bf16", "lptl", "bundle", "bf16-shifted", "plate", 1999, 501, 1000, 256),
        # uneven channels of the dataset generation
        {"name": "batch 96 channels f32", "kind": "batch", "count": 96, "hmin": 64, "hmax": 1024, "vmin": 32,
         "vmax": 256, "steps": 400, "storage": "f32"},
        # warm-start inference on 256 x 256 channels
        {"name": "predict 64x256x256 bf16", "kind": "predict", "h": 256, "v": 256, "batch": 64, "chunk": 32,
         "bf16": True},
        # one training batch of the warm-start network
        {"name": "gradient 16x256x256", "kind": "gradient", "h": 256, "v": 256, "batch": 16},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["lattice", "batch", "predict", "gradient"], [8, 1, 1, 1])[0]
    if kind == "batch":
        return {"kind": "batch", "count": _log_int(rng, 8, 96), "hmin": 64, "hmax": _log_int(rng, 128, 1024),
                "vmin": 32, "vmax": _log_int(rng, 48, 256), "steps": rng.randrange(150, 401),
                "storage": rng.choice(["f32", "f32", "f64"])}
    if kind in ("predict", "gradient"):
        h, v = 16 * rng.randrange(4, 17), 16 * rng.randrange(4, 17)
        if kind == "predict":
            return {"kind": kind, "h": h, "v": v, "batch": rng.randrange(1, 65), "chunk": rng.choice([16, 32]),
                    "bf16": rng.random() < 0.7}
        return {"kind": kind, "h": h, "v": v, "batch": rng.randrange(1, 17)}
    algorithm = rng.choice(["nptl", "nptl", "lptl", "npol", "nsol"])
    storage, rounding = rng.choice([("f64", "nearest"), ("f64", "nearest"), ("f32", "nearest"),
                                    ("f16-shifted", "nearest"), ("f16-shifted", "stochastic"),
                                    ("bf16-shifted", "nearest")])
    h, v = _log_int(rng, 160, 8192), _log_int(rng, 40, 2048)
    most = min(2000, int(1.2e10 / (h * v)))  # at most about a third of the largest listed case
    case = _lattice("", algorithm, rng.choice(["collision", "stream", "bundle"]), storage,
                    rng.choice(["porous-circles", "porous-circles", "Hagen-Poiseuille", "circle", "plate"]), h, v,
                    _log_int(rng, 50, most), rng.choice([256, 1024]), rounding,
                    rng.choice([0, 0, 0, rng.randrange(5, 40)]) if h * v < 300_000 else 0)
    del case["name"]
    return case


def _document(case, seed):
    """The settings document of a lattice case: the seed sets the obstacles,
    the relaxation time and the pressure drop.  The drop keeps the steady
    velocity near or below 0.05 in open channels and between obstacles, so that
    the flow stays in the method's range however long it is advanced."""
    rng = np.random.default_rng(seed)
    tau = float(rng.uniform(0.6, 0.9))
    gap = 30.0 if case["scenario"] == "porous-circles" else float(case["v"])
    drop = 0.05 * 24.0 * case["h"] * (tau - 0.5) / 3.0 / (gap * gap)
    drop = min(0.02, max(drop, 0.005)) if case["scenario"] == "cylinder" else min(0.05, drop)
    drop *= float(rng.uniform(0.8, 1.0))
    ext = {"storage": case["storage"], "rounding": case["rounding"]}
    if case["scenario"] == "porous-circles":
        small = case["v"] < 512
        ext |= {"seed": int(rng.integers(1, 2**62)), "porosity": 0.7, "radiusMin": 2.0 if small else 4.0,
                "radiusMax": 8.0 if small else 16.0, "obstacleMargin": 8 if small else 32, "maxAttempts": 400_000}
    elif case["scenario"] == "cylinder":
        ext |= {"cylinderX": case["h"] // 8, "cylinderRadius": case["v"] / 32.0}
    return pa.settings(case["algorithm"], case["layout"], inner_h=case["h"], inner_v=case["v"],
                       scenario=case["scenario"], work_group_size=case["group"], time_steps=case["steps"], tau=tau,
                       rho_in=1.0 + drop, rho_out=1.0, **ext)


def _documents(case, seed):
    """Uneven porous channels as in workloads.batch_channels; the case sets
    the extents, the seed the rest."""
    sizes, rng = np.random.default_rng(case["count"]), np.random.default_rng(seed)
    docs = []
    for _ in range(case["count"]):
        docs.append(pa.settings("lptl", "stream", inner_h=int(sizes.integers(case["hmin"], case["hmax"] + 1)),
                                inner_v=int(sizes.integers(case["vmin"], case["vmax"] + 1)),
                                scenario="porous-circles", time_steps=case["steps"],
                                tau=float(rng.uniform(0.55, 1.0)), rho_in=float(rng.uniform(1.005, 1.05)),
                                rho_out=1.0, storage=case["storage"], seed=int(rng.integers(1, 2**62)),
                                porosity=float(rng.uniform(0.5, 0.9)), radiusMin=2.0, radiusMax=8.0,
                                obstacleMargin=8, maxAttempts=20000))
    return docs


def _network_inputs(case, seed):
    """Feature maps of seeded channels (a fluid mask of discs, the ramp and
    the two scalars), smooth targets, and weights of the network's scale."""
    rng = np.random.default_rng(seed)
    ny, nx = case["v"], case["h"]
    yy, xx = np.mgrid[0:ny, 0:nx]
    x = np.empty((case["batch"], surrogate.INPUTS, ny, nx), dtype=np.float32)
    t = np.empty((case["batch"], surrogate.OUTPUTS, ny, nx), dtype=np.float32)
    for b in range(case["batch"]):
        mask = np.ones((ny, nx), dtype=bool)
        mask[0] = mask[-1] = False
        for _ in range(max(1, ny * nx // 400)):
            r, cx, cy = rng.uniform(2, 8), rng.integers(8, nx - 8), rng.integers(2, ny - 2)
            y0, y1, x0, x1 = max(0, cy - 8), cy + 9, max(0, cx - 8), cx + 9
            mask[y0:y1, x0:x1] &= (xx[y0:y1, x0:x1] - cx) ** 2 + (yy[y0:y1, x0:x1] - cy) ** 2 > r * r
        x[b] = surrogate.features(mask, float(rng.uniform(0.55, 0.9)), 1.0 + float(rng.uniform(0.01, 0.05)), 1.0)
        a, p = rng.uniform(0.5, 2.0, surrogate.OUTPUTS), rng.uniform(0.0, 6.0, surrogate.OUTPUTS)
        for k in range(surrogate.OUTPUTS):
            t[b, k] = np.where(mask, np.sin(a[k] * xx / 40.0 + p[k]) * np.cos(yy / 30.0), 0.0)
    return x, t, int(rng.integers(1, 2**62))


def prepare(case, seed):
    if case["kind"] == "lattice":
        return case, pa.Lattice.from_settings(_document(case, seed))
    if case["kind"] == "batch":
        return case, pa.Batch(_documents(case, seed), storage=case["storage"])
    x, t, weights = _network_inputs(case, seed)
    net = surrogate.Surrogate(case["v"], case["h"], case.get("chunk", case["batch"]))
    net.init_params(weights)
    return case, net, x, t


def run(state):
    case = state[0]
    if case["kind"] == "lattice":
        lattice = state[1]
        if case["frames"]:
            lattice.run_frames(case["steps"], case["frames"])
            return {"fields": lattice.macros(), "frame": lattice.frame()[1]}
        lattice.run(case["steps"])
        return {"fields": lattice.macros()}
    if case["kind"] == "batch":
        batch = state[1]
        batch.run(case["steps"] - 100, "graph")
        batch.residuals()
        batch.run(100, "graph")
        residuals = batch.residuals()
        fields = [batch.macros(d) for d in range(case["count"])]
        return {"residuals": residuals, "fields": [np.concatenate([f[k] for f in fields]) for k in range(4)]}
    _, net, x, t = state
    if case["kind"] == "predict":
        return net.predict(x, bf16=case["bf16"])
    loss, grad = net.loss_grad(x, t)
    return {"loss": loss, "gradient": grad}


_CHANNELS = (4, 16, 16, 32, 32, 48, 48, 64, 64, 64, 48, 32, 16, 16, 3)


def _convolution_macs(h, v):
    """Multiply-adds of one forward pass over one sample."""
    level = (0, 0, 1, 1, 2, 2, 3, 3, 4, 3, 2, 1, 0, 0)
    return sum(9 * _CHANNELS[k] * _CHANNELS[k + 1] * (h >> lv) * (v >> lv) for k, lv in enumerate(level))


def work(case):
    """One call's state read once and written once with its results, and its
    arithmetic.  (Taking a lattice through HBM at every step, as a one-step
    kernel has to, moves ``steps`` times the state; the call does not need it.)"""
    if case["kind"] == "lattice":
        nodes, size = case["h"] * case["v"], pa.STORAGE_BYTES[case["storage"]]
        frames = case["steps"] // case["frames"] if case["frames"] else 0
        return {"bytes": nodes * (18.0 * size + 2.0 + 32.0 * (1 + frames)),
                "flops": float(FLOPS_PER_UPDATE) * nodes * case["steps"]}
    if case["kind"] == "batch":
        nodes = case["count"] * (case["hmin"] + case["hmax"]) * (case["vmin"] + case["vmax"]) / 4.0
        return {"bytes": nodes * (18.0 * pa.STORAGE_BYTES[case["storage"]] + 2.0 + 32.0),
                "flops": float(FLOPS_PER_UPDATE) * nodes * case["steps"]}
    pixels, macs = float(case["batch"] * case["h"] * case["v"]), case["batch"] * _convolution_macs(case["h"], case["v"])
    if case["kind"] == "predict":
        return {"bytes": 28.0 * pixels, "flops": 2.0 * macs}
    return {"bytes": 28.0 * pixels, "flops": 6.0 * macs}


# ---------------------------------------------------------------------------
# the same results in 64 bits, in plain torch
# ---------------------------------------------------------------------------
_CX = [d % 3 - 1 for d in range(9)]
_CY = [d // 3 - 1 for d in range(9)]
_W = [1 / 36, 1 / 9, 1 / 36, 1 / 9, 4 / 9, 1 / 9, 1 / 36, 1 / 9, 1 / 36]


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


class _Channels:
    """Several channels side by side in one padded FP64 array [domain, y, x],
    advanced by pull streaming with half-way bounce-back, the Zou-He pressure
    outlet and BGK collision.  A geometry is 0 fluid, 1 solid, -1 ghost."""

    def __init__(self, docs):
        dev = _device()
        sizes = [(d["domain"]["verticalNodes"] + 2, d["domain"]["horizontalNodes"] + 2) for d in docs]
        V, H = max(s[0] for s in sizes), max(s[1] for s in sizes)
        B = len(docs)
        phase = np.ones((B, V, H), dtype=np.int8)
        rho_in, rho_out, omega = (np.empty(B) for _ in range(3))
        f = np.empty((9, B, V, H))
        for d in range(9):
            f[d] = _W[d]
        out, source = np.zeros((B, V, H), dtype=bool), np.zeros((B, V, H), dtype=bool)
        for b, (doc, (v, h)) in enumerate(zip(docs, sizes)):
            linear = {**doc, "algorithmic": {**doc["algorithmic"], "algorithm": "lptl"}}
            phase[b, :v, :h] = pa.build_phase(linear).reshape(v, h)
            physical = doc["physical"]
            rho_in[b], rho_out[b] = physical["inletDensity"], physical["outletDensity"]
            omega[b] = 1.0 / physical["relaxationTime"]
            for d in range(9):
                f[d, b, 1:v - 1, 0] = _W[d] * rho_in[b]
                f[d, b, 1:v - 1, h - 1] = _W[d] * rho_out[b]
            out[b, 2:v - 2, h - 2] = True
            source[b, 2:v - 2, h - 3] = True
        self.sizes, self.B = sizes, B
        self.f = torch.from_numpy(f).to(dev)
        ph = torch.from_numpy(phase).to(dev)
        self.fluid = ph == 0
        solid = ph == 1
        self.bounce = [torch.roll(solid, (_CY[d], _CX[d]), (1, 2)) for d in range(9)]
        self.bounce[4] = torch.zeros_like(solid)
        at = (torch.from_numpy(out).to(dev) & self.fluid).nonzero(as_tuple=True)
        self.out = at
        self.left = (at[0], at[1], at[2] - 1)
        self.known = (torch.from_numpy(source).to(dev) & self.fluid)[self.left]
        self.uy = torch.zeros(at[0].shape[0], dtype=torch.float64, device=dev)
        self.rho_out = torch.from_numpy(rho_out).to(dev)[at[0]]
        self.omega = torch.from_numpy(omega).to(dev).view(B, 1, 1)

    def step(self):
        """One step; the density and momentum that its collision works with."""
        f = self.f
        g = [torch.where(self.bounce[d], f[8 - d], torch.roll(f[d], (_CY[d], _CX[d]), (1, 2))) if d != 4 else f[4]
             for d in range(9)]
        e = [v[self.out] for v in g]
        jx = e[1] + e[4] + e[7] + 2.0 * (e[2] + e[5] + e[8]) - self.rho_out
        g[0][self.out] = e[8] - 0.5 * (e[1] - e[7]) - jx / 6.0 - 0.5 * self.uy
        g[3][self.out] = e[5] - 2.0 / 3.0 * jx
        g[6][self.out] = e[2] + 0.5 * (e[1] - e[7]) - jx / 6.0 + 0.5 * self.uy
        jx = (g[2] + g[5] + g[8]) - (g[0] + g[3] + g[6])
        jy = (g[6] + g[7] + g[8]) - (g[0] + g[1] + g[2])
        rho = sum(g[1:], g[0].clone())
        self.uy = torch.where(self.known, jy[self.left], self.uy)
        rest = rho - 1.5 * (jx * jx + jy * jy)
        new = torch.empty_like(f)
        for d in range(9):
            cu = _CX[d] * jx + _CY[d] * jy
            eq = (rest + 3.0 * cu).addcmul_(cu, cu, value=4.5).mul_(_W[d])
            new[d] = torch.where(self.fluid, g[d] + self.omega * (eq - g[d]), f[d])
        self.f = new
        return rho, jx, jy

    def fields(self, rho, jx, jy):
        """The four results of every domain's inner nodes; a node that is not
        fluid keeps density -1 at rest."""
        rho = torch.where(self.fluid, rho, -1.0)
        jx, jy = (torch.where(self.fluid, j, 0.0) for j in (jx, jy))
        four = (rho, jx, jy, torch.sqrt(jx * jx + jy * jy))
        return [torch.cat([a[b, 1:v - 1, 1:h - 1].reshape(-1) for b, (v, h) in enumerate(self.sizes)]).cpu()
                for a in four]

    def momentum(self):
        jx = sum(_CX[d] * self.f[d] for d in range(9) if _CX[d])
        jy = sum(_CY[d] * self.f[d] for d in range(9) if _CY[d])
        return torch.where(self.fluid, jx, 0.0), torch.where(self.fluid, jy, 0.0)


def _conv(x, w, b):
    n, c, h, wd = x.shape
    xp = torch.nn.functional.pad(x, (1, 1, 1, 1))
    y = b.view(1, -1, 1, 1).expand(n, -1, h, wd).reshape(n, -1, h * wd)
    for k in range(9):
        y = y + w[:, :, k // 3, k % 3] @ xp[:, :, k // 3:k // 3 + h, k % 3:k % 3 + wd].reshape(n, c, h * wd)
    return y.view(n, -1, h, wd)


def _network(x, params):
    """The encoder-decoder of the warm start on FP64 tensors."""
    at, convs = 0, []
    for k in range(14):
        ci, co = _CHANNELS[k], _CHANNELS[k + 1]
        w = params[at:at + 9 * ci * co].view(co, ci, 3, 3)
        convs.append((w, params[at + 9 * ci * co:at + 9 * ci * co + co]))
        at += 9 * ci * co + co
    relu, pool = torch.relu, lambda a: torch.nn.functional.avg_pool2d(a, 2)
    skips = []
    a = x
    for level in range(4):
        a = relu(_conv(a, *convs[2 * level]))
        a = relu(_conv(a, *convs[2 * level + 1]))
        skips.append(a)
        a = pool(a)
    a = relu(_conv(a, *convs[8]))
    for m in range(4):
        a = a.repeat_interleave(2, 2).repeat_interleave(2, 3) + skips[3 - m]
        a = relu(_conv(a, *convs[9 + m]))
    return _conv(a, *convs[13])


def exact(case, seed):
    if case["kind"] == "lattice":
        if float(case["h"]) * case["v"] * case["steps"] > 8e9:
            return None
        channel = _Channels([_document(case, seed)])
        found = {}
        for i in range(case["steps"]):
            macros = channel.step()
            if case["frames"] and i % case["frames"] == case["frames"] - 1 and i + case["frames"] >= case["steps"]:
                found["frame"] = channel.fields(*macros)
        found["fields"] = channel.fields(*macros)
        if pa.STORAGE_BYTES[case["storage"]] == 2:  # its momentum is only as good as 16 bits hold it
            found = {k: [v[0], None, None, None] for k, v in found.items()}
        return found
    if case["kind"] == "batch":
        if float(case["count"]) * case["hmax"] * case["vmax"] * case["steps"] > 1.2e10:
            return None
        channels = _Channels(_documents(case, seed))
        for i in range(case["steps"]):
            if i == case["steps"] - 100:
                x0, y0 = channels.momentum()
            macros = channels.step()
        x1, y1 = channels.momentum()
        change = ((x1 - x0) ** 2 + (y1 - y0) ** 2).sum((1, 2)) / (x1 * x1 + y1 * y1).sum((1, 2))
        return {"residuals": torch.sqrt(change).cpu(), "fields": channels.fields(*macros)}
    x, t, weights = _network_inputs(case, seed)
    with surrogate.Surrogate(16, 16, 1) as net:  # the seeded initial weights, an input here
        net.init_params(weights)
        params = torch.from_numpy(net.params()).to(_device(), torch.float64)
    chunk = max(1, int(2e6 / (case["h"] * case["v"])))
    if case["kind"] == "predict":
        with torch.no_grad():
            return torch.cat([_network(torch.from_numpy(x[b:b + chunk]).to(_device(), torch.float64), params).cpu()
                              for b in range(0, case["batch"], chunk)])
    params.requires_grad_(True)
    norm, loss = 3.0 * float(x[:, 0].astype(np.float64).sum()), 0.0
    for b in range(0, case["batch"], 4):
        xb, tb = (torch.from_numpy(a[b:b + 4]).to(_device(), torch.float64) for a in (x, t))
        part = (xb[:, :1] * (_network(xb, params) - tb) ** 2).sum() / norm
        part.backward()
        loss += float(part.detach())
    return {"loss": loss, "gradient": params.grad.cpu()}
