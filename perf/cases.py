"""Timed cases: what a program does with this framework, through its public calls.

A case is one pass of one such program: an interactive frame, a channel run that
ends with its fields, a large grid advanced between two looks at it, a batch of
domains stepped and collected, a training step's gradients, a network
prediction, a surrogate rollout, an FP64 run.  ``prepare`` makes what the
program has in hand (grid, obstacles, tuned variant, weights, host inputs),
``run`` is one pass, ``exact`` the same pass in 64 bits with torch alone.
"""
import math
import os
import random

import numpy as np
import torch
import torch.nn.functional as F

import lbm_amd
from lbm_amd import LBM, LBM64, Batch
from lbm_amd.surrogate import UNet, load_params

PRECISION = {"f32": lbm_amd.PRECISION_F32, "f16s": lbm_amd.PRECISION_F16S, "f16e": lbm_amd.PRECISION_F16E}
BOUNDARY = {"reference": lbm_amd.BOUNDARY_REFERENCE, "zero_gradient": lbm_amd.BOUNDARY_ZERO_GRADIENT}
WEIGHTS = os.path.join(os.path.dirname(os.path.abspath(lbm_amd.__file__)), "data", "surrogate_f2.npy")


# ---- the cases ------------------------------------------------------------------------

def grid(name, nx, ny, steps, read, precision="f32", boundary="reference", tau=0.6, u=0.05, circles=12, r_min=8,
         r_max=32, tune=True):
    return {"name": name, "kind": "grid", "nx": nx, "ny": ny, "steps": steps, "read": read, "precision": precision,
            "boundary": boundary, "tau": tau, "u": u, "circles": circles, "r_min": r_min, "r_max": r_max,
            "tune": tune}


def listed():
    return [
        # one frame of the interactive program: 15 steps, then the coloured curl (the reference's default canvas)
        grid("frame_640x360", 640, 360, 15, "render", tau=0.56, u=0.1, tune=False),
        # the plain channel run around one cylinder, 2000 steps from rest to its fields, as the driver script runs it
        grid("channel_400x160", 400, 160, 2000, "fields", tau=0.56, u=0.1, circles=1, r_min=16, r_max=16,
             tune=False),
        # a ragged size with the other outlet and the storage made for accuracy, tuned once by its program
        grid("ragged_f16e_1021x777", 1021, 777, 200, "ux", precision="f16e", boundary="zero_gradient"),
        # the obstacle channels the framework is benchmarked on, advanced between two looks at a field
        grid("f32_4096x2048", 4096, 2048, 200, "curl", circles=200, r_max=64),
        grid("f32_8192x4096", 8192, 4096, 300, "curl", circles=200, r_max=64),
        grid("f16s_8192x4096", 8192, 4096, 300, "ux", precision="f16s", circles=200, r_max=64),
        # a parameter study: domains of uneven size, obstacles, viscosity and inflow, tuned, then all fields collected
        {"name": "batch_128", "kind": "batch", "domains": 128, "layout": 1, "size": 0, "steps": 200,
         "precision": "f32", "tune": True},
        # snapshot pairs for training: square domains stepped one jump (64 steps) and read, as the trainer does
        {"name": "pairs_24x512", "kind": "batch", "domains": 24, "layout": 2, "size": 512, "steps": 64,
         "precision": "f32", "tune": False},
        # loss and gradients of the surrogate for one minibatch of the trainer
        {"name": "gradients_8x256x256", "kind": "gradients", "batch": 8, "height": 256, "width": 256},
        # one prediction of the surrogate from host fields, at the size of a half-resolution rollout
        {"name": "predict_256x512", "kind": "predict", "batch": 1, "height": 256, "width": 512},
        # surrogate rollout: cycles of a 64-step jump and 8 corrector steps, then the fields
        {"name": "rollout_1024x512", "kind": "rollout", "nx": 1024, "ny": 512, "cycles": 10, "tau": 0.6, "u": 0.05},
        # the FP64 solver that errors are measured against
        {"name": "f64_2048x1024", "kind": "f64", "nx": 2048, "ny": 1024, "steps": 100, "tau": 0.6, "u": 0.05,
         "circles": 40},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["frame", "channel", "grid", "grid", "grid", "batch", "pairs", "gradients", "predict", "rollout",
                       "f64"])
    tau, u = round(rng.uniform(0.56, 0.8), 4), round(rng.uniform(0.02, 0.06), 4)
    if kind == "frame":
        return _drop(grid("", _log(rng, 320, 1280), _log(rng, 180, 720), 15, "render", tau=tau, u=u, tune=False))
    if kind == "channel":
        return _drop(grid("", _log(rng, 200, 1200), _log(rng, 80, 480), rng.randrange(200, 2001), "fields", tau=tau,
                          u=u, circles=1, r_min=8, r_max=16, tune=False))
    if kind == "grid":
        precision = rng.choice(["f32", "f16s", "f16e"])
        nx, ny = _log(rng, 700, 8192), _log(rng, 500, 4096)
        return _drop(grid("", nx, ny, rng.randrange(50, 251), "curl" if precision == "f32" else "ux",
                          precision=precision, boundary=rng.choice(["reference", "zero_gradient"]), tau=tau, u=u,
                          circles=max(4, nx * ny // 170000), r_max=48))
    if kind == "batch":
        return {"kind": "batch", "domains": _log(rng, 6, 128), "layout": rng.randrange(1 << 20), "size": 0,
                "steps": rng.randrange(50, 201), "precision": rng.choice(["f32", "f16s", "f16e"]), "tune": True}
    if kind == "pairs":
        return {"kind": "batch", "domains": rng.randrange(8, 25), "layout": rng.randrange(1 << 20),
                "size": rng.choice([256, 384, 512]), "steps": 64, "precision": "f32", "tune": False}
    if kind == "gradients":
        return {"kind": "gradients", "batch": rng.randrange(1, 9), "height": 8 * rng.randrange(8, 33), "width": 256}
    if kind == "predict":
        return {"kind": "predict", "batch": rng.randrange(1, 5), "height": 8 * rng.randrange(8, 33),
                "width": rng.choice([256, 512])}
    if kind == "rollout":
        return {"kind": "rollout", "nx": rng.choice([512, 1024]), "ny": 16 * rng.randrange(8, 33),
                "cycles": rng.randrange(2, 11), "tau": tau, "u": u}
    return {"kind": "f64", "nx": _log(rng, 300, 2048), "ny": _log(rng, 150, 1024), "steps": rng.randrange(20, 101),
            "tau": tau, "u": u, "circles": 10}


def _drop(case):
    return {k: v for k, v in case.items() if k != "name"}


# ---- inputs -----------------------------------------------------------------------------

def obstacles(nx, ny, seed, count, r_min, r_max):
    """Channel walls and `count` random circles clear of the inlet, u8 (ny, nx), 1 = solid."""
    rng = np.random.default_rng([seed, nx, ny])
    mask = np.zeros((ny, nx), np.uint8)
    mask[0] = mask[-1] = 1
    for _ in range(count):
        r = int(rng.integers(r_min, r_max + 1))
        cx, cy = int(rng.integers(2 * r + 2, nx - r)), int(rng.integers(r, ny - r))
        y, x = np.ogrid[-r:r + 1, -r:r + 1]
        mask[cy - r:cy + r + 1, cx - r:cx + r + 1] |= (x * x + y * y <= r * r).astype(np.uint8)
    return mask


def domains(case):
    """(nx, ny, omega, u_in) of a batch: multiples of 32 from 128 x 64 to 1024 x 512, or all of one size."""
    rng, out = random.Random(case["layout"]), []
    for _ in range(case["domains"]):
        nx, ny = 128 + 32 * rng.randrange(29), 64 + 32 * rng.randrange(15)
        if case["size"]:
            nx = ny = case["size"]
        out.append((nx, ny, 1.0 / rng.uniform(0.56, 0.8), rng.uniform(0.02, 0.06)))
    return out


def domain_mask(case, i, nx, ny, seed):
    return obstacles(nx, ny, 1000 * seed + i, 1 + (seed + i) % 12, 4, max(5, min(nx, ny) // 12))


def grid_mask(case, seed):
    return obstacles(case["nx"], case["ny"], seed, case["circles"], case["r_min"], case["r_max"])


def rollout_mask(case, seed):
    return obstacles(case["nx"], case["ny"], seed, 12, 8, 32)


def net_inputs(case, seed):
    """Network input (B, H, W, 8), targets (B, H, W, 3) and loss weights (B, H, W): smooth fields around obstacles."""
    b, h, w = case["batch"], case["height"], case["width"]
    rng = np.random.default_rng([seed, b, h, w])
    y, x = np.mgrid[0:h, 0:w].astype(np.float32)

    def field(scale):
        f = np.zeros((h, w), np.float32)
        for k in range(1, 5):
            a, p, q, s = rng.normal() / k, *rng.uniform(-k, k, 2), rng.uniform(0, 2 * np.pi)
            f += np.float32(a) * np.sin(np.float32(2 * np.pi) * (np.float32(p) * x / w + np.float32(q) * y / h)
                                        + np.float32(s))
        return np.float32(scale) * f

    xs, ys = np.zeros((b, h, w, 8), np.float32), np.zeros((b, h, w, 3), np.float32)
    ws = np.zeros((b, h, w), np.float32)
    for i in range(b):
        fluid = 1.0 - obstacles(w, h, 100 * seed + i, 8, 3, 12).astype(np.float32)
        tau, u = rng.uniform(0.52, 0.8), rng.uniform(0.02, 0.1)
        xs[i, ..., 0] = 1.0 - fluid
        for c, (mean, scale) in enumerate(((0.0, 0.2), (10.0 * u, 0.05), (0.0, 0.05))):
            xs[i, ..., 1 + c] = (np.float32(mean) + field(scale)) * fluid
        xs[i, ..., 4], xs[i, ..., 5] = (tau - 0.5) / 0.2, 10.0 * u
        for c in range(3):
            ys[i, ..., c] = field(0.5) * fluid
        ws[i] = fluid
    return xs, ys, ws


# ---- one pass -----------------------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind == "grid":
        g = LBM(1.0 / case["tau"], case["nx"], case["ny"], precision=PRECISION[case["precision"]],
                boundary=BOUNDARY[case["boundary"]])
        g.mask = grid_mask(case, seed)
        g.custom_speed(case["u"])
        if case["tune"]:
            g.autotune(20)
        return {"case": case, "grid": g}
    if kind == "batch":
        doms = domains(case)
        b = Batch(doms, precision=PRECISION[case["precision"]])
        for i, (nx, ny, _, _) in enumerate(doms):
            b.set_mask(i, domain_mask(case, i, nx, ny, seed))
        if case["tune"]:
            b.autotune(6)
        return {"case": case, "batch": b, "fields": np.zeros((3, sum(d[0] * d[1] for d in doms)), np.float32)}
    if kind in ("gradients", "predict"):
        net = UNet(case["batch"], case["height"], case["width"])
        net.set_params(load_params(WEIGHTS))
        return {"case": case, "net": net, "inputs": net_inputs(case, seed)}
    if kind == "rollout":
        g = LBM(1.0 / case["tau"], case["nx"], case["ny"])
        g.mask = rollout_mask(case, seed)
        g.custom_speed(case["u"])
        g.autotune(20)
        net = UNet(1, case["ny"] // 2, case["nx"] // 2)
        net.set_params(load_params(WEIGHTS))
        return {"case": case, "grid": g, "net": net}
    s = LBM64(1.0 / case["tau"], case["nx"], case["ny"], case["u"])
    s.set_mask(obstacles(case["nx"], case["ny"], seed, case["circles"], 6, 24))
    return {"case": case, "solver": s}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "grid":
        g = state["grid"]
        g.step(case["steps"])
        if case["read"] == "render":
            return g.render()
        if case["read"] == "fields":
            return g.fields()
        return g.calculate_summary(lbm_amd.SummaryStat.Curl if case["read"] == "curl" else lbm_amd.SummaryStat.Ux)
    if kind == "batch":
        b, out, at = state["batch"], state["fields"], 0
        b.step(case["steps"])
        for i, (nx, ny, _, _) in enumerate(b.domains):
            for c, plane in enumerate(b.moments(i)):
                out[c, at:at + nx * ny] = plane.ravel()
            at += nx * ny
        return out
    if kind == "gradients":
        return state["net"].loss_grad(*state["inputs"])
    if kind == "predict":
        return state["net"].forward(state["inputs"][0])
    if kind == "rollout":
        g = state["grid"]
        for _ in range(case["cycles"]):
            g.surrogate_jump(state["net"])
            g.step(8)
        return g.fields()
    state["solver"].step(case["steps"])
    return state["solver"].macro()


# ---- what a pass cannot do without ---------------------------------------------------------

COLLIDE_FLOPS = 117  # one BGK update of nine populations, common terms computed once
NET_LAYERS = [(9, 32, 32, 0), (9, 32, 32, 0), (9, 32, 64, 1), (9, 64, 64, 1), (9, 64, 128, 2), (9, 128, 128, 2),
              (9, 128, 256, 3), (9, 256, 256, 3), (1, 256, 128, 3), (9, 256, 128, 2), (9, 128, 128, 2),
              (1, 128, 64, 2), (9, 128, 64, 1), (9, 64, 64, 1), (1, 64, 32, 1), (9, 64, 32, 0), (9, 32, 32, 0),
              (1, 32, 32, 0)]  # taps, inputs, outputs, level (resolution halved per level)


def net_flops(batch, h, w):
    return sum(2.0 * t * ci * co * batch * (h >> lv) * (w >> lv) for t, ci, co, lv in NET_LAYERS)


def work(case):
    """Inputs read once, outputs written once; the arithmetic of every step."""
    kind = case["kind"]
    if kind in ("grid", "f64"):
        cells = case["nx"] * case["ny"]
        size = 8 if kind == "f64" else 4 if case["precision"] == "f32" else 2
        planes = {"render": 12, "fields": 16}.get(case.get("read"), 4) if kind == "grid" else 24
        return {"bytes": cells * (18.0 * size + 1 + planes), "flops": 1.0 * COLLIDE_FLOPS * cells * case["steps"]}
    if kind == "batch":
        cells = sum(d[0] * d[1] for d in domains(case))
        return {"bytes": cells * (18.0 * (4 if case["precision"] == "f32" else 2) + 1 + 12),
                "flops": 1.0 * COLLIDE_FLOPS * cells * case["steps"]}
    params = sum(t * ci * co + co for t, ci, co, _ in NET_LAYERS)
    if kind == "rollout":
        cells = case["nx"] * case["ny"]
        return {"bytes": cells * (18.0 * 4 + 1 + 16) + 2.0 * params,
                "flops": case["cycles"] * (net_flops(1, case["ny"] // 2, case["nx"] // 2)
                                           + 8.0 * COLLIDE_FLOPS * cells)}
    pixels = case["batch"] * case["height"] * case["width"]
    flops = net_flops(case["batch"], case["height"], case["width"])
    if kind == "predict":
        return {"bytes": 44.0 * pixels + 2.0 * params, "flops": flops}
    return {"bytes": 48.0 * pixels + 6.0 * params, "flops": 3.0 * flops}


# ---- the same passes in 64 bits ---------------------------------------------------------------

CX = [-1, 0, 1, -1, 0, 1, -1, 0, 1]
CY = [-1, -1, -1, 0, 0, 0, 1, 1, 1]  # rows grow southwards
W9 = [1 / 36, 1 / 9, 1 / 36, 1 / 9, 4 / 9, 1 / 9, 1 / 36, 1 / 9, 1 / 36]


class Exact:
    """D2Q9 in float64: collide, then pull with half-way bounce-back; solid cells, column 0 and the last row are
    not streamed and keep the inflow equilibrium they start from."""

    def __init__(self, mask, omega, u, boundary="reference"):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.c = torch.tensor([CX, CY], dtype=torch.float64, device=self.dev)
        self.w = torch.tensor(W9, dtype=torch.float64, device=self.dev)[:, None]
        solid = torch.from_numpy(mask.astype(bool)).to(self.dev)
        ny, nx = mask.shape
        n = nx * ny
        self.nx, self.ny, self.n, self.omega, self.solid = nx, ny, n, omega, solid
        y, x = torch.meshgrid(torch.arange(ny, device=self.dev), torch.arange(nx, device=self.dev), indexing="ij")
        self.streamed = (~solid & (x > 0) & (y < ny - 1)).reshape(-1)
        own = y * nx + x
        self.source = torch.empty((9, n), dtype=torch.int32 if 9 * n < 2 ** 31 else torch.int64, device=self.dev)
        for k in range(9):
            ux, uy = x - CX[k], y - CY[k]
            past = ux >= nx
            if boundary == "reference":  # the flattened index wraps to the next row
                ux, uy = torch.where(past, 0, ux), torch.where(past, uy + 1, uy)
            else:
                ux = torch.where(past, nx - 1, ux)
            out = (ux < 0) | (uy < 0) | (uy >= ny)
            up = uy.clamp(0, ny - 1) * nx + ux.clamp(0, nx - 1)
            bounce = out | solid.reshape(-1)[up]
            self.source[k] = torch.where(bounce, (8 - k) * n + own, k * n + up).reshape(-1)
        one = torch.ones((1, 1), dtype=torch.float64, device=self.dev)
        self.start = self.equilibrium(one, u * one, 0 * one).reshape(9, 1)
        self.f = self.start.repeat(1, n)

    def equilibrium(self, rho, ux, uy):
        """uy in rows (southwards)."""
        cu = self.c[0][:, None] * ux + self.c[1][:, None] * uy
        return self.w * rho * (1 + 3 * cu + 4.5 * cu * cu - 1.5 * (ux * ux + uy * uy))

    def moments(self):
        """rho, jx and jy (north-positive)."""
        rho, j = self.f.sum(0), self.c @ self.f
        return rho, j[0], -j[1]

    def step(self, steps):
        for _ in range(steps):
            rho, j = self.f.sum(0), self.c @ self.f
            self.lagged = (rho, j[0], -j[1])
            g = self.f + self.omega * (self.equilibrium(rho, j[0] / rho, j[1] / rho) - self.f)
            pulled = torch.take(g, self.source) if self.source.dtype == torch.int64 else \
                g.reshape(-1).index_select(0, self.source.reshape(-1)).reshape(9, -1)
            self.f = torch.where(self.streamed, pulled, self.start)

    def plane(self, v):
        return v.reshape(self.ny, self.nx)

    def curl(self, rho, jx, jy):
        """10 (jy east - jy west - jx north + jx south) / rho; 0 in column 0 and the last row."""
        def shifted(v, by):
            v = torch.cat([torch.zeros(self.nx, dtype=v.dtype, device=v.device), v,
                           torch.zeros(self.nx, dtype=v.dtype, device=v.device)])
            return v[self.nx + by:self.nx + by + self.n]
        c = 10 * (shifted(jy, 1) - shifted(jy, -1) - shifted(jx, -self.nx) + shifted(jx, self.nx)) / rho
        c = self.plane(c).clone()
        c[:, 0] = 0
        c[-1] = 0
        return c

    def fields(self):
        rho, jx, jy = self.moments()
        return tuple(self.plane(v) for v in (rho, jx / rho, jy / rho)) + (self.curl(rho, jx, jy),)

    def render(self):
        """The lagged curl through the nine-colour map, solid cells black."""
        table = torch.tensor([[0, 0, .5], [0, 0, 1], [0, .5, 1], [0, 1, 1], [.5, 1, .5], [1, 1, 0], [1, .5, 0],
                              [1, 0, 0], [.5, 0, 0]], dtype=torch.float64, device=self.dev)
        c = (20 * self.curl(*self.lagged)).clamp(-4, 4)
        b = c.floor().clamp(-4, 3)
        part = (c - b)[..., None]
        at = (b + 4).long()
        return torch.where(self.solid[..., None], 0.0, (1 - part) * table[at] + part * table[at + 1])


class ExactNet:
    """The surrogate in float64 (NHWC): 3x3 convolutions as nine shifted products, bf16-valued weights."""

    def __init__(self, params, grads=False):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.p = torch.from_numpy(params.astype(np.float64)).to(dev).requires_grad_(grads)
        self.layers, at = [], 0
        for taps, ci, co, _ in NET_LAYERS:
            self.layers.append((taps, self.p[at:at + taps * ci * co].reshape(taps, co, ci),
                                self.p[at + taps * ci * co:at + taps * ci * co + co]))
            at += taps * ci * co + co

    def conv(self, i, x):
        taps, w, b = self.layers[i]
        if taps == 1:
            y = x @ w[0].T + b
        else:
            h, wd = x.shape[1:3]
            pad = F.pad(x, (0, 0, 1, 1, 1, 1))
            y = b
            for t in range(9):
                y = y + pad[:, t // 3:t // 3 + h, t % 3:t % 3 + wd] @ w[t].T
        return y if i == len(self.layers) - 1 else torch.relu(y)

    @staticmethod
    def pool(x):
        b, h, w, c = x.shape
        return x.reshape(b, h // 2, 2, w // 2, 2, c).mean((2, 4))

    @staticmethod
    def up(x):
        return x.repeat_interleave(2, 1).repeat_interleave(2, 2)

    def __call__(self, x):
        x = F.pad(x, (0, 32 - x.shape[-1]))
        e1 = self.conv(1, self.conv(0, x))
        e2 = self.conv(3, self.conv(2, self.pool(e1)))
        e3 = self.conv(5, self.conv(4, self.pool(e2)))
        e4 = self.conv(7, self.conv(6, self.pool(e3)))
        d3 = self.conv(10, self.conv(9, torch.cat([self.up(self.conv(8, e4)), e3], -1)))
        d2 = self.conv(13, self.conv(12, torch.cat([self.up(self.conv(11, d3)), e2], -1)))
        d1 = self.conv(16, self.conv(15, torch.cat([self.up(self.conv(14, d2)), e1], -1)))
        return self.conv(17, d1)[..., :3]


def _jump(g, net, u):
    """One surrogate jump of an Exact grid with a half-resolution network."""
    rho, jx, jy = (g.plane(v) for v in g.moments())
    fluid = (~g.solid).double()

    def blocks(v):
        return v.reshape(g.ny // 2, 2, g.nx // 2, 2).sum((1, 3))
    count = blocks(fluid)
    some = count > 0

    def mean(v):
        return blocks(v * fluid) / count.clamp(min=1)
    x = torch.stack([1 - count / 4, torch.where(some, (mean(rho) - 1) / 0.01, 0.0), mean(jx / rho) / 0.1,
                     mean(jy / rho) / 0.1, torch.full_like(count, (1 / g.omega - 0.5) * 5),
                     torch.full_like(count, u / 0.1)], -1)
    change = net(x[None]).permute(0, 3, 1, 2)
    d = F.interpolate(change, scale_factor=2, mode="bilinear", align_corners=False)[0].reshape(3, -1)
    rho, ux, uy = rho.reshape(-1), (jx / rho).reshape(-1), (jy / rho).reshape(-1)
    feq = g.equilibrium(rho + 0.01 * d[0], ux + 0.003 * d[1], -(uy + 0.003 * d[2]))
    g.f = torch.where(g.streamed, feq, g.f)


def exact(case, seed):
    kind = case["kind"]
    if kind == "grid":
        g = Exact(grid_mask(case, seed), 1.0 / case["tau"], case["u"], case["boundary"])
        g.step(case["steps"])
        if case["read"] == "render":
            return g.render()
        if case["read"] == "fields":
            return g.fields()
        return g.curl(*g.lagged) if case["read"] == "curl" else g.plane(g.lagged[1])
    if kind == "batch":
        planes = [[], [], []]
        for i, (nx, ny, omega, u) in enumerate(domains(case)):
            g = Exact(domain_mask(case, i, nx, ny, seed), omega, u)
            g.step(case["steps"])
            rho, jx, jy = g.lagged
            for p, v in zip(planes, (jx, jy, rho)):
                p.append(v.reshape(-1))
        return torch.stack([torch.cat(p) for p in planes])
    if kind == "f64":
        g = Exact(obstacles(case["nx"], case["ny"], seed, case["circles"], 6, 24), 1.0 / case["tau"], case["u"])
        g.step(case["steps"])
        return g.fields()[:3]
    params = load_bf16(WEIGHTS)
    if kind == "rollout":
        g, net = Exact(rollout_mask(case, seed), 1.0 / case["tau"], case["u"]), ExactNet(params)
        for _ in range(case["cycles"]):
            _jump(g, net, case["u"])
            g.step(8)
        return g.fields()
    x, y, w = (torch.from_numpy(a.astype(np.float64)) for a in net_inputs(case, seed))
    net = ExactNet(params, grads=kind == "gradients")
    x, y, w = (a.to(net.p.device) for a in (x, y, w))
    if kind == "predict":
        return net(x)
    total = 0.0
    for i in range(case["batch"]):  # image by image: the graph of one holds every activation
        loss = (w[i:i + 1, ..., None] * (net(x[i:i + 1]) - y[i:i + 1]) ** 2).sum() / w.sum()
        loss.backward(retain_graph=i + 1 < case["batch"])
        total += float(loss.detach())
    return total, net.p.grad


def load_bf16(path):
    """The stored weights (bfloat16 bit patterns) as float32."""
    return (np.load(path, allow_pickle=False).astype(np.uint32) << 16).view(np.float32)
