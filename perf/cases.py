"""The work that is timed on the GPU: what programs built on this package run.

A case is one pass through the public entry points: a training step of a
``NeuralODE`` layer (solve, loss, gradients), a solve alone, an ``FFJORD``
training step or density evaluation, a batch of per-trajectory solves with
their gradients, or one multiple-shooting loss with its gradient.  Sizes are
those of the package's workloads, examples and tests; ``draw`` gives other
sizes of the same ranges.

A program builds its layer once and calls it for every new batch of inputs
and every new parameter vector.  So the layer (or handle) of a configuration
is made once and kept while its case is the current one; every pass hands it
its own parameters and inputs.
"""
import functools
import math
import os
import sys

import numpy as np
import torch
import torch.utils.checkpoint

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "diffeqflux.jl_amd"))
from diffeqflux_hip import (FFJORD, BacksolveAdjoint, Chain, Cube, Dense, EnsembleProblem,  # noqa: E402
                            EnsembleThreads, Handle, NeuralODE, Tsit5, group_ranges, multiple_shoot)

DEVICE = "cuda"


# ---------------------------------------------------------------- the cases
def _train(widths, act, batch, saves, t1, rtol, atol, precision="fp32", cube=False,
           sensealg="interpolating"):
    return dict(kind="train", widths=widths, act=act, batch=batch, saves=saves, t1=t1, rtol=rtol,
                atol=atol, precision=precision, cube=cube, sensealg=sensealg)


def _solve(widths, act, batch, saves, t1, rtol, atol, precision="fp32", cube=False):
    return dict(kind="solve", widths=widths, act=act, batch=batch, saves=saves, t1=t1, rtol=rtol,
                atol=atol, precision=precision, cube=cube)


def _flow(kind, widths, act, batch, rtol, atol, precision):
    return dict(kind=kind, widths=widths, act=act, batch=batch, rtol=rtol, atol=atol,
                precision=precision)


def _ragged(widths, act, n, tmax, max_saves, rtol, atol):
    return dict(kind="ragged", widths=widths, act=act, n=n, tmax=tmax, max_saves=max_saves,
                rtol=rtol, atol=atol)


def _shoot(hidden, trajectories, points, group):
    return dict(kind="shoot", widths=f"2-{hidden}-2", act="tanh", trajectories=trajectories,
                points=points, group=group, rtol=1e-3, atol=1e-6)


def listed():
    return [
        # the documentation's first example: one trajectory, one gradient at a
        # time; nothing but latency
        dict(_train("2-50-2", "tanh", 1, 30, 1.5, 1e-6, 1e-6, cube=True), name="spiral_1"),
        # the same model over a small batch with the reference's other adjoint
        # and its default tolerances
        dict(_train("2-50-2", "tanh", 50, 30, 1.5, 1e-3, 1e-6, cube=True, sensealg="backsolve"),
             name="spiral_backsolve_50"),
        # an ordinary FP32 training step: middling width, a full batch
        dict(_train("32-256-256-32", "tanh", 4096, 20, 1.0, 1e-5, 1e-7), name="plain_4096"),
        # the same model on the last, ragged batch of an epoch
        dict(_train("32-256-256-32", "tanh", 333, 20, 1.0, 1e-5, 1e-7), name="plain_333"),
        # prediction alone, batch that fills no tile
        dict(_solve("32-256-256-32", "tanh", 1000, 20, 1.0, 1e-5, 1e-7), name="plain_solve_1000"),
        # the large training step: wide layers, split-BF16 products
        dict(_train("64-1024-1024-1024-64", "softplus", 4096, 32, 1.0, 1e-4, 1e-6, "bf16x3"),
             name="wide_4096_bf16x3"),
        # the wide model in plain FP32 on a smaller, odd batch
        dict(_train("64-1024-1024-1024-64", "softplus", 1000, 8, 1.0, 1e-4, 1e-6),
             name="wide_1000_fp32"),
        # many trajectories, each with its own span, save times and step sizes
        dict(_ragged("16-128-128-16", "tanh", 10000, 5.0, 200, 1e-5, 1e-6), name="ragged_10000"),
        # density evaluation and the training step of a normalizing flow
        dict(_flow("flow_density", "17-512-512-16", "tanh", 8192, 1e-5, 1e-5, "bf16x3"),
             name="flow_density_8192"),
        dict(_flow("flow_train", "17-512-512-16", "tanh", 8192, 1e-5, 1e-5, "bf16x3"),
             name="flow_train_8192"),
        # a small flow in FP32 (two-dimensional data, a few hundred samples)
        dict(_flow("flow_train", "3-64-64-2", "tanh", 500, 1e-3, 1e-6, "fp32"),
             name="flow_train_500"),
        # ensemble multiple shooting of the documentation's spiral
        dict(_shoot(16, 1024, 30, 3), name="shoot_1024"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["train", "train", "train", "spiral", "solve", "flow_train", "flow_density",
                       "ragged", "shoot"])
    if kind == "spiral":
        return _train(f"2-{_log(rng, 16, 64)}-2", "tanh", _log(rng, 1, 256), rng.randint(5, 40),
                      round(rng.uniform(0.8, 1.5), 2), rng.choice([1e-3, 1e-4, 1e-5]), 1e-6,
                      cube=True, sensealg=rng.choice(["interpolating", "backsolve"]))
    if kind in ("train", "solve"):
        precision = rng.choice(["fp32", "bf16x3"])
        d, h, n = rng.randint(2, 64), _log(rng, 16, 1024), rng.randint(1, 3)
        widths = [d] + [h] * n + [d]
        size = sum(a * b for a, b in zip(widths[:-1], widths[1:]))
        most = 4096 * 2228224 // (1 if precision == "bf16x3" else 4)
        batch = max(1, min(_log(rng, 1, 8192), most // size, 4096 * 64 // d))
        rtol = rng.choice([1e-3, 1e-4, 1e-5] if precision == "fp32" else [1e-3, 1e-4])
        make = _train if kind == "train" else _solve
        return make("-".join(map(str, widths)), rng.choice(["tanh", "softplus", "sigmoid"]), batch,
                    rng.randint(2, 32), round(rng.uniform(0.5, 1.5), 2), rtol, rtol / 100,
                    precision)
    if kind.startswith("flow"):
        precision = rng.choice(["fp32", "bf16x3"])
        d, h, n = rng.randint(2, 16), _log(rng, 32, 512), rng.randint(1, 2)
        batch = _log(rng, 100, 8192 if precision == "bf16x3" else 2048)
        rtol = rng.choice([1e-3, 1e-4])
        return _flow(kind, "-".join(map(str, [d + 1] + [h] * n + [d])),
                     rng.choice(["tanh", "softplus"]), batch, rtol, 1e-5, precision)
    if kind == "ragged":
        d, h, n = rng.randint(2, 16), _log(rng, 16, 128), rng.randint(1, 2)
        return _ragged("-".join(map(str, [d] + [h] * n + [d])), rng.choice(["tanh", "softplus"]),
                       _log(rng, 10, 10000), round(rng.uniform(1.0, 5.0), 2), rng.randint(10, 200),
                       rng.choice([1e-3, 1e-4, 1e-5]), 1e-6)
    return _shoot(_log(rng, 8, 50), _log(rng, 1, 1024), rng.randint(20, 40), rng.randint(2, 10))


# ---------------------------------------------------------------- inputs
def _widths(case):
    return [int(w) for w in case["widths"].split("-")]


def _chain(case):
    w = _widths(case)
    dense = [Dense(a, b, case["act"]) for a, b in zip(w[:-2], w[1:-1])] + [Dense(w[-2], w[-1])]
    return Chain(*([Cube()] if case.get("cube") or case["kind"] == "shoot" else []), *dense)


@functools.lru_cache(maxsize=1)
def _layer(key):
    """The layer or handle of a configuration (one kept at a time)."""
    case = dict(key)
    kind = case["kind"]
    if kind == "ragged":
        w = _widths(case)
        return Handle(w, [case["act"]] * (len(w) - 2) + ["identity"])
    chain = _chain(case)
    if kind.startswith("flow"):
        return FFJORD(chain, (0.0, 1.0), (_widths(case)[-1],), Tsit5(), abstol=case["atol"],
                      reltol=case["rtol"], precision=case["precision"])
    if kind == "shoot":
        t = np.linspace(0.0, 5.0, case["points"])
        return NeuralODE(chain, (0.0, 5.0), Tsit5(), saveat=list(t))
    more = {"sensealg": BacksolveAdjoint()} if case.get("sensealg") == "backsolve" else {}
    return NeuralODE(chain, (0.0, case["t1"]), Tsit5(), saveat=list(_saves(case)),
                     abstol=case["atol"], reltol=case["rtol"], precision=case["precision"], **more)


def _saves(case):
    return np.linspace(0.0, case["t1"], case["saves"])


def _parameters(case, seed):
    """Glorot weights and small biases, flat, layer by layer (column-major
    weight, then bias)."""
    rng = np.random.default_rng([seed, 1])
    p, w = [], _widths(case)
    for a, b in zip(w[:-1], w[1:]):
        lim = math.sqrt(6.0 / (a + b))
        p += [rng.uniform(-lim, lim, a * b), 0.05 * rng.standard_normal(b)]
    return np.concatenate(p).astype(np.float32)


def _rk4(f, u, dt, t=None):
    k1 = f(u) if t is None else f(u, t)
    k2 = f(u + 0.5 * dt * k1) if t is None else f(u + 0.5 * dt * k1, t + 0.5 * dt)
    k3 = f(u + 0.5 * dt * k2) if t is None else f(u + 0.5 * dt * k2, t + 0.5 * dt)
    k4 = f(u + dt * k3) if t is None else f(u + dt * k3, t + dt)
    return u + dt / 6 * (k1 + 2 * k2 + 2 * k3 + k4)


def _initial(case, seed):
    """Initial states: N(0, 1), or points on the spiral's radius."""
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    d, b = _widths(case)[0], case["batch"]
    if case["cube"]:
        ang = 2 * math.pi * torch.rand(b, generator=g, device=DEVICE)
        rad = 1.5 + 0.5 * torch.rand(b, generator=g, device=DEVICE)
        return torch.stack([rad * torch.cos(ang), rad * torch.sin(ang)], 1)
    return torch.randn(b, d, generator=g, device=DEVICE)


def _targets(case, u0, seed):
    """States at the save times of the system that the model is fitted to: the
    cubic spiral, or a random linear-plus-tanh system."""
    d = u0.shape[1]
    if case["cube"]:
        a = torch.tensor([[-0.1, 2.0], [-2.0, -0.1]], device=DEVICE)
        f = lambda u: (u ** 3) @ a                                        # noqa: E731
    else:
        rng = np.random.default_rng([seed, 2])
        a = -np.eye(d) + 0.5 * rng.standard_normal((d, d)) / math.sqrt(d)
        c = rng.standard_normal((d, d)) / math.sqrt(d)
        a = torch.tensor(a.T.astype(np.float32), device=DEVICE)
        c = torch.tensor(c.T.astype(np.float32), device=DEVICE)
        f = lambda u: u @ a + torch.tanh(u @ c)                           # noqa: E731
    ts, u = _saves(case), u0
    out = [u]
    for dt in np.diff(ts):
        n = max(1, math.ceil(dt / 0.04))
        for _ in range(n):
            u = _rk4(f, u, float(dt) / n)
        out.append(u)
    return torch.stack(out)


def _ragged_inputs(case, seed):
    rng = np.random.default_rng([seed, 3])
    n, d = case["n"], _widths(case)[0]
    u0 = rng.standard_normal((n, d)).astype(np.float32)
    t1 = rng.uniform(0.1, case["tmax"], n)
    # the same save counts for every seed, over other trajectories
    counts = rng.permutation(np.random.default_rng(n).integers(5, case["max_saves"] + 1, n))
    times = np.concatenate([np.linspace(0.0, t, c) for t, c in zip(t1, counts)])
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    return u0, t1, counts, times, offsets


def _ring(n, d, seed):
    """Eight clusters on a ring in the first two coordinates, N(0, 1) in the others."""
    rng = np.random.default_rng([seed, 4])
    k = rng.integers(0, 8, n)
    x = rng.standard_normal((n, d)).astype(np.float32)
    ang = 2 * math.pi * k / 8
    x[:, 0] = 4 * np.cos(ang) + 0.5 * rng.standard_normal(n)
    x[:, 1] = 4 * np.sin(ang) + 0.5 * rng.standard_normal(n)
    return x


def _shoot_data(case, seed):
    rng = np.random.default_rng([seed, 5])
    n = case["trajectories"]
    t = np.linspace(0.0, 5.0, case["points"])
    ang, rad = rng.uniform(0, 2 * math.pi, n), rng.uniform(1.5, 2.5, n)
    u = np.stack([rad * np.cos(ang), rad * np.sin(ang)], 1)
    a = np.array([[-0.1, 2.0], [-2.0, -0.1]])
    out = [u]
    for dt in np.diff(t):
        for _ in range(24):
            u = _rk4(lambda x: (x ** 3) @ a, u, dt / 24)
        out.append(u)
    return t, np.stack(out, 1).astype(np.float32)


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "layer": _layer(tuple(sorted((k, v) for k, v in case.items()
                                                    if k != "name")))}
    p = _parameters(case, seed)
    if kind in ("train", "solve"):
        s["p"] = torch.from_numpy(p).to(DEVICE)
        s["u0"] = _initial(case, seed)
        if kind == "train":
            s["target"] = _targets(case, s["u0"], seed)
    elif kind.startswith("flow"):
        n, d = case["batch"], _widths(case)[-1]
        s["p"] = torch.from_numpy(p).to(DEVICE)
        s["x"] = torch.from_numpy(_ring(n, d, seed)).to(DEVICE)
        probe = np.random.default_rng([seed, 6]).choice(np.array([-1.0, 1.0], np.float32), (n, d))
        s["state"] = {"regularize": False, "monte_carlo": True, "probe": probe}
    elif kind == "ragged":
        u0, t1, counts, times, offsets = _ragged_inputs(case, seed)
        s.update(p=p, u0=u0, t1=t1, saves=(times, offsets),
                 weight=np.repeat((0.5 * counts * case["n"]).astype(np.float32), counts)[:, None])
    else:
        s["t"], s["data"] = _shoot_data(case, seed)
        s["p"] = torch.from_numpy(p)
    return s


# ---------------------------------------------------------------- one pass
def _squares(u, v):
    return ((u - v) ** 2).sum()


def run(state):
    case, layer = state["case"], state["layer"]
    kind = case["kind"]
    if kind == "solve":
        sol, _ = layer(state["u0"], state["p"])
        return sol.array
    if kind == "train":
        u0 = state["u0"].detach().requires_grad_()
        p = state["p"].detach().requires_grad_()
        sol, _ = layer(u0, p)
        loss = ((sol.array - state["target"]) ** 2).mean()
        loss.backward()
        return {"states": sol.array.detach(), "du0": u0.grad, "dp": p.grad}
    if kind == "flow_density":
        with torch.no_grad():
            (logpx, delta, _), _ = layer(state["x"], state["p"], state["state"])
        return {"logpx": logpx, "delta": delta}
    if kind == "flow_train":
        x = state["x"].detach().requires_grad_()
        p = state["p"].detach().requires_grad_()
        (logpx, _, _), _ = layer(x, p, state["state"])
        (-logpx.mean()).backward()
        return {"logpx": logpx.detach(), "dx": x.grad, "dp": p.grad}
    if kind == "ragged":
        # gradients of sum |u|^2 / (counts * n); the parameters' in their own type
        layer.set_params(state["p"])
        u, _, _, _ = layer.ragged_forward(state["u0"], state["t1"], state["saves"],
                                          abstol=case["atol"], reltol=case["rtol"], flat_out=True)
        du0, dp, _, _, _, _ = layer.ragged_backward(u / state["weight"])
        return {"states": u, "du0": du0, "dp": dp.astype(np.float32)}
    p = state["p"].detach().requires_grad_()
    loss, preds = multiple_shoot(p, state["data"], state["t"], EnsembleProblem(layer),
                                 EnsembleThreads(), _squares, Tsit5(), case["group"],
                                 continuity_term=200, trajectories=case["trajectories"],
                                 abstol=case["atol"], reltol=case["rtol"])
    loss.backward()
    return {"loss": loss.detach(), "preds": [x.detach() for x in preds], "dp": p.grad}


# ---------------------------------------------------------------- work
def work(case):
    """Bytes: every input read once and every output written once.  Flops: the
    products of one right-hand side (and of one pullback) at each stage of the
    fewest steps that the save times and the order of the method allow: a step
    per interval between saved times on the way back, and a step per 0.1 of
    time (0.05 at tight tolerances) on the way out."""
    w, kind = _widths(case), case["kind"]
    size = sum(a * b for a, b in zip(w[:-1], w[1:]))
    params = size + sum(w[1:])
    d = w[-1]
    step = 0.05 if case["rtol"] < 1e-4 else 0.1
    if kind in ("train", "solve"):
        b, n = case["batch"], case["saves"]
        fwd = 6 * max(2, math.ceil(case["t1"] / step))
        if kind == "solve":
            return {"bytes": 4.0 * (b * d * (1 + n) + params), "flops": 2.0 * b * size * fwd}
        return {"bytes": 4.0 * (b * d * (2 + 2 * n) + 2 * params),
                "flops": 2.0 * b * size * (fwd + 3 * 6 * (n - 1))}
    if kind.startswith("flow"):
        b, fwd = case["batch"], 6 * math.ceil(1.0 / step)
        if kind == "flow_density":
            return {"bytes": 4.0 * (b * (2 * d + 2) + params), "flops": 4.0 * b * size * fwd}
        return {"bytes": 4.0 * (b * (3 * d + 2) + 2 * params), "flops": 2.0 * b * size * fwd * 8}
    if kind == "ragged":
        n, saves = case["n"], (5 + case["max_saves"]) / 2
        fwd = 6 * max(2, math.ceil(case["tmax"] / 2 / (2 * step)))
        return {"bytes": 4.0 * (n * d * (2 + 2 * saves) + 2 * params) + 8.0 * n * saves,
                "flops": 2.0 * n * size * (fwd + 3 * 6 * (saves - 1))}
    n, pts = case["trajectories"], case["points"]
    groups = group_ranges(pts, case["group"])
    return {"bytes": 4.0 * (2 * n * pts * 2 + 2 * params),
            "flops": 2.0 * n * size * (6 * len(groups) + 3 * 6 * (pts - 1))}


# ---------------------------------------------------------------- in 64 bits
def _double_model(case, p):
    """The model and its directional derivative in 64 bits: x -> f(x) and
    (x, v) -> f(x), df/dx v."""
    w, layers, at = _widths(case), [], 0
    for a, b in zip(w[:-1], w[1:]):
        layers.append((p[at:at + a * b].reshape(a, b), p[at + a * b:at + a * b + b]))
        at += a * b + b
    act = {"tanh": torch.tanh, "softplus": torch.nn.functional.softplus,
           "sigmoid": torch.sigmoid}[case["act"]]
    slope = {"tanh": lambda z, y: 1 - y * y, "softplus": lambda z, y: torch.sigmoid(z),
             "sigmoid": lambda z, y: y * (1 - y)}[case["act"]]
    cube = case.get("cube") or case["kind"] == "shoot"

    def f(x):
        h = x ** 3 if cube else x
        for k, (wt, b) in enumerate(layers):
            h = h @ wt + b
            h = act(h) if k < len(layers) - 1 else h
        return h

    def jvp(x, v):
        h = x
        for k, (wt, b) in enumerate(layers):
            z, v = h @ wt + b, v @ wt
            h = act(z) if k < len(layers) - 1 else z
            v = v * slope(z, h) if k < len(layers) - 1 else v
        return h, v
    return f, jvp


def _step(f, u, dt, *t):
    """One step of the classical fourth-order method; its stages are not kept
    for the way back but computed again."""
    return torch.utils.checkpoint.checkpoint(lambda x: _rk4(f, x, dt, *t), u, use_reentrant=False)


def _path(f, u, ts, h):
    out = [u]
    for dt in np.diff(ts):
        n = max(1, math.ceil(dt / h - 1e-9))
        for _ in range(n):
            u = _step(f, u, float(dt) / n)
        out.append(u)
    return torch.stack(out)


def exact(case, seed):
    """The solution of the differential equation and the gradients through
    it in 64 bits, by small fixed steps."""
    dev = DEVICE if torch.cuda.is_available() else "cpu"
    dbl = lambda x: torch.as_tensor(x).to(dev, torch.float64)             # noqa: E731
    kind = case["kind"]
    p = dbl(_parameters(case, seed)).requires_grad_()
    f, jvp = _double_model(case, p)
    if kind in ("train", "solve"):
        x = _initial(case, seed)
        u0 = dbl(x).requires_grad_()
        ts = _saves(case)
        h = 0.002 if case["cube"] else 0.01
        if kind == "solve":
            with torch.no_grad():
                return _path(f, u0, ts, h)
        u = _path(f, u0, ts, h)
        ((u - dbl(_targets(case, x, seed))) ** 2).mean().backward()
        return {"states": u.detach(), "du0": u0.grad, "dp": p.grad}
    if kind.startswith("flow"):
        n, d = case["batch"], _widths(case)[-1]
        x = dbl(_ring(n, d, seed)).requires_grad_()
        e = dbl(np.random.default_rng([seed, 6]).choice(np.array([-1.0, 1.0], np.float32), (n, d)))

        def g(u, t):
            z = torch.cat([u[:, :d], torch.full_like(u[:, :1], t)], 1)
            y, v = jvp(z, torch.cat([e, torch.zeros_like(e[:, :1])], 1))
            return torch.cat([y, -(e * v).sum(1, keepdim=True)], 1)

        u = torch.cat([x, torch.zeros_like(x[:, :1])], 1)
        with torch.set_grad_enabled(kind == "flow_train"):
            for k in range(64):
                u = _step(g, u, 1 / 64, k / 64)
        z, delta = u[:, :d], u[:, d].reshape(1, n)
        logpx = (-0.5 * (z * z).sum(1) - 0.5 * d * math.log(2 * math.pi)).reshape(1, n) - delta
        if kind == "flow_density":
            return {"logpx": logpx, "delta": delta}
        (-logpx.mean()).backward()
        return {"logpx": logpx.detach(), "dx": x.grad, "dp": p.grad}
    if kind == "ragged":
        u0, t1, counts, _, _ = _ragged_inputs(case, seed)
        gap = t1 / (counts - 1)
        sub = np.ceil(gap / 0.02).astype(np.int64)
        total = sub * (counts - 1)
        u0 = dbl(u0).requires_grad_()
        u, out = u0, [u0]
        dt = dbl(gap / sub)[:, None]
        left = torch.as_tensor(total, device=dev)[:, None]
        for k in range(int(total.max())):
            u = _step(f, u, torch.where(left > k, dt, torch.zeros_like(dt)))
            out.append(u)
        step = np.concatenate([np.arange(c) * m for c, m in zip(counts, sub)])
        which = np.repeat(np.arange(len(counts)), counts)
        u = torch.stack(out)[torch.as_tensor(step, device=dev), torch.as_tensor(which, device=dev)]
        weight = dbl(np.repeat(0.5 * counts * case["n"], counts))[:, None]
        (u * u / (2 * weight)).sum().backward()
        return {"states": u.detach(), "du0": u0.grad, "dp": p.grad}
    t, data = _shoot_data(case, seed)
    data = dbl(data)
    loss, preds, end = 0.0, [], None
    for rg in group_ranges(case["points"], case["group"]):
        u = _path(f, data[:, rg.start], t[rg.start:rg.stop], 0.005).transpose(0, 1)
        loss = loss + _squares(data[:, rg.start:rg.stop], u)
        if end is not None:
            loss = loss + 200 * (end - data[:, rg.start]).abs().sum()
        preds.append(u.detach())
        end = u[:, -1]
    loss.backward()
    return {"loss": loss.detach(), "preds": preds, "dp": p.grad}
