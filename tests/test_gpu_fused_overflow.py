"""Infinities on the fused FP32 steps stay where they belong.

A hidden relu or softplus value that overflows is inf; the saturating layer
behind it makes it 1, so the solve is an ordinary one.  The oracle, in FP64,
has no overflow there and the same values: FP32 bound 2e-5, that of the
fixed-dt tests, for states and lambda, 1e-4 for the last layer's gradient.
Widths with and without padding of the 16- and 64-feature tiles."""
import numpy as np
import pytest
import torch  # noqa: F401  (before the library: one HIP runtime per process)

from oracle import adjoint as OA
from oracle.mlp import MLP

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.abs(np.asarray(a, np.float64) - b).max() / np.abs(b).max())


@pytest.mark.parametrize("act", ["relu", "softplus"])
@pytest.mark.parametrize("hidden", [(5, 7), (16, 16), (17, 33), (70, 3), (140, 150), (300, 130)])
def test_overflow_behind_a_saturating_layer(hidden, act):
    from diffeqflux_hip import Handle
    widths, acts = [2, *hidden, 2], [act, "tanh", "identity"]
    m = MLP(widths, acts)
    rng = np.random.default_rng(sum(hidden))
    p = []
    for l, (a, b) in enumerate(zip(widths[:-1], widths[1:])):  # W1 u overflows where u > 0
        p += [rng.uniform(0.1, 1.0, a * b) * (1e38, 1.0, 1.0 / b)[l], np.zeros(b)]
    p = np.concatenate(p).astype(np.float32)
    u0 = np.array([[30.0, 40.0], [100.0, 20.0], [-1.0, -2.0]], np.float32)
    h = Handle(widths, acts, 0, "fp32", 3)
    h.set_params(p)
    kw = dict(adaptive=False, dt=0.25)
    out, _, st = h.forward(u0, Handle.make_opts(0.0, 1.0, **kw))
    p64 = p.astype(np.float64)
    ref = OA.forward(m, p64, u0.astype(np.float64), 0.0, 1.0, saveat=[0.0, 1.0], **kw)
    assert st["retcode"] == 1 and rel(out, np.array(ref.u)) < 2e-5
    cot = rng.standard_normal(out.shape).astype(np.float32)
    du0, dp, sb = h.backward(cot)
    gu, gp, _ = OA.backward(m, p64, ref, list(cot.astype(np.float64)), **kw)
    last = -(hidden[1] * 2 + 2)
    assert sb["retcode"] == 1 and rel(du0, gu) < 2e-5
    assert rel(dp[last:], gp[last:]) < 1e-4  # (the second layer's holds inf * 0)


@pytest.mark.parametrize("prec,tol", [("fp32", 1e-4), ("bf16x3", 5e-4)])
@pytest.mark.parametrize("B", [1, 600, 4097])
@pytest.mark.parametrize("hidden", [[], [4]])
def test_last_stage_outside_the_quadrature(hidden, B, prec, tol):
    """lambda overflows in the last stage of a step, which has no weight in the
    parameter gradient: lambda(t0) is inf, the gradient is the oracle's (bounds
    of the fused step tests).  One step of z = w dt = 15: the stage values grow
    by up to 900, the new state by 25442."""
    from diffeqflux_hip import Handle
    widths, acts = [1, *hidden, 1], ["identity"] * (len(hidden) + 1)
    m = MLP(widths, acts)
    p = np.float32([2.0**-7, 0] if not hidden else [2.0**-3] * 4 + [0] * 4 + [2.0**-6] * 4 + [0])
    u0 = np.full((B, 1), 1e-6, np.float32)
    kw, t1 = dict(adaptive=False, dt=1920.0), 1920.0
    h = Handle(widths, acts, 0, prec, B)
    h.set_params(p)
    h.forward(u0, Handle.make_opts(0.0, t1, **kw))
    ref = OA.forward(m, p.astype(np.float64), u0.astype(np.float64), 0.0, t1, saveat=[0.0, t1], **kw)
    cot = np.zeros((2, B, 1), np.float32)
    cot[1] = 5e34 / B
    cot[1, 0] = 5e34
    du0, dp, st = h.backward(cot)
    gu, gp, _ = OA.backward(m, p.astype(np.float64), ref, list(cot.astype(np.float64)), **kw)
    assert st["retcode"] == 1 and gu[0, 0] > 1e39 and np.isposinf(du0[0, 0])
    assert np.linalg.norm(dp - gp) < tol * np.linalg.norm(gp)
