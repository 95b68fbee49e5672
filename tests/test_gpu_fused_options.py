"""The fused steps where their variants meet the handle's options.

* BacksolveAdjoint through every kind of row block (16 rows and 8 rows, one and
  several tiles, remainders, more rows than blocks at once), fixed dt, against
  the FP64 oracle: the gradient bounds of the fused step tests.
* FP32 rounding: the same states, bit for bit, as on the GEMM path (which a tape
  budget selects) for adaptive solves of models up to 32 wide.  There both
  paths have one order for every sum: one K tile per product, whatever plan the
  GEMMs are given.  An adaptive solve's first error estimates are differences of
  rounding-sized terms, so another order shows as other step sizes.  Gradients
  within 50 * tol, as the adaptive tests' (the weight gradients' row sums differ)."""
import numpy as np
import pytest
import torch  # noqa: F401  (before the library: one HIP runtime per process)

from oracle import adjoint as OA
from oracle.mlp import MLP, MAP_CUBE

pytestmark = pytest.mark.gpu

GRAD = {"fp32": 1e-4, "bf16x3": 5e-4}


def rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def model(widths, act, imap=0):
    m = MLP(widths, [act] * (len(widths) - 2) + ["identity"], input_map=imap)
    rng = np.random.default_rng(sum(widths))
    p = m.glorot_init(rng).astype(np.float32)
    for _, b0, b1 in m.offsets:
        p[b0:b1] = 0.1 * rng.standard_normal(b1 - b0)
    return m, p, rng


@pytest.mark.parametrize("ckpt", [True, False])
@pytest.mark.parametrize("prec", ["fp32", "bf16x3"])
@pytest.mark.parametrize("widths,act,B", [
    ([1, 1, 1], "tanh", 1), ([2, 17, 2], "softplus", 17), ([33, 70, 33], "sigmoid", 40),
    ([5, 140, 130, 5], "tanh", 9), ([64, 129, 200, 64], "softplus", 21), ([3, 24, 3], "tanh", 4097)])
def test_backsolve(widths, act, B, prec, ckpt):
    from diffeqflux_hip import Handle
    m, p, rng = model(widths, act)
    u0 = (0.7 * rng.standard_normal((B, widths[0]))).astype(np.float32)
    h = Handle(widths, m.acts, 0, prec, B)
    h.set_params(p)
    h.set_option("sensealg", "backsolve" if ckpt else "backsolve_nockpt")
    kw = dict(adaptive=False, dt=0.125)
    ts = [0.0, 0.2, 0.55, 0.75]
    out, _, _ = h.forward(u0, Handle.make_opts(0.0, 0.75, **kw), ts[1:-1])
    p64 = p.astype(np.float64)
    ref = OA.forward(m, p64, u0.astype(np.float64), 0.0, 0.75, saveat=ts, **kw)
    cot = rng.standard_normal(out.shape).astype(np.float32) / B
    du0, dp, sb = h.backward(cot)
    gu, gp, adj = OA.backward_backsolve(m, p64, ref, list(cot.astype(np.float64)),
                                        checkpointing=ckpt, **kw)
    print(f"\n[backsolve {widths} B={B} {prec} ckpt={ckpt}] dp {rel(dp, gp):.1e} du0 "
          f"{rel(du0, gu):.1e}", flush=True)
    assert sb["retcode"] == 1 and sb["naccept"] == adj.naccept
    assert rel(dp, gp) < GRAD[prec] and rel(du0, gu) < GRAD[prec]


@pytest.mark.parametrize("sense", ["interpolating", "backsolve"])
@pytest.mark.parametrize("tol", [1e-3, 1e-5])
@pytest.mark.parametrize("widths,act,imap,B", [
    ([2, 24, 2], "tanh", MAP_CUBE, 1), ([4, 24, 4], "softplus", 0, 17),
    ([2, 16, 2], "sigmoid", MAP_CUBE, 256), ([9, 31, 32, 9], "tanh", 0, 33),
    ([3, 7, 3], "tanh", 0, 100)])
def test_fp32_states_equal_the_gemm_paths(widths, act, imap, B, tol, sense):
    from diffeqflux_hip import Handle
    m, p, rng = model(widths, act, imap)
    u0 = rng.standard_normal((B, widths[0])).astype(np.float32)
    ts = np.linspace(0.0, 1.2, 7)
    got = []
    for budget in (0, 1 << 30):
        h = Handle(widths, m.acts, imap, "fp32", B)
        h.set_params(p)
        h.set_option("tape_budget", budget)
        h.set_option("sensealg", sense)
        out, _, st = h.forward(u0, Handle.make_opts(0.0, 1.2, abstol=tol, reltol=tol), ts[1:-1])
        cot = np.random.default_rng(5).standard_normal(out.shape).astype(np.float32) / B
        du0, dp, sb = h.backward(cot)
        assert st["retcode"] == 1 and sb["retcode"] == 1
        got.append((out, st["naccept"], st["nreject"], du0, dp))
    (a, *sa, au, ap), (b, *sb, bu, bp) = got
    assert sa == sb and np.array_equal(a, b)
    assert rel(au, bu) < 50 * tol and rel(ap, bp) < 50 * tol
