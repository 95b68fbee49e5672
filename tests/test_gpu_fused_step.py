"""The fused step kernels at the sizes where they can go wrong (one and many
16-feature tiles, remainders of tiles and K tiles, one row, a row more than a
block, more rows than CU-filling blocks, one Dense layer, the widest layer),
forward and adjoint, against the FP64 oracle on one fixed-dt step sequence.

Tolerances: those of the fixed-dt parity tests (FP32 2e-5 on states, 1e-4 on
gradients; split BF16, ~16 mantissa bits per operand, 5e-5 and 5e-4)."""
import numpy as np
import pytest
import torch  # (before the library: one HIP runtime per process)

from oracle import adjoint as OA
from oracle import ffjord as FF
from oracle.mlp import MLP, MAP_CUBE

pytestmark = pytest.mark.gpu

TOL = {"fp32": (2e-5, 1e-4), "bf16x3": (5e-5, 5e-4)}
# (no relu here: operand rounding moves units across its kink, whose effect on a
# gradient the operands' precision does not bound)
ACT = ["tanh", "softplus", "sigmoid"]


def rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def model(widths, acts, seed=0, imap=0):
    m = MLP(widths, acts, input_map=imap) if imap else MLP(widths, acts)
    rng = np.random.default_rng(seed)
    p = m.glorot_init(rng).astype(np.float32)
    for _, b0, b1 in m.offsets:
        p[b0:b1] = 0.1 * rng.standard_normal(b1 - b0)
    return m, p, rng


@pytest.mark.parametrize("prec", ["fp32", "bf16x3"])
@pytest.mark.parametrize("hidden,D,B", [
    ([], 5, 3), ([1], 1, 1), ([16], 2, 16), ([17], 2, 17), ([50], 2, 1), ([33, 70], 33, 65),
    ([128, 32], 16, 33), ([100, 300, 40], 64, 20), ([512], 64, 16), ([256, 256], 32, 130),
    ([24], 3, 4097), ([70], 5, 512), ([70], 5, 513),
    ([130, 200], 7, 9), ([129, 513], 64, 21), ([140, 130], 3, 2048), ([140, 130], 3, 2049)])
def test_neural_ode(hidden, D, B, prec):
    from diffeqflux_hip import Handle
    widths = [D] + hidden + [D]
    acts = [ACT[(i + len(hidden) + D) % 3] for i in range(len(hidden))] + ["identity"]
    imap = MAP_CUBE if D == 2 else 0
    print(f"\n[fused step {widths} {acts} B={B} {prec}]", flush=True)
    m, p, rng = model(widths, acts, imap=imap)
    u0 = (0.7 * rng.standard_normal((B, D))).astype(np.float32)
    h = Handle(widths, acts, imap, prec, B)
    h.set_params(p)
    kw = dict(adaptive=False, dt=0.125)
    ts = [0.0, 0.2, 0.55, 0.75]
    out, t, st = h.forward(u0, Handle.make_opts(0.0, 0.75, **kw), ts[1:-1])
    p64 = p.astype(np.float64)
    ref = OA.forward(m, p64, u0.astype(np.float64), 0.0, 0.75, saveat=ts, **kw)
    assert st["retcode"] == 1 and np.array_equal(t, ts)
    assert rel(out, ref.u) < TOL[prec][0]
    cot = rng.standard_normal(out.shape).astype(np.float32) / B
    du0, dp, sb = h.backward(cot)
    gu, gp, adj = OA.backward(m, p64, ref, list(cot.astype(np.float64)), **kw)
    print(f"  states {rel(out, ref.u):.1e} dp {rel(dp, gp):.1e} du0 {rel(du0, gu):.1e}", flush=True)
    assert sb["retcode"] == 1 and sb["naccept"] == adj.naccept
    assert rel(dp, gp) < TOL[prec][1] and rel(du0, gu) < TOL[prec][1]


@pytest.mark.parametrize("prec", ["fp32", "bf16x3"])
@pytest.mark.parametrize("hidden,D,tcat,B", [
    ([1], 1, True, 1), ([20], 2, False, 17), ([64, 64], 2, True, 33), ([100, 40], 15, True, 16),
    ([130], 31, False, 40), ([512, 512], 16, True, 20), ([24], 3, True, 4099)])
def test_flow(hidden, D, tcat, B, prec):
    from diffeqflux_hip import Handle, _lib
    widths = [D + tcat] + hidden + [D]
    acts = [ACT[(i + D) % 3] for i in range(len(hidden))] + ["identity"]
    print(f"\n[fused flow step {widths} {acts} B={B} {prec}]", flush=True)
    m, p, rng = model(widths, acts)
    x = rng.standard_normal((B, D)).astype(np.float32)
    e = rng.choice(np.array([-1.0, 1.0], np.float32), size=(B, D))
    h = Handle(widths, acts, _lib.MAP_CNF_TIME if tcat else _lib.MAP_CNF, prec, B)
    h.set_params(p)
    kw = dict(adaptive=False, dt=0.25)
    lp, z, dl, st = h.cnf_forward(x, e, 0.0, 0.75, **kw)
    p64 = p.astype(np.float64)
    rlp, rz, rdl, sol = FF.forward(m, p64, x.astype(np.float64), 0.0, 0.75,
                                   probe=e.astype(np.float64), time_concat=tcat, **kw)
    assert st["retcode"] == 1
    assert rel(z, rz) < TOL[prec][0] and rel(lp, rlp) < TOL[prec][0]
    # (delta_logp is a sum of signed terms: on the scale of logpx)
    assert np.abs(dl - rdl).max() < 4 * TOL[prec][0] * np.abs(rlp).max()
    gz, gd = FF.nll_cotangents(rz, B)
    dx, dp, sb = h.cnf_backward(gz.astype(np.float32), gd.astype(np.float32))
    rx, rp, _ = FF.backward(m, p64, sol, e.astype(np.float64), gz, gd, time_concat=tcat, **kw)
    print(f"  z {rel(z, rz):.1e} logpx {rel(lp, rlp):.1e} dp {rel(dp, rp):.1e} dx {rel(dx, rx):.1e}",
          flush=True)
    assert sb["retcode"] == 1
    assert rel(dp, rp) < TOL[prec][1] and rel(dx, rx) < TOL[prec][1]


@pytest.mark.parametrize("prec", ["fp32", "bf16x3"])
def test_parameters_from_host_and_device_agree(prec):
    from diffeqflux_hip import Handle
    widths, acts = [33, 65, 130, 33], ["tanh", "softplus", "identity"]
    _, p, rng = model(widths, acts)
    u = rng.standard_normal((5, 33)).astype(np.float32)
    got = []
    for q in (p, torch.from_numpy(p).cuda()):
        h = Handle(widths, acts, 0, prec, 5)
        h.set_params(q)
        out, _, _ = h.forward(u, Handle.make_opts(0.0, 1.0, adaptive=False, dt=0.25))
        got.append((h.rhs(u), out))
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
