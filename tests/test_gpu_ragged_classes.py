"""The per-trajectory kernels are compiled per width class (longest dimension
of any layer: 16, 32, 64 or 128 features) and state size (up to 16, up to 32):
every class against the oracle's adjoint of each trajectory alone, at widths
that leave partial tiles, and with more trajectories than waves, so that a wave
serves several slots.  Four trajectories repeated: all copies must come out
equal bit for bit, whatever slot they ran in.

Bounds: FP32 50 * tol + 1e-5 and BF16 operands 2e-2 of the largest entry, those
of the other per-trajectory adjoint tests (solver tolerance through the adjoint;
operand rounding of 2^-9).
"""
import numpy as np
import pytest

from oracle import adjoint as OA
from oracle.mlp import MLP

pytestmark = pytest.mark.gpu

CLASSES = [  # (repeated 700 times; the last two so often that slots take trajectories
             # from the queue)
    ([3, 13, 3], ["tanh", "identity"]),
    ([2, 16, 16, 9, 2], ["tanh", "softplus", "sigmoid", "identity"]),
    ([9, 17, 31, 9], ["softplus", "tanh", "identity"]),
    ([21, 25, 21], ["tanh", "identity"]),
    ([6, 33, 64, 6], ["sigmoid", "tanh", "identity"]),
    ([30, 50, 30], ["tanh", "identity"]),
    ([5, 65, 5], ["tanh", "identity"]),
    ([18, 100, 18], ["softplus", "identity"]),
    ([2, 16, 16, 8, 2], ["tanh", "softplus", "sigmoid", "identity"]),
    ([4, 13, 4], ["tanh", "identity"]),
]
COPIES = {2: 4000, 4: 8300}  # by state size


@pytest.mark.parametrize("vjp", ["fp32", "bf16"])
@pytest.mark.parametrize("widths,acts", CLASSES, ids=["-".join(map(str, w)) for w, _ in CLASSES])
def test_every_width_class(widths, acts, vjp):
    from diffeqflux_hip import Handle
    tol, distinct = 1e-6, 4
    copies = COPIES[widths[0]] if widths in [c[0] for c in CLASSES[-2:]] else 700
    m = MLP(widths, acts)
    rng = np.random.default_rng(sum(widths))
    p32 = m.glorot_init(rng).astype(np.float32)
    u0 = rng.standard_normal((distinct, widths[0])).astype(np.float32)
    t1 = rng.uniform(0.3, 1.0, distinct)
    saves = [np.linspace(0.0, t, k) for t, k in zip(t1, (2, 3, 5, 4))]
    h = Handle(widths, acts, 0, "fp32", 1)
    h.set_params(p32)
    h.set_option("ragged_vjp_precision", vjp)
    outs, ret, _, _ = h.ragged_forward(np.tile(u0, (copies, 1)), np.tile(t1, copies), saves * copies,
                                       abstol=tol, reltol=tol)
    assert np.all(ret == 1)
    cots = [rng.standard_normal((len(s), widths[0])).astype(np.float32) for s in saves]
    du0, dp, rows, aret, _, _ = h.ragged_backward(cots * copies, per_trajectory=True)
    assert np.all(aret == 1)
    for k in range(1, copies):
        assert np.array_equal(du0[:distinct], du0[k * distinct:(k + 1) * distinct])
        assert np.array_equal(rows[:distinct], rows[k * distinct:(k + 1) * distinct])
    p = p32.astype(np.float64)
    bound = 50 * tol + 1e-5 if vjp == "fp32" else 2e-2
    for i in range(distinct):
        ref = OA.forward(m, p, u0[i:i + 1].astype(np.float64), 0.0, float(t1[i]), saveat=list(saves[i]),
                         abstol=tol, reltol=tol)
        gu0, gp, _ = OA.backward(m, p, ref, [c[None].astype(np.float64) for c in cots[i]],
                                 abstol=tol, reltol=tol)
        assert np.abs(du0[i] - gu0[0]).max() < bound * np.abs(gu0).max()
        assert np.abs(rows[i] - gp).max() < bound * np.abs(gp).max()
    assert np.allclose(dp, rows.astype(np.float64).sum(0), rtol=1e-6, atol=1e-9)
