"""A trajectory's per-trajectory gradient does not depend on where it runs: its
slot, the trajectories beside it in the wave, or the order that a repeated
backward pass starts them in (by the steps of the solve before it, so another
one the second time).  Four trajectories of different lengths, repeated so
often that the waves hold two slots each; every copy equal bit for bit."""
import numpy as np
import pytest

from oracle.mlp import MLP

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("copies", [700, 1000])
@pytest.mark.parametrize("widths", [[4, 13, 4], [9, 17, 31, 9], [6, 40, 6]],
                         ids=lambda w: "-".join(map(str, w)))
def test_copies_are_equal_in_every_slot(widths, copies):
    from diffeqflux_hip import Handle
    m = MLP(widths, ["tanh"] * (len(widths) - 2) + ["identity"])
    rng = np.random.default_rng(sum(widths))
    h = Handle(widths, ["tanh"] * (len(widths) - 2) + ["identity"], 0, "fp32", 1)
    h.set_params(m.glorot_init(rng).astype(np.float32))
    u0 = rng.standard_normal((4, widths[0])).astype(np.float32)
    t1 = rng.uniform(0.3, 1.0, 4)
    saves = [np.linspace(0.0, t, k) for t, k in zip(t1, (2, 3, 5, 4))]
    cots = [rng.standard_normal((len(s), widths[0])).astype(np.float32) for s in saves]
    h.ragged_forward(np.tile(u0, (copies, 1)), np.tile(t1, copies), saves * copies, abstol=1e-6,
                     reltol=1e-6)
    for _ in range(2):
        du0, dp, rows, ret, _, _ = h.ragged_backward(cots * copies, per_trajectory=True)
        assert np.all(ret == 1)
        for x in (du0, rows):
            x = x.reshape(copies, 4, -1)
            assert np.array_equal(x, np.broadcast_to(x[:1], x.shape))
