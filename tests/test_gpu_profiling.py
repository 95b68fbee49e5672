"""node_prof_enable records the launches that a solve makes, on either path:
the products of the layers, or the fused steps' kernels."""
import numpy as np
import pytest
import torch  # noqa: F401  (before the library: one HIP runtime per process)

pytestmark = pytest.mark.gpu

GEMM = {(0, 0), (1, 1), (2, 0), (3, 1), (4, 0), (4, 1), (5, 0)}
FUSED = {(6, 0), (7, 0), (7, 1), (7, 2)}


@pytest.mark.parametrize("budget,keys", [(0, FUSED), (1 << 30, GEMM)], ids=["fused", "gemm"])
def test_records_of_a_solve_and_its_adjoint(budget, keys):
    from diffeqflux_hip import Handle
    h = Handle([3, 20, 3], ["tanh", "identity"], 0, "fp32", 17)
    h.set_params(0.1 * np.ones(h.P, np.float32))
    h.set_option("tape_budget", budget)
    u0, cot = np.ones((17, 3), np.float32), np.ones((2, 17, 3), np.float32)
    opts = Handle.make_opts(0.0, 1.0, adaptive=False, dt=0.25)

    def records():
        h.forward(u0, opts)
        h.backward(cot)
        return h.prof_collect()
    assert records() == []
    h.prof_enable(None)
    recs = records()
    assert {k for k, _ in recs} == keys and all(ms > 0 for _, ms in recs)
    one = sorted(keys)[1]
    h.prof_enable([one])
    assert {k for k, _ in records()} == {one}
    h.prof_enable([])
    assert records() == []
