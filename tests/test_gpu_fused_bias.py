"""Hidden bias gradients of the fused adjoint are sums of FP32 output
gradients: the split-BF16 operand rows (hi + lo planes, ~16 bits) serve the
weight products only.

The model makes everything but that sum exact.  A zero first layer: the state
does not reach the output, so lambda is the end state's cotangent throughout;
a last layer of ones behind identity activations: a hidden output gradient is
the sum of lambda, 1 + 2^-9 + 2^-17, 18 bits of FP32 and 1 + 2^-9 (7.6e-6 less)
in two BF16 planes.  The bias gradient is T * B times it.  Bound 3e-6: sums of up
to 64 rows are exact, the stage weights and the sum over the stages round a
dozen times (6e-8 each), and at most 64 row ranges are added one after the
other (64 / 2 times 6e-8)."""
import numpy as np
import pytest
import torch  # noqa: F401  (before the library: one HIP runtime per process)

pytestmark = pytest.mark.gpu

LAM = np.array([1.0, 2.0**-9, 2.0**-17])
T = 0.75


def parameters(widths):
    p, last = [], len(widths) - 2
    for l, (a, b) in enumerate(zip(widths[:-1], widths[1:])):
        w = np.ones(a * b) if l == last else np.zeros(a * b)
        p += [w, np.full(b, 0.25)]
    return np.concatenate(p).astype(np.float32)


def check(widths, dp, B):
    want, b1 = T * B * LAM.sum(), 0
    for l, (a, b) in enumerate(zip(widths[:-2], widths[1:-1])):
        b1 += a * b
        got, b1 = dp[b1:b1 + b], b1 + b
        if l < len(widths) - 3:  # (behind a zero layer)
            assert np.all(got == 0.0)
        else:
            print(f"  {widths} B={B}: {np.abs(got / want - 1).max():.1e}", flush=True)
            assert np.abs(got / want - 1).max() < 3e-6


@pytest.mark.parametrize("prec", ["fp32", "bf16x3"])
@pytest.mark.parametrize("hidden,B", [([1], 1), ([70], 17), ([128], 130), ([20, 300], 33),
                                      ([24], 4097)])
def test_neural_ode(hidden, B, prec):
    from diffeqflux_hip import Handle
    widths = [3] + hidden + [3]
    h = Handle(widths, ["identity"] * (len(widths) - 1), 0, prec, B)
    h.set_params(parameters(widths))
    h.forward(np.zeros((B, 3), np.float32), Handle.make_opts(0.0, T, adaptive=False, dt=0.25))
    cot = np.zeros((2, B, 3), np.float32)
    cot[1] = LAM
    _, dp, st = h.backward(cot)
    assert st["retcode"] == 1
    check(widths, dp, B)


@pytest.mark.parametrize("prec", ["fp32", "bf16x3"])
@pytest.mark.parametrize("hidden,B", [([1], 1), ([70], 17), ([130], 40), ([20, 300], 33),
                                      ([200], 4099)])
def test_flow(hidden, B, prec):
    from diffeqflux_hip import Handle, _lib
    widths = [4] + hidden + [3]
    h = Handle(widths, ["identity"] * (len(widths) - 1), _lib.MAP_CNF_TIME, prec, B)
    h.set_params(parameters(widths))
    h.cnf_forward(np.zeros((B, 3), np.float32), np.ones((B, 3), np.float32), 0.0, T,
                  adaptive=False, dt=0.25)
    _, dp, st = h.cnf_backward(np.tile(LAM, (B, 1)), np.zeros(B))
    assert st["retcode"] == 1
    check(widths, dp, B)
