"""GPU: the gate's training gradient at batch sizes around its tiles (32
samples) and above the 256 tiles that one pass of the grid takes, against the
float64 oracle.

Tolerance: an output unit's error is a few dozen roundings of the 64-term
sums before it (u = 2^-24 each, relative to the absolute terms), and a
parameter's sum over the batch adds at most a tile chain (32 per tile of its
block) and the partials' chain, which for n samples stays below n / 8 + 64
roundings; they add in quadrature at worst to (150 + n / 8) u of the norm."""
import numpy as np
import pytest

import delta2_amd as d2
import mlp_oracle as mo
from delta2_amd import learned

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 31, 32, 33, 1000, 8192, 8193, 20011])
def test_gradient_batch_sizes(n):
    rng = np.random.default_rng(n)
    X = rng.normal(0.0, 0.5, size=(n, 24)).astype(np.float32)
    T = rng.uniform(0.0, 1.3, size=(n, 2)).astype(np.float32)
    params = learned.init_params(n)
    with d2.Context(0, d2.D2_FP32) as ctx:
        ctx.mlp_set_params(params)
        loss, g = ctx.mlp_loss_grad(X, T, learned.LW, learned.DELTA)
        loss2, g2 = ctx.mlp_loss_grad(X, T, learned.LW, learned.DELTA)
    ol, og = mo.loss_grad(params, X, T, lw=learned.LW, delta=learned.DELTA)
    tol = (150 + n / 8) * 2.0 ** -24
    err = np.linalg.norm(g - og) / np.linalg.norm(og)
    print(f"[grad n={n}] loss {loss:.7f} oracle {ol:.7f}, gradient off {err:.2e} (bound {tol:.2e})", flush=True)
    assert np.array_equal(g, g2) and loss == loss2  # a fixed order
    assert abs(loss - ol) <= tol * abs(ol)
    assert err <= tol
