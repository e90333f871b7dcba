"""GPU: every sample of a training batch counts, the ragged last tile's last one
too: batches whose final sample carries most of the loss and of the gradient,
and plain ones, against the float64 oracle.

Tolerance (u = 2^-24): an output unit's error is at most 150 u of the 64-term
sums before it; a parameter's sum over the batch is a chain of 32 products for
each tile its block takes (the tiles divided over at most 256 blocks), then of
the blocks' partials, 1 in 8 per wavefront and 8 wavefronts.  One sample left
out of a plain batch of 20011 moves the gradient by 1e-4, seven times the
bound there."""
import numpy as np
import pytest

import delta2_amd as d2
import mlp_oracle as mo
from delta2_amd import learned

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heavy", [False, True])
@pytest.mark.parametrize("n", [1, 31, 33, 257, 8193, 16385, 20011])
def test_last_sample_counts(n, heavy):
    rng = np.random.default_rng(n)
    X = rng.normal(0.0, 0.5, size=(n, 24)).astype(np.float32)
    T = rng.uniform(0.0, 1.3, size=(n, 2)).astype(np.float32)
    delta = learned.DELTA
    if heavy:  # a residual of 1e6, on the quadratic branch
        T[-1] = 1e6
        delta = 1e9
    params = learned.init_params(n)
    with d2.Context(0, d2.D2_FP32) as ctx:
        ctx.mlp_set_params(params)
        loss, g = ctx.mlp_loss_grad(X, T, learned.LW, delta)
    ol, og = mo.loss_grad(params, X, T, lw=learned.LW, delta=delta)
    if heavy and n > 1:  # the others are a small part
        ol1, og1 = mo.loss_grad(params, X[:-1], T[:-1], lw=learned.LW, delta=delta)
        assert ol1 < 1e-3 * ol and np.linalg.norm(og1) < 0.1 * np.linalg.norm(og)
    tiles = -(-n // 32)
    blocks = min(tiles, 256)
    tol = (150 + 32 * -(-tiles // blocks) + blocks / 8 + 8) * 2.0 ** -24
    err = np.linalg.norm(g - og) / np.linalg.norm(og)
    print(f"[grad n={n} heavy={heavy}] loss off {abs(loss / ol - 1):.2e}, gradient off {err:.2e} (bound {tol:.2e})", flush=True)
    assert abs(loss - ol) <= tol * abs(ol)
    assert err <= tol
