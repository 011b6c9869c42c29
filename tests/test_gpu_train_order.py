"""The training step's sums are sequential: over a layer's inputs or outputs
and over the batch's rows, one fused multiply-add a term in increasing order
(a bias gradient: one addition a row).  The gradient is compared bit for bit
(no tolerance) with those sums taken term by term on the CPU: a product of a
bfloat16 value and a float has 32 bits, so it and its sum with a float are
formed in 64 bits and rounded to float once.

The gradient at the outputs, which has the sigmoid in it, comes from batches
of one row: its only sum over rows is the bias gradient, and for a batch of a
power of two rows it is that divided by the row count, exactly."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import mlp_oracle as M  # noqa: E402

pytestmark = pytest.mark.gpu


def _chain(a, b):
    """s[m][n] = the terms a[k][m] b[k][n] in the order of k."""
    s = np.zeros((a.shape[1], b.shape[1]), np.float32)
    for k in range(a.shape[0]):
        s = (a[k].astype(np.longdouble)[:, None] * b[k].astype(np.longdouble)[None, :] + s).astype(np.float32)
    return s


def _relu(z):
    return M.bf16_round(np.maximum(z, np.float32(0))).astype(np.float32)


@pytest.mark.parametrize("rows", [2, 16, 64, 256])
def test_gradient_sums_are_sequential(ctx, rows):
    rng = np.random.default_rng(rows)
    theta = M.init_params(rows + 1)
    theta += rng.normal(0, 0.05, theta.shape).astype(np.float32)     # biases too
    x = rng.normal(0, 1.5, (rows, 66)).astype(np.float32)
    t = rng.uniform(0, 1, (rows, 64)).astype(np.float32)
    ctx.mlp_set(theta)
    _, got = ctx.mlp_grad(x, t)
    d3 = np.stack([ctx.mlp_grad(x[r:r + 1], t[r:r + 1])[1][-64:] for r in range(rows)]) / np.float32(rows)

    p = {k: v.astype(np.float32) for k, v in M.unpack(theta).items()}
    w1, w2, w3 = (M.bf16_round(p[k]).astype(np.float32) for k in ("W1", "W2", "W3"))
    x0 = M.bf16_round(x).astype(np.float32)
    z1 = _chain(x0.T, w1) + p["b1"]
    h1 = _relu(z1)
    z2 = _chain(h1.T, w2) + p["b2"]
    h2 = _relu(z2)
    d2 = np.where(z2 > 0, _chain(d3.T, w3.T), np.float32(0))
    d1 = np.where(z1 > 0, _chain(d2.T, w2.T), np.float32(0))
    one = np.ones((rows, 1), np.float32)
    want = np.concatenate([v.ravel() for h, d in ((x0, d1), (h1, d2), (h2, d3)) for v in (_chain(h, d), _chain(one, d))])
    assert want.dtype == np.float32 and np.count_nonzero(want) > 0.5 * want.size
    assert np.array_equal(got, want)
