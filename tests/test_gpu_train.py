"""Training kernels (mlp_rows / mlp_wgrad / mlp_update) at the edges of their
blocks of 16 rows and splits of 128: loss and gradient against the float64
oracle, and Adam steps on batches drawn from a larger set against the same
steps on those rows taken as a whole set.

Tolerances: fp32 accumulation moves a layer input across a bfloat16 rounding
boundary now and then, worth 2^-9 of one input of one row: at most 1e-3 of a
one-row gradient's norm, and 1e-5 of the loss for the squared error's slope.
The drawn batch and its rows in order are the same launches on the same
values: bitwise equal."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import mlp_oracle as M  # noqa: E402

pytestmark = pytest.mark.gpu


def _rows(n, seed):
    rng = np.random.default_rng(seed)
    x = rng.normal(0, 1.5, (n, 66)).astype(np.float32)
    return x, rng.uniform(0, 1, (n, 64)).astype(np.float32)


@pytest.mark.parametrize("rows", [1, 15, 16, 17, 127, 128, 129, 273, 8193])
def test_gradient_at_block_and_split_edges(ctx, rows):
    theta = M.init_params(rows)
    x, t = _rows(rows, rows + 1)
    ctx.mlp_set(theta)
    loss, g = ctx.mlp_grad(x, t)
    lref, gref = M.backward(theta.astype(np.float64), x.astype(np.float64), t.astype(np.float64))
    assert np.linalg.norm(g - gref) <= 1e-3 * np.linalg.norm(gref)
    assert abs(loss - lref) <= 1e-5 * lref


@pytest.mark.parametrize("batch,rows", [(33, 500), (160, 161)])
def test_drawn_batches_are_their_rows(ctx, batch, rows):
    import torch
    theta = M.init_params(5)
    x, t = _rows(rows, 6)
    dx, dt = torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda()
    torch.cuda.synchronize()
    ctx.mlp_set(theta)
    la = ctx.mlp_train_dev(dx.data_ptr(), dt.data_ptr(), rows, batch, 1, 1e-3, seed=9)
    a = ctx.mlp_get()
    low = (np.arange(batch, dtype=np.uint64) * np.uint64(2654435761) + np.uint64(0x9E3779B9)) & np.uint64(0xFFFFFFFF)
    with np.errstate(over="ignore"):
        s = (np.uint64(9) << np.uint64(32)) ^ low
        s = s * np.uint64(6364136223846793005) + np.uint64(1442695040888963407)
        s ^= s >> np.uint64(33)
        s *= np.uint64(0xff51afd7ed558ccd)
        s ^= s >> np.uint64(33)
    pick = (s % np.uint64(rows)).astype(np.int64)
    dx2, dt2 = dx[pick].contiguous(), dt[pick].contiguous()
    torch.cuda.synchronize()
    ctx.mlp_set(theta)
    lb = ctx.mlp_train_dev(dx2.data_ptr(), dt2.data_ptr(), batch, batch, 1, 1e-3)
    assert np.array_equal(la, lb) and np.array_equal(a, ctx.mlp_get())
    assert not np.array_equal(a, theta)
