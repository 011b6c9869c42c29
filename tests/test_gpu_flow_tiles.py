"""The TV-L1 iteration blocks at the edges of their tiles (56 x 8 pixels for a
single pair, 56 x 24 for many) against the CPU oracle.  With epsilon 0 every
solve runs its 300 iterations, so the flows are equal (no tolerance; zero
updates end both at the same count); with epsilon 0.01 the stopping test
decides, and where the counts agree the flows are equal."""
import numpy as np
import pytest

import oracle as O
from conftest import bm4dof_amd as A, synth

pytestmark = pytest.mark.gpu


def _frames(w, h, n, kind):
    f = synth.add_noise(synth.video(w, h, n, n_shapes=4, seed=w + h), 10.0, 5)[:, 0]
    if kind == "flat":      # no gradient in half of the image
        f[:, :, : w // 2] = np.float32(64.0)
    if kind == "still":     # no difference at all
        f[:] = f[0]
    return np.ascontiguousarray(f)


@pytest.mark.parametrize("w,h", [(20, 17), (55, 7), (56, 8), (57, 9), (60, 24), (64, 25), (113, 31), (52, 48), (117, 33)])
@pytest.mark.parametrize("kind", ["noise", "flat", "still"])
@pytest.mark.parametrize("eps", [0.0, 0.01])
def test_single_pair_tiles(ctx, w, h, kind, eps):
    I0, I1 = _frames(w, h, 2, kind)
    kw = dict(nscales=1, warps=2, eps=eps)
    u, v, it = ctx.tvl1(I0, I1, **kw)
    uo, vo, ito = O.tvl1(I0, I1, **kw)
    assert np.abs(it - ito).max() <= (1 if eps else 0)
    if np.array_equal(it, ito):
        assert np.array_equal(u, uo) and np.array_equal(v, vo)


@pytest.mark.parametrize("w,h", [(57, 25), (56, 24), (113, 23), (60, 49)])
def test_many_pair_tiles(ctx, w, h):
    tiles = -(-w // 56) * -(-h // 24)
    n = 512 // tiles // 2 + 2          # 2 (n - 1) pairs: the larger tiles
    f = _frames(w, h, 8, "noise")
    f = np.ascontiguousarray(f[np.arange(n) % 8])
    kw = dict(nscales=1, warps=1, eps=0.0)
    ff, bf = ctx.tvl1_sequence(f, **kw)
    for i in range(3):
        uo, vo, _ = O.tvl1(f[i], f[i + 1], **kw)
        assert np.array_equal(ff[i, 0], uo) and np.array_equal(ff[i, 1], vo)
        uo, vo, _ = O.tvl1(f[i + 1], f[i], **kw)
        assert np.array_equal(bf[i + 1, 0], uo) and np.array_equal(bf[i + 1, 1], vo)
    for i in range(8, n - 1):          # the same frames again
        assert np.array_equal(ff[i], ff[i - 8]) and np.array_equal(bf[i + 1], bf[i - 7])
