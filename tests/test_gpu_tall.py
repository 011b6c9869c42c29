"""Images whose places inside a tile need more than 15 bits: the window records
of the one-wave matchers (fast_bm 2) against the general matcher (fast_bm 0),
which has none.  Equal outputs (no tolerance).  Beyond 16 bits the general
matcher takes every shape."""
import numpy as np
import pytest

from conftest import bm4dof_amd as A, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(24, 33011), (33011, 24), (20, 65536)])
@pytest.mark.parametrize("px,pt,np_,wx", [(7, 1, 8, 15), (11, 1, 16, 9), (8, 1, 16, 27)])
def test_places_of_sixteen_bits(ctx, w, h, px, pt, np_, wx):
    small = synth.add_noise(synth.video(min(w, 500), min(h, 500), 1, n_shapes=9, seed=px), 20.0, 3)
    noisy = np.ascontiguousarray(np.tile(small, (1, 1, -(-h // small.shape[2]), -(-w // small.shape[3])))[:, :, :h, :w])
    rng = np.random.default_rng(w + px)
    noisy += rng.normal(0, 2, noisy.shape).astype(np.float32)
    a1, a2 = (A.cli_params(s, 20.0, noisy.shape, px=px, pt=pt, wx=wx, np_=np_) for s in (1, 2))
    try:
        ctx.set_option("fast_bm", 0)
        b0, f0, _ = ctx.run(a1, a2, noisy, nparts=1)
        ctx.set_option("fast_bm", 2)
        b1, f1, _ = ctx.run(a1, a2, noisy, nparts=1)
    finally:
        ctx.set_option("fast_bm", 2)
    assert np.array_equal(b0, b1) and np.array_equal(f0, f1)
