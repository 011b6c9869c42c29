"""The register filters (fast_filter 1, with and without the coefficient
tables) against the general ones (fast_filter 0), which sum and transform
term by term: the matrix instructions add their terms in order and the sum of
the squared gains is the sequential one bit for bit, so the outputs are equal
(no tolerance).

The noise levels put the sum of squared gains where a folded sum could come
out otherwise: gains that round to one or sit just below it (sigma 0.05 and
1: ties at every power of two), gains near zero (sigma 200), and 8-bit
samples, whose coefficients are coarse."""
import numpy as np
import pytest

from conftest import bm4dof_amd as A, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("px,pt,np_,f,c", [(4, 4, 32, 6, 1), (4, 4, 16, 5, 3), (4, 4, 8, 7, 1), (8, 1, 32, 1, 1),
                                           (8, 1, 16, 2, 4), (8, 1, 8, 3, 1), (4, 4, 2, 5, 1), (7, 1, 8, 3, 1),
                                           (7, 1, 32, 2, 3), (7, 1, 4, 2, 1)])
@pytest.mark.parametrize("sigma,u8", [(0.05, False), (1.0, False), (20.0, True), (200.0, False)])
def test_register_filters_equal_the_general_ones(ctx, px, pt, np_, f, c, sigma, u8):
    noisy = synth.add_noise(synth.video(52, 44, f, channels=c, n_shapes=5, seed=np_), sigma, px + 1)
    if u8:
        noisy = np.clip(np.round(noisy), 0, 255).astype(np.float32)
    a1, a2 = (A.cli_params(s, sigma, noisy.shape, px=px, pt=pt, wx=9, np_=np_) for s in (1, 2))
    try:
        ctx.set_option("fast_filter", 0)
        b0, f0, _ = ctx.run(a1, a2, noisy, nparts=2)
        ctx.set_option("fast_filter", 1)
        b1, f1, _ = ctx.run(a1, a2, noisy, nparts=2)
        ctx.set_option("coef_budget", 0)
        b2, f2, _ = ctx.run(a1, a2, noisy, nparts=2)
    finally:
        ctx.set_option("fast_filter", 1)
        ctx.set_option("coef_budget", 96 << 30)
    for b, o in ((b1, f1), (b2, f2)):
        assert np.array_equal(b0, b, equal_nan=True) and np.array_equal(f0, o, equal_nan=True)


@pytest.mark.parametrize("px,pt,np_,f,c", [(11, 1, 16, 1, 1), (11, 1, 32, 2, 1), (11, 1, 8, 1, 3), (9, 1, 32, 2, 1),
                                           (5, 3, 16, 4, 1), (6, 3, 16, 6, 3), (8, 2, 8, 3, 4), (6, 2, 2, 3, 1),
                                           (10, 1, 4, 1, 1), (6, 3, 24, 6, 1)])
@pytest.mark.parametrize("sigma,u8", [(0.05, False), (1.0, False), (20.0, True), (200.0, False)])
def test_wide_filter_equals_the_general_one(ctx, px, pt, np_, f, c, sigma, u8):
    """Second-step patches of 65 to 128 samples, odd and even counts."""
    noisy = synth.add_noise(synth.video(47, 40, f, channels=c, n_shapes=5, seed=np_ + px), sigma, px + 1)
    noisy[:, :, :20, :20] = np.float32(77.0)      # equal patches: written raw
    if u8:
        noisy = np.clip(np.round(noisy), 0, 255).astype(np.float32)
    a1 = A.cli_params(1, sigma, noisy.shape, px=4 if f >= 4 else 8, pt=4 if f >= 4 else 1, wx=9, np_=8)
    a2 = A.cli_params(2, sigma, noisy.shape, px=px, pt=pt, wx=9, np_=np_)
    try:
        ctx.set_option("fast_filter", 0)
        _, f0, _ = ctx.run(a1, a2, noisy, nparts=2)
        ctx.set_option("fast_filter", 1)
        _, f1, _ = ctx.run(a1, a2, noisy, nparts=2)
    finally:
        ctx.set_option("fast_filter", 1)
    assert np.array_equal(f0, f1, equal_nan=True)
