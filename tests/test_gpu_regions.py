"""The region fold of the binned aggregation (agg_region_fold_kernel) against
the per-frame chunked aggregation (option agg_binned 0), which sorts the rows
of every block itself: both add the same float terms in the same order, so
the outputs are equal bit for bit (no tolerance).

Shapes: patches of one frame that are no multiple of the wave (7x7, 5x5),
that take two and four sample slots per lane (11x11, 15x15) and that have an
aggregation window (10x10); 4x4x4 patches in regions of many frames, with
more frames than a region has, in colour, and tiles whose borders cut
regions."""
import numpy as np
import pytest

from conftest import bm4dof_amd as A, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,f,c,nparts,px,pt,np_", [
    (61, 45, 5, 1, 4, 7, 1, 8), (50, 38, 3, 1, 6, 5, 1, 16), (75, 59, 1, 1, 2, 11, 1, 32),
    (70, 64, 2, 1, 4, 15, 1, 8), (66, 52, 1, 1, 2, 10, 1, 16), (58, 44, 2, 3, 2, 11, 1, 8),
    (57, 49, 2, 4, 2, 7, 1, 8), (331, 310, 5, 1, 4, 4, 4, 16), (317, 319, 34, 1, 2, 4, 4, 8),
    (320, 312, 6, 3, 4, 4, 4, 8)])
def test_region_fold_equals_the_chunked_aggregation(ctx, w, h, f, c, nparts, px, pt, np_):
    rng = np.random.default_rng(w * h + px)
    noisy = synth.add_noise(synth.video(w, h, f, channels=c, n_shapes=6, seed=px), 20, px + 1)
    ff = bf = None
    if f > 1:
        ff, bf = (rng.uniform(-2, 2, (f, 2, h, w)).astype(np.float32) for _ in range(2))
    a1, a2 = (A.cli_params(s, 20, noisy.shape, px=px, pt=pt, wx=7, np_=np_) for s in (1, 2))
    try:
        ctx.set_option("agg_binned", 0)
        b0, f0, _ = ctx.run(a1, a2, noisy, ff, bf, nparts=nparts)
        assert ctx.stats()["agg_bt"] == 1
    finally:
        ctx.set_option("agg_binned", 1)
    b1, f1, _ = ctx.run(a1, a2, noisy, ff, bf, nparts=nparts)
    big = w * h > 300 * 300
    assert ctx.stats()["agg_bt"] == ((16 if c > 1 else 32) if big else 1)
    assert np.array_equal(b0, b1, equal_nan=True) and np.array_equal(f0, f1, equal_nan=True)


@pytest.mark.parametrize("w,h,f,c,px,pt,np_", [
    (41, 33, 4, 1, 4, 4, 32), (57, 39, 7, 3, 4, 4, 8), (33, 30, 1, 1, 8, 1, 16), (73, 41, 5, 4, 8, 1, 8),
    (37, 50, 2, 1, 7, 1, 8), (47, 35, 1, 3, 11, 1, 8), (49, 33, 1, 1, 15, 1, 4),      # four waves a region
    (296, 296, 9, 1, 4, 4, 8), (441, 440, 1, 1, 8, 1, 8), (460, 430, 4, 1, 7, 1, 4)])  # one
@pytest.mark.parametrize("flat", [False, True])
def test_split_regions_equal_the_chunked_aggregation(ctx, w, h, f, c, px, pt, np_, flat):
    """Few regions: four waves share a region's list; flat areas make lists of
    one place, and rows that miss a quarter."""
    noisy = synth.add_noise(synth.video(w, h, f, channels=c, n_shapes=6, seed=px), 20, px + 1)
    if flat:
        noisy[:, :, 5:, : w // 2] = np.float32(40.0)
    a1, a2 = (A.cli_params(s, 20, noisy.shape, px=px, pt=pt, wx=7, np_=np_) for s in (1, 2))
    try:
        ctx.set_option("agg_binned", 0)
        b0, f0, _ = ctx.run(a1, a2, noisy, nparts=2)
    finally:
        ctx.set_option("agg_binned", 1)
    b1, f1, _ = ctx.run(a1, a2, noisy, nparts=2)
    assert np.array_equal(b0, b1, equal_nan=True) and np.array_equal(f0, f1, equal_nan=True)
