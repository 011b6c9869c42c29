"""Matching by bounded distances (fast_bm 2) against the general matcher
(fast_bm 0), which sums every candidate's distance: a bound only leaves out
candidates that cannot be among the nearest, so the outputs are equal (no
tolerance).

The clips put the bound where it could go wrong: 8-bit samples and flat areas
(ties, and groups that keep more candidates than the list holds), a constant
image and values without a finite range (no bound at all), ranges at the ends
of what the integer samples take, a small range on a large offset, and one
outlier that leaves the rest a few integer steps."""
import functools

import numpy as np
import pytest

from conftest import bm4dof_amd as A, synth

pytestmark = pytest.mark.gpu


@functools.lru_cache(maxsize=None)
def _noisy(f, c):
    # large enough for the bounded matching to be taken in both steps
    return synth.add_noise(synth.video(176, 161, f, channels=c, n_shapes=9, seed=f + c), 20.0, 3)


def _clip(kind, f, c):
    v = _noisy(f, c).copy()
    h, w = v.shape[2:]
    if kind == "u8":
        return np.clip(np.round(v), 0, 255).astype(np.float32)
    if kind == "flat":
        v[:, :, : h // 2] = np.float32(90.0)
    if kind == "constant":
        v[:] = np.float32(0.1)
    if kind == "bad":
        v[0, 0, h // 3, w // 3] = np.nan
        v[-1, -1, h // 2, w // 2] = np.inf
    if kind == "outlier":
        v[0, 0, h // 3, w // 3] = np.float32(1e6)
    if kind == "offset":
        v = v + np.float32(65536.0)
    if kind in ("huge", "tiny", "vast"):
        v = v * np.float32({"huge": 1e16, "tiny": 1e-19, "vast": 3e33}[kind])
    return np.ascontiguousarray(v, dtype=np.float32)


@pytest.mark.parametrize("px,pt,np_,wx,f,c", [(4, 4, 32, 11, 7, 1), (4, 4, 16, 15, 6, 3), (4, 4, 8, 7, 8, 1),
                                              (8, 1, 32, 39, 1, 1), (8, 1, 16, 15, 4, 3), (7, 1, 8, 15, 4, 1),
                                              (7, 1, 64, 27, 1, 3), (11, 1, 16, 13, 3, 1), (11, 1, 8, 39, 1, 3)])
@pytest.mark.parametrize("kind", ["noise", "u8", "flat", "constant", "bad", "outlier", "offset", "huge", "tiny", "vast"])
def test_bounded_matching_equals_the_general_matcher(ctx, px, pt, np_, wx, f, c, kind):
    noisy = _clip(kind, f, c)
    a1, a2 = (A.cli_params(s, 20.0, noisy.shape, px=px, pt=pt, wx=wx, np_=np_) for s in (1, 2))
    try:
        ctx.set_option("fast_bm", 0)
        b0, f0, _ = ctx.run(a1, a2, noisy, nparts=2)
        ctx.set_option("fast_bm", 2)
        b1, f1, _ = ctx.run(a1, a2, noisy, nparts=2)
    finally:
        ctx.set_option("fast_bm", 2)
    assert np.array_equal(b0, b1, equal_nan=True) and np.array_equal(f0, f1, equal_nan=True)
