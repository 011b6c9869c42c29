"""Which groups the matching by bounded distances keeps: on noise nearly all,
none where no distance can be bounded (a constant image, samples without a
finite range, one sample that leaves the rest few integer steps: those clips
go to the other matcher as a whole), and those with too many candidates left
where part of the image is flat.  The outputs equal the general matcher's
(fast_bm 0; no tolerance).

The clips are large enough for the bounded matching in both steps, which the
statistics confirm; group counts that are no multiple of the lists' number."""
import numpy as np
import pytest

from conftest import bm4dof_amd as A, synth

pytestmark = pytest.mark.gpu


def _clip(kind, f, c):
    v = synth.add_noise(synth.video(243, 205, f, channels=c, n_shapes=9, seed=f + c), 20.0, 3)
    h, w = v.shape[2:]
    if kind == "flat":
        v[:, :, : h // 2] = np.float32(90.0)
    if kind == "constant":
        v[:] = np.float32(0.1)
    if kind == "bad":
        v[0, 0, h // 3, w // 3] = np.nan
        v[-1, -1, h // 2, w // 2] = np.inf
    if kind == "outlier":
        v[0, 0, h // 3, w // 3] = np.float32(1e6)
    return v


@pytest.mark.parametrize("px,pt,np_,wx,f,c", [(4, 4, 16, 11, 6, 1), (4, 4, 8, 9, 8, 3), (8, 1, 32, 39, 1, 1),
                                              (8, 1, 16, 21, 4, 3), (7, 1, 8, 15, 4, 1), (11, 1, 16, 15, 3, 1)])
@pytest.mark.parametrize("kind", ["noise", "flat", "constant", "bad", "outlier"])
def test_groups_left_to_the_other_matcher(ctx, px, pt, np_, wx, f, c, kind):
    noisy = _clip(kind, f, c)
    a1, a2 = (A.cli_params(s, 20.0, noisy.shape, px=px, pt=pt, wx=wx, np_=np_) for s in (1, 2))
    try:
        ctx.set_option("fast_bm", 0)
        b0, f0, _ = ctx.run(a1, a2, noisy, nparts=2)
        s = ctx.stats()
        assert s["bm_redone1"] == -1 and s["bm_redone2"] == -1
    finally:
        ctx.set_option("fast_bm", 2)
    b1, f1, _ = ctx.run(a1, a2, noisy, nparts=2)
    s = ctx.stats()
    assert np.array_equal(b0, b1, equal_nan=True) and np.array_equal(f0, f1, equal_nan=True)
    assert s["chunks1"] == s["chunks2"] == 1
    for step in (1, 2):
        n, left = s["groups%d" % step], s["bm_redone%d" % step]
        # (equal distances can have a colour clip's full grid matched as well)
        if kind == "noise":
            assert 0 <= left <= n // 4
        elif kind == "flat" and step == 1:             # step 2 may shrink its distances
            assert n // 4 <= left and (c > 1 or left <= 3 * n // 4)
        elif kind == "constant" and step == 2:         # constant but for the sums' roundings
            assert left >= n // 2
        elif kind != "flat":
            assert left >= n                           # groups left out of the grid among them
