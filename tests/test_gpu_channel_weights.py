"""Several channels: where the region fold sums the rows it applies their
weight itself to all channels but the last (the filters then store those
unweighted), the chunked fold (agg_binned 0) and the general filters
(fast_filter 0) read weighted rows.  The products and the order of the sums
are the same, so the outputs are equal (no tolerance).  Groups of equal
patches are weighted by a pass of their own, in one chunk of groups or in
many (est_budget)."""
import numpy as np
import pytest

from conftest import bm4dof_amd as A, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("c", [3, 4])
@pytest.mark.parametrize("px,pt,np_,f", [(4, 4, 16, 6), (8, 1, 32, 2), (7, 1, 8, 2), (11, 1, 16, 1)])
def test_weights_in_the_fold_equal_weighted_rows(c, px, pt, np_, f):
    noisy = synth.add_noise(synth.video(61, 50, f, channels=c, n_shapes=5, seed=np_ + px), 15.0, px + c)
    noisy[:, :, :22, 5:30] = np.float32(77.0)     # equal patches: written raw
    a1 = A.cli_params(1, 15.0, noisy.shape, px=4 if f >= 4 else 8, pt=4 if f >= 4 else 1, wx=9, np_=8)
    a2 = A.cli_params(2, 15.0, noisy.shape, px=px, pt=pt, wx=9, np_=np_)
    out = []
    for opts in ({}, {"coef_budget": 0}, {"agg_binned": 0}, {"fast_filter": 0}):
        ctx = A.Context(0)
        try:
            for k, v in opts.items():
                ctx.set_option(k, v)
            out.append(ctx.run(a1, a2, noisy, nparts=2)[:2])
        finally:
            ctx.close()
    for b, o in out[1:]:
        assert np.array_equal(out[0][0], b, equal_nan=True) and np.array_equal(out[0][1], o, equal_nan=True)
