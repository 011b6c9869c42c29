"""Step 2 without shrinkage (beta 0: every gain is y^2 / y^2 = 1, and 0 / 0 only
where a coefficient of the patch itself is 0) by the register filters against
the general filter (fast_filter 0), with patches that leave lanes without a
sample.  Equal outputs (no tolerance), and finite ones: on noise no
coefficient is 0."""
import numpy as np
import pytest

from conftest import bm4dof_amd as A, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("px,pt,np_,f,c", [(px, pt, np_, f, c) for px, pt, np_, f in (
    (7, 1, 8, 3), (7, 1, 16, 1), (7, 1, 32, 2), (9, 1, 16, 2), (10, 1, 32, 1), (11, 1, 16, 1), (11, 1, 32, 2),
    (5, 3, 8, 4), (8, 1, 16, 2), (4, 4, 32, 5)) for c in (1, 3)
    if (c + 2) * px * px * pt * np_ <= 16384])    # larger groups are refused
def test_beta_zero(ctx, px, pt, np_, f, c):
    noisy = synth.add_noise(synth.video(48, 41, f, channels=c, n_shapes=5, seed=np_ + px), 20.0, px + 1)
    a1 = A.cli_params(1, 20.0, noisy.shape, px=8, pt=1, wx=9, np_=8)
    a2 = A.cli_params(2, 20.0, noisy.shape, px=px, pt=pt, wx=9, np_=np_)
    a2.beta = 0.0
    try:
        ctx.set_option("fast_filter", 0)
        _, f0, _ = ctx.run(a1, a2, noisy, nparts=2)
        ctx.set_option("fast_filter", 1)
        _, f1, _ = ctx.run(a1, a2, noisy, nparts=2)
        ctx.set_option("coef_budget", 0)
        _, f2, _ = ctx.run(a1, a2, noisy, nparts=2)
    finally:
        ctx.set_option("fast_filter", 1)
        ctx.set_option("coef_budget", 96 << 30)
    assert np.array_equal(f0, f1, equal_nan=True) and np.array_equal(f0, f2, equal_nan=True)
    assert np.isfinite(f0).all()
