"""TV-L1 with samples that are no number or infinite, and with denominators
beyond 2^126, against the CPU oracle: where the gradient is zero the update
takes nothing from such a sample (tvl1flow_lib.c:186-200), elsewhere it spreads
as the formulas have it.  Equal values, and no number where the oracle has
none."""
import numpy as np
import pytest

import oracle as O
from conftest import bm4dof_amd as A  # noqa: F401

pytestmark = pytest.mark.gpu


def _pair(kind, w, h):
    rng = np.random.default_rng(w)
    I0 = rng.uniform(0, 255, (h, w)).astype(np.float32)
    I1 = np.roll(I0, 1, 1).copy()
    if kind.startswith("flat"):       # no gradient of the second frame around the sample
        I1[:, 30:] = 100.0
        I0[:, 30:] = 101.0
    if kind == "large":
        return I0 * np.float32(1e30), I1 * np.float32(1e30)
    if not kind.endswith("none"):
        I0[h // 2, 60] = {"nan": np.nan, "inf": np.inf, "-inf": -np.inf}[kind.split("_")[1]]
    return I0, I1


@pytest.mark.parametrize("kind", ["flat_nan", "flat_inf", "flat_-inf", "texture_nan", "texture_inf", "large"])
@pytest.mark.parametrize("w,h", [(80, 64), (117, 33)])
def test_samples_that_are_no_number(ctx, kind, w, h):
    I0, I1 = _pair(kind, w, h)
    kw = dict(nscales=1, warps=2)
    u, v, it = ctx.tvl1(I0, I1, **kw)
    uo, vo, ito = O.tvl1(I0, I1, **kw)
    assert np.array_equal(it, ito)
    assert np.array_equal(u, uo, equal_nan=True) and np.array_equal(v, vo, equal_nan=True)


@pytest.mark.parametrize("kind", ["flat_none", "texture_none"])
@pytest.mark.parametrize("lam,theta", [(1.6e37, 6e-38), (1e37, 0.3), (1e30, 1e-30)])
def test_denominators_beyond_the_float_reciprocal(ctx, kind, lam, theta):
    """Weights that send u and the gradients' norms to the ends of the floats."""
    I0, I1 = _pair(kind, 80, 64)
    kw = dict(nscales=1, warps=1, lam=lam, theta=theta)
    u, v, it = ctx.tvl1(I0, I1, **kw)
    uo, vo, ito = O.tvl1(I0, I1, **kw)
    assert np.array_equal(it, ito)
    assert np.array_equal(u, uo, equal_nan=True) and np.array_equal(v, vo, equal_nan=True)
