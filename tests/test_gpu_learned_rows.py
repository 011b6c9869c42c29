"""The learned filter's way from samples to rows with a network of known
gains: all weights 0, so every gain is the sigmoid of its bias.  Equal gains
commute with the transforms, so the pass is linear in the gain, and with a
basis that its inverse undoes (4x4x4) it gives the gain times the input, where
patches were taken (pixels in no patch of a group get 0 over the input).

Tolerance: samples and coefficients are split in two halves of 11 bits and so
are the bases, four roundings of 2^-22 on values that add up over a patch's 64
samples as independent errors, times the 1.6 an 8x8 biorthogonal basis can
stretch them, and float sums of a few hundred rows: below 64 * 2^-22 of the
largest value."""
import numpy as np
import pytest

from conftest import bm4dof_amd as A, synth
from oracle import mlp_oracle as M

pytestmark = pytest.mark.gpu


def _theta(bias):
    d = M.unpack(np.zeros(M.N_PARAMS, np.float32))
    d["b3"][:] = bias
    return M.pack(d).astype(np.float32)


@pytest.fixture(scope="module")
def own():
    c = A.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("px,pt,np_,f,c", [(4, 4, 1, 4, 1), (4, 4, 2, 5, 1), (4, 4, 32, 7, 1), (4, 4, 8, 5, 3),
                                           (8, 1, 16, 1, 1), (8, 1, 32, 3, 1), (8, 1, 4, 2, 4)])
@pytest.mark.parametrize("scale,shift", [(1.0, 0.0), (1e4, 0.0), (1e-4, 0.0), (1.0, 3000.0)])
def test_equal_gains_scale_the_input(own, px, pt, np_, f, c, scale, shift):
    noisy = synth.add_noise(synth.video(45, 39, f, channels=c, n_shapes=5, seed=px + np_), 20.0, 3)
    noisy = (noisy * np.float32(scale) + np.float32(shift)).astype(np.float32)
    noisy[:, :, 3:12, 4:14] = noisy[0, 0, 0, 0]          # equal patches
    p1 = A.cli_params(1, 20.0 * scale, noisy.shape, px=px, pt=pt, wx=7, np_=np_)
    own.mlp_set(_theta(40.0))            # gains 1
    one, _ = own.run_learned(p1, None, noisy)
    own.mlp_set(_theta(0.0))             # gains 1/2
    half, _ = own.run_learned(p1, None, noisy)
    tol = 64 * 2.0 ** -22 * np.abs(noisy).max()
    taken = np.nan_to_num(one) != 0
    assert taken.mean() > 0.8
    assert np.array_equal(np.isnan(half), np.isnan(one))
    assert np.abs(half - 0.5 * one.astype(np.float64))[taken].max() < tol
    if px == 4:
        assert np.abs(one - noisy.astype(np.float64))[taken].max() < tol
