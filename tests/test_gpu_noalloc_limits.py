"""The pairs that fit the fixed scratch of bm4dof_tvl1_noalloc: by an account
that does not depend on the iterations' tiles.  The largest heights of some
widths run and equal bm4dof_tvl1 (no tolerance), the next ones are refused."""
import ctypes as C

import pytest
import torch

from conftest import bm4dof_amd as A, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,fits", [(665, 813, True), (625, 865, True), (641, 843, True), (777, 695, True),
                                      (960, 563, True), (641, 844, False), (777, 696, False), (960, 564, False),
                                      (57, 9, True), (9, 9, True)])
def test_sizes_at_the_limit(ctx, w, h, fits):
    prm = A.TVL1Params(0.25, 0.15, 0.3, 3 if w > 100 else 1, 0, 0.5, 1, 0.01, 0)
    v = synth.add_noise(synth.video(w, h, 2, seed=w), 10, 2)[:, 0]
    d = torch.from_numpy(v).cuda()
    out = torch.zeros((2, h, w), device="cuda")
    torch.cuda.synchronize()
    rc = A.lib().bm4dof_tvl1_noalloc(ctx.h, C.byref(prm), d[0].data_ptr(), d[1].data_ptr(), out[0].data_ptr(),
                                     out[1].data_ptr(), w, h, None)
    assert rc == (0 if fits else -1)
    if fits:
        torch.cuda.synchronize()
        u, v, _ = ctx.tvl1(v[0].copy(), v[1].copy(), lam=0.15, nscales=prm.nscales, warps=1)
        assert (out[0].cpu().numpy() == u).all() and (out[1].cpu().numpy() == v).all()
