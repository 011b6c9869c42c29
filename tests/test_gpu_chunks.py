"""A step whose groups are filtered and aggregated in several chunks (option
est_budget) against the same step in one: the sums of a region go on where the
chunk before left them, in the same order, so the outputs are equal (no
tolerance).  Groups of equal patches take the weight that groups of an earlier
chunk left; several channels' weights are applied by the fold (default), by
the filters (agg_binned 0), or by the general filter (fast_filter 0)."""
import numpy as np
import pytest

from conftest import bm4dof_amd as A, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("px,pt,np_,f,c", [(4, 4, 16, 6, 1), (4, 4, 16, 6, 3), (8, 1, 32, 2, 1), (8, 1, 8, 2, 4),
                                           (7, 1, 8, 2, 1), (7, 1, 16, 2, 3), (11, 1, 16, 1, 1), (11, 1, 8, 1, 3)])
@pytest.mark.parametrize("opt", [None, "agg_binned", "fast_filter"])
def test_chunks_equal_one(px, pt, np_, f, c, opt):
    noisy = synth.add_noise(synth.video(63, 50, f, channels=c, n_shapes=5, seed=np_ + px), 15.0, px + c)
    noisy[:, :, :24, 5:34] = np.float32(77.0)     # equal patches: written raw
    a1 = A.cli_params(1, 15.0, noisy.shape, px=4 if f >= 4 else 8, pt=4 if f >= 4 else 1, wx=9, np_=8)
    a2 = A.cli_params(2, 15.0, noisy.shape, px=px, pt=pt, wx=9, np_=np_)
    out = []
    for chunks in (1, 3, 7):
        ctx = A.Context(0)
        try:
            if opt:
                ctx.set_option(opt, 0)
            if chunks > 1:
                # step 2's groups, its rows' bytes, in `chunks` parts and a rest
                row = c * px * px * pt * 4
                ctx.set_option("est_budget", max(1, (groups - 1) // chunks) * np_ * row)
            out.append(ctx.run(a1, a2, noisy, nparts=2)[:2])
            s = ctx.stats()
            groups = s["groups2"]
            assert s["chunks2"] == 1 if chunks == 1 else s["chunks2"] > chunks
        finally:
            ctx.close()
    for b, o in out[1:]:
        assert np.array_equal(out[0][0], b, equal_nan=True) and np.array_equal(out[0][1], o, equal_nan=True)
    assert np.isfinite(out[0][1]).mean() > 0.5     # (colour: no number where no patch lies)


def test_last_chunk_of_a_captured_step():
    """A last chunk of 131075 rows takes as many sort tiles of the smallest
    size as a chunk may have; the buffers were sized for a larger first chunk,
    whose tiles are larger and half as many.  Nothing may grow in a capture."""
    import torch
    noisy = torch.from_numpy(synth.add_noise(synth.video(81, 81, 1, n_shapes=6, seed=4), 20.0, 5)).cuda()
    p1, p2 = (A.cli_params(s, 20.0, noisy.shape, px=8, pt=1, wx=9, np_=49) for s in (1, 2))
    p1.offSet = p2.offSet = 1
    one = [torch.zeros_like(noisy) for _ in range(2)]
    many = [torch.zeros_like(noisy) for _ in range(2)]
    torch.cuda.synchronize()
    ctx = A.Context(0)
    try:
        ctx.run_dev(p1, p2, noisy.data_ptr(), noisy.shape, None, None, one[0].data_ptr(), one[1].data_ptr(), nparts=1)
        groups = ctx.stats()["groups1"]
        assert groups == ctx.stats()["groups2"] and 2 * 2675 < groups < 2675 + 5350
    finally:
        ctx.close()
    ctx = A.Context(0)
    try:
        ctx.set_option("est_budget", (groups - 2675) * 49 * 64 * 4)
        seq = A.Seq(noisy.data_ptr(), None, None, many[0].data_ptr(), many[1].data_ptr(), 81, 81, 1)
        batch = ctx.batch([seq], [p1], [p2], nparts=1, graph=True)
        for _ in range(3):
            for m in many:
                m.zero_()
            torch.cuda.synchronize()
            batch.run()
            torch.cuda.synchronize()
            for a, b in zip(one, many):
                assert torch.equal(a, b)
        batch.close()
    finally:
        ctx.close()
