"""The coefficient tables' memory between calls: it stays allocated and idle
(a call allocates nothing once its shape has run), any context of the device
takes it, and setting a coef_budget gives it back.  Device memory is read as
the runtime reports it, in steps of 2 MiB and per buffer; the tables are 36 MB
each."""
import numpy as np
import pytest
import torch

from conftest import bm4dof_amd as A, synth

pytestmark = pytest.mark.gpu

SHAPE = (6, 1, 136, 176)
TABLE = 6 * 136 * 176 * 64 * 4
SLACK = 16 << 20


def _free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_tables_stay_idle_between_calls_and_go_back():
    noisy = synth.add_noise(synth.video(176, 136, 6, n_shapes=6, seed=2), 20.0, 3)
    assert noisy.shape == SHAPE
    p1, p2 = (A.cli_params(s, 20.0, noisy.shape, px=4, pt=4, wx=7, np_=8) for s in (1, 2))
    made = []

    def context(budget=None):
        c = A.Context(0)
        made.append(c)
        if budget is not None:
            c.set_option("coef_budget", budget)       # nothing idle from here on
        return c

    try:
        warm = context(0)                             # code objects, flow scratch
        b0, f0, _ = warm.run(p1, p2, noisy, nparts=2)
        c = context(0)
        before = _free()
        c.run(p1, p2, noisy, nparts=2)
        other = before - _free()                      # what a run takes beside the tables

        a = context()
        before = _free()
        b1, f1, _ = a.run(p1, p2, noisy, nparts=2)
        first = _free()
        assert before - first >= other + 2 * TABLE - SLACK
        for _ in range(3):
            a.run(p1, p2, noisy, nparts=2)
            assert _free() == first
        b = context()
        before = _free()
        b2, f2, _ = b.run(p1, p2, noisy, nparts=2)
        assert before - _free() <= other + SLACK      # the same tables
        before = _free()
        a.set_option("coef_budget", 96 << 30)
        assert _free() - before >= 2 * TABLE - SLACK
        b3, f3, _ = a.run(p1, p2, noisy, nparts=2)
        for x, y in ((b1, f1), (b2, f2), (b3, f3)):
            assert np.array_equal(b0, x) and np.array_equal(f0, y)
        a.set_option("coef_budget", 3 * TABLE)        # two tables fit, and may stay idle
        before = _free()
        a.run(p1, p2, noisy, nparts=2)
        assert before - _free() >= 2 * TABLE - SLACK
        small = synth.add_noise(synth.video(150, 136, 6, n_shapes=6, seed=2), 20.0, 3)
        before = _free()
        a.set_option("coef_budget", TABLE * 175 // 100)   # two of the smaller clip's
        a.run(p1, p2, small, nparts=2)
        a.run(p1, p2, noisy, nparts=2)                # only step 1's table fits: it displaces those
        assert abs(_free() - before - TABLE) <= SLACK  # of the two blocks before one is left
        a.set_option("keep_tables", 1)                # with the context: not idle
        a.run(p1, p2, noisy, nparts=2)
        before = _free()
        b.set_option("coef_budget", 96 << 30)
        assert _free() - before < SLACK
    finally:
        for c in made:
            c.close()


def test_contexts_on_threads_share_idle_tables():
    """Two contexts, each on its own thread, on clips of different sizes in turn:
    the blocks change hands between calls."""
    import threading
    clips = [synth.add_noise(synth.video(w, 60, 6, n_shapes=5, seed=w), 20.0, 3) for w in (72, 96, 140)]
    prm = [[A.cli_params(s, 20.0, v.shape, px=4, pt=4, wx=7, np_=8) for s in (1, 2)] for v in clips]
    ctxs = [A.Context(0) for _ in range(2)]
    try:
        want = [ctxs[0].run(*p, v, nparts=2)[:2] for p, v in zip(prm, clips)]
        wrong = []

        def go(k):
            for i in range(12):
                j = (i * (k + 1) + k) % 3
                b, f, _ = ctxs[k].run(*prm[j], clips[j], nparts=2)
                if not (np.array_equal(b, want[j][0]) and np.array_equal(f, want[j][1])):
                    wrong.append((k, i))

        threads = [threading.Thread(target=go, args=(k,)) for k in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join(60)
        assert not wrong and not any(t.is_alive() for t in threads)
    finally:
        for c in ctxs:
            c.close()
