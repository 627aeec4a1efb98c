"""Contexts made at once on one device from several threads: the kernels are
resolved by whichever comes first, and every context runs."""
import threading

import numpy as np
import pytest

import ming_dit_amd as m
from helpers import bf16, empty_bf16, from_dev, randn, sync, to_dev

pytestmark = pytest.mark.gpu


def test_contexts_from_threads(ctx):
    rows, D = 5, 256
    x, w = bf16(randn(4300, (rows, D))), bf16(randn(4301, (D,)))
    xd, wd, ys, bad = to_dev(x), to_dev(w), [empty_bf16(rows, D) for _ in range(6)], []
    sync()

    def one(y):
        try:
            c = m.Ctx(0)
            c.rmsnorm(xd, wd, y, rows, D)
            c.synchronize()
            c.close()
        except Exception as e:      # seen by the main thread
            bad.append(e)

    ts = [threading.Thread(target=one, args=(y,)) for y in ys]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad
    want = empty_bf16(rows, D)
    ctx.rmsnorm(xd, wd, want, rows, D)
    ctx.synchronize()
    assert all(np.array_equal(from_dev(y), from_dev(want)) for y in ys)
