"""Contexts made and destroyed in turn, in two threads at once, on loads of
different sizes: device buffers that pass from one context to the next change
no result."""
import threading

import numpy as np
import pytest

from haccsr import Context

pytestmark = pytest.mark.gpu

SIZES = [(3000, 16), (500, 8), (20000, 64), (1, 4), (9000, 32)]


def step(n, nd):
    rng = np.random.default_rng(n)
    p = (rng.random((n, 3)) * 9).astype(np.float32)
    x, y, z = (p[:, k].copy() for k in range(3))
    ctx = Context(nd=nd)
    ctx.build(x, y, z, np.ones(n, np.float32), min_loc=(0, 0, 0), max_loc=(9, 9, 9))
    ctx.lists((-1, -1, -1), (10, 10, 10))
    F = np.stack(ctx.forces(), 1)
    g = np.stack(ctx.adjoint(*(F[:, k].copy() for k in range(3))), 1)
    ctx.close()
    return np.concatenate([F, g]).view(np.uint32)


def test_buffers_passed_on():
    print("case contexts in turn and in two threads", flush=True)
    ref = {s: step(*s) for s in SIZES}
    bad = []

    def work(order):
        for s in order * 3:
            if not np.array_equal(step(*s), ref[s]):
                bad.append(s)

    ts = [threading.Thread(target=work, args=(o,)) for o in (SIZES, SIZES[::-1])]
    for t in ts:
        t.start()
    for t in ts:
        t.join(100)
    assert not any(t.is_alive() for t in ts)
    assert not bad
