"""Device buffers kept from destroyed contexts: given back on request, with
other contexts alive and from another thread, and no error or result of a
context changes by it."""
import threading

import pytest

import haccsr
from haccsr import Context
from test_gpu_contexts import SIZES, step

import numpy as np

pytestmark = pytest.mark.gpu


def test_memory_is_given_back():
    import torch
    print("case release", flush=True)
    live = Context(nd=32)
    n = 300000
    rng = np.random.default_rng(1)
    p = (rng.random((n, 3)) * 40).astype(np.float32)

    def build(ctx):
        x, y, z = (p[:, k].copy() for k in range(3))
        ctx.build(x, y, z, np.ones(n, np.float32), min_loc=(0, 0, 0), max_loc=(40, 40, 40))
        ctx.lists((-1, -1, -1), (41, 41, 41))
        return np.stack(ctx.forces(), 1)

    F = build(live)
    ctx = Context(nd=32)
    build(ctx)
    ctx.close()
    before = torch.cuda.mem_get_info()[0]
    freed = haccsr.release_buffers(0)
    after = torch.cuda.mem_get_info()[0]
    print(f"  freed {freed} bytes, free memory grew by {after - before}", flush=True)
    assert freed > 10 * n * 4
    # an allocation may share a page with others, and its page stays then
    assert after - before > freed // 2
    assert haccsr.release_buffers(0) == 0
    assert np.array_equal(build(live), F)
    live.close()
    with pytest.raises(haccsr.HsrError, match="out of range"):
        haccsr.release_buffers(1 << 20)


def test_contexts_in_threads_with_releases():
    print("case contexts in two threads, releases in a third", flush=True)
    ref = {s: step(*s) for s in SIZES}
    done, bad, stop = [], [], threading.Event()

    def work(order):
        try:
            for s in order * 3:
                if not np.array_equal(step(*s), ref[s]):
                    bad.append(s)
                done.append(s)
        except Exception as e:  # an error status of any call
            bad.append(e)

    def release():
        try:
            while not stop.wait(0.002):
                haccsr.release_buffers(0)
        except Exception as e:
            bad.append(e)

    ts = [threading.Thread(target=work, args=(o,)) for o in (SIZES, SIZES[::-1])]
    r = threading.Thread(target=release)
    for t in ts + [r]:
        t.start()
    for t in ts:
        t.join(50)
    stop.set()
    r.join(10)
    assert not any(t.is_alive() for t in ts + [r])
    assert not bad, bad
    assert len(done) == 6 * len(SIZES)
