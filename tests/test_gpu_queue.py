"""The work queue and the work items of the force phase: forces do not depend
on how many waves share the queue (every wave owns an item, most pop, one wave
per compute unit pops nearly all), nor fail when a cap on the plan's memory
rules out the finer cut of short lists."""
import sys

import numpy as np
import pytest

from haccsr import Context
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def load(n, box, seed):
    rng = np.random.default_rng(seed)
    p = (rng.random((n, 3)) * box).astype(np.float32)
    p[: n // 4] = (box / 2 + 0.4 * rng.standard_normal((n // 4, 3))).astype(np.float32)
    return [p[:, k].copy() for k in range(3)], np.ones(n, np.float32)


@pytest.mark.parametrize("n,box,nd", [(40, 3.0, 64), (3000, 8.0, 7), (30000, 14.0, 96)])
def test_forces_do_not_depend_on_the_queue(n, box, nd):
    print(f"case queue n={n} nd={nd}", flush=True)
    sys.stdout.flush()
    (x, y, z), m = load(n, box, 5)
    lo, hi = np.zeros(3, np.float32), np.full(3, box, np.float32)
    flo, fhi = np.full(3, -1, np.float32), np.full(3, box + 1, np.float32)
    tp = O.TreeParams(lo, hi, flo, fhi, nd=nd)
    tree = O.build_tree(tp, x, y, z, m)
    R = np.stack(O.forces_step16(tp, tree, O.build_lists(tp, tree)), 1)
    ctx = Context(nd=nd)
    ctx.build(x.copy(), y.copy(), z.copy(), m.copy(), min_loc=lo, max_loc=hi)
    ctx.lists(flo, fhi)
    first = None
    for wpc in (0, 1, 2, 7, 256):
        ctx.set_tuning(waves_per_cu=wpc)
        F = np.stack(ctx.forces(), 1)
        st = ctx.stats()
        if first is None:
            first, counts = F, (st.evaluated_pairs, st.unmasked_pairs)
            # 1e-5: the force tolerance
            assert np.sqrt(np.sum((F - R) ** 2) / np.sum(R ** 2)) <= 1e-5
        assert np.array_equal(F.view(np.uint32), first.view(np.uint32)), wpc
        assert (st.evaluated_pairs, st.unmasked_pairs) == counts, wpc
    # a cap below the finer cut's partial sums: one item per list
    ctx.set_tuning(waves_per_cu=0, max_plan_bytes=1 << 20)
    ctx.lists(flo, fhi)
    F = np.stack(ctx.forces(), 1)
    assert np.sqrt(np.sum((F - R) ** 2) / np.sum(R ** 2)) <= 1e-5
    ctx.close()
