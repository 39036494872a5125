"""The list walk with its stack at the bound (1024 nodes beside the reserve):
rounds narrowed to the room left, then one node at a time.  Bit-exact with the
oracle on a load whose stack gets there, as a model of the walk shows."""
import numpy as np
import pytest

from haccsr import Context
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SLOTS, WIDTH = 1024, 64


def load(m):
    """Clusters of m particles at -0.3^k along x: the right child holds all but
    the leftmost few, so the walk opens a chain with a bushy subtree at each
    step and comes back to those last."""
    rng = np.random.default_rng(m)
    s = 0.3 ** np.arange(70)
    p = (rng.random((70, m, 3)) - 0.5) * 0.2 * s[:, None, None]
    p[:, :, 0] -= s[:, None]
    return p.reshape(-1, 3).astype(np.float32)


def heights(nodes, leaf):
    """Rounds of a leaf's walk with every node opened: the greatest stack
    height, the rounds narrowed to the room left, those of one node."""
    cl, cr, off, cnt = (nodes[f] for f in ("cl", "cr", "offset", "count"))
    stack, peak, narrow, single = [(0, False)], 0, 0, 0  # (node, decided), top last
    while stack:
        h = len(stack)
        room = SLOTS - h
        b = min(WIDTH, h, room) if room > 0 else 1
        peak = max(peak, h)
        narrow += 0 < room < min(WIDTH, h)
        single += room <= 0
        top = stack[:-b - 1:-1]
        del stack[-b:]
        back, opened = [], False
        for t, decided in top:
            if not decided and (cl[t] > 0 or cr[t] > 0):
                over = t < leaf and off[t] <= off[leaf] and off[leaf] + cnt[leaf] <= off[t] + cnt[t]
                opened = True
                back += [(k, False) for k in (cr[t], cl[t]) if k > 0 and k != leaf and (over or cnt[k] > 0)]
            elif opened:
                back.append((t, True))
        stack += back[::-1]
    return peak, narrow, single


@pytest.mark.parametrize("m", [32, 64])
def test_stack_at_its_bound(m):
    p = load(m)
    n = p.shape[0]
    x, y, z = (p[:, k].copy() for k in range(3))
    w = np.ones(n, np.float32)
    lo, hi = np.full(3, -2, np.float32), np.full(3, 1, np.float32)
    tp = O.TreeParams(lo, hi, lo - 1, hi + 1, nd=1, oa=0.0)
    tree = O.build_tree(tp, x, y, z, w)
    ref = O.build_lists(tp, tree)
    peak, narrow, single = heights(tree.nodes, int(ref.leaves[0]))
    print(f"case walk bound n={n}: stack up to {peak}, {narrow} rounds narrowed, {single} of one node", flush=True)
    assert peak > SLOTS and narrow > 10 and single > 10
    ctx = Context(nd=1, oa=0.0)
    ctx.build(x, y, z, w, min_loc=lo, max_loc=hi)
    ctx.lists(lo - 1, hi + 1)
    leaves, seg_ptr, sa, sb, ent = ctx.get_lists()
    assert np.array_equal(leaves, ref.leaves)
    assert np.array_equal(seg_ptr, ref.seg_ptr)
    assert np.array_equal(sa, ref.seg_a) and np.array_equal(sb, ref.seg_b)
    assert np.array_equal(ent, ref.entries)
    ctx.close()
