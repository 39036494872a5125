"""GPU lists at the edges of the wave walk: lists longer than the segment
cache (walked twice), stacks at their bound (walked node by node near it),
deep trees, a tree of one node.  Bit-exact with the oracle."""
import sys

import numpy as np
import pytest

from haccsr import Context
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def load(kind):
    rng = np.random.default_rng(3)
    if kind == "long":        # every leaf a particle, all within the cutoff
        p, box, nd, oa, force = rng.random((20000, 3)) * 2.0, 2.0, 1, 0.0, (0.9, 1.1)
    elif kind == "cache":     # lists on both sides of the cache's 512 segments
        p, box, nd, oa, force = rng.random((6000, 3)) * 9.0, 9.0, 2, 0.1, (1.0, 8.0)
    elif kind == "deep":      # a geometric cloud: the tree is a chain
        s = 0.5 ** (np.arange(4000) % 100)
        p, box, nd, oa, force = s[:, None] * (0.5 + 0.5 * rng.random((4000, 3))) * 4.0, 4.0, 4, 0.2, (-1.0, 5.0)
    else:                     # the root is the only leaf
        p, box, nd, oa, force = rng.random((50, 3)) * 4.0, 4.0, 64, 0.1, (-1.0, 5.0)
    p = p.astype(np.float32)
    return p, box, nd, oa, force


@pytest.mark.parametrize("kind", ["long", "cache", "deep", "root"])
def test_walk_edges(kind):
    p, box, nd, oa, (f0, f1) = load(kind)
    print(f"case walk {kind} n={p.shape[0]}", flush=True)
    sys.stdout.flush()
    x, y, z = (p[:, k].copy() for k in range(3))
    m = np.ones(p.shape[0], np.float32)
    lo, hi = np.zeros(3, np.float32), np.full(3, box, np.float32)
    flo, fhi = np.full(3, f0, np.float32), np.full(3, f1, np.float32)
    tp = O.TreeParams(lo, hi, flo, fhi, nd=nd, oa=oa)
    tree = O.build_tree(tp, x, y, z, m)
    ref = O.build_lists(tp, tree)
    ctx = Context(nd=nd, oa=oa)
    ctx.build(x, y, z, m, min_loc=lo, max_loc=hi)
    ctx.lists(flo, fhi)
    leaves, seg_ptr, sa, sb, ent = ctx.get_lists()
    longest = int(np.diff(seg_ptr).max())
    print(f"  leaves {leaves.shape[0]} longest list {longest} depth {ctx.stats().max_depth}", flush=True)
    assert np.array_equal(leaves, ref.leaves)
    assert np.array_equal(seg_ptr, ref.seg_ptr)
    assert np.array_equal(sa, ref.seg_a) and np.array_equal(sb, ref.seg_b)
    assert np.array_equal(ent, ref.entries)
    if kind == "long":
        assert longest > 4096
    ctx.close()
