"""Subtrees built by one workgroup: node counts around their limit, a subtree
too deep for them (the level passes take the build), a launch that runs out of
node slots (repeated with more).  Bit-exact with the oracle."""
import numpy as np
import pytest

from haccsr import Context
from oracle import oracle as O

pytestmark = pytest.mark.gpu

FIELDS = ["count", "ppm", "tdr", "xmin", "xmax", "xc"]


def same(nodes, ref):
    assert nodes.shape == ref.shape
    for f in FIELDS:
        a, b = nodes[f], ref[f]
        if a.dtype.kind == "f":
            a, b = a.view(np.uint32), b.view(np.uint32)
        assert np.array_equal(a, b), f


def oracle_tree(p, box, nd):
    lo, hi = np.zeros(3, np.float32), np.full(3, box, np.float32)
    tp = O.TreeParams(lo, hi, lo - 1, hi + 1, nd=nd)
    return O.build_tree(tp, *(p[:, k].copy() for k in range(3)), np.ones(p.shape[0], np.float32))


def geometric():
    """Each axis holds a geometric sequence: a tree of 63 levels of a few
    particles each."""
    k = np.arange(1800)
    return np.stack([np.where(k % 3 == d, 0.8 ** (k // 3), 0) for d in range(3)], 1).astype(np.float32)


@pytest.mark.parametrize("n,nd", [(1, 1), (2, 1), (3, 1), (64, 1), (65, 8), (2047, 16), (2048, 16),
                                  (2049, 16), (2048, 1), (4097, 24), (9000, 2500), (6000, 3)])
def test_sizes(n, nd):
    print(f"case subtree n={n} nd={nd}", flush=True)
    rng = np.random.default_rng(n + nd)
    p = (rng.random((n, 3)) * 5).astype(np.float32)
    p[: n // 8] = p[0]  # and a degenerate node
    p[n // 2: n // 2 + n // 8, 0] *= np.float32(1e-6)  # sums that round
    ref = oracle_tree(p, 5.0, nd)
    ctx = Context(nd=nd)
    x, y, z = (p[:, k].copy() for k in range(3))
    ids = np.arange(n, dtype=np.int64)
    ctx.build(x, y, z, np.ones(n, np.float32), ids=ids, min_loc=(0, 0, 0), max_loc=(5, 5, 5))
    assert np.array_equal(ids, ref.id)
    assert np.array_equal(x, ref.x) and np.array_equal(z, ref.z)
    same(ctx.nodes(), ref.nodes)
    for f in ("offset", "cl", "cr"):
        assert np.array_equal(ctx.nodes()[f], ref.nodes[f]), f
    ctx.close()


@pytest.mark.parametrize("boxes,nd", [(1, 1), (40, 300)])  # too deep; out of node slots
def test_geometric(boxes, nd):
    print(f"case subtree geometric boxes={boxes} nd={nd}", flush=True)
    p = geometric()
    ref = oracle_tree(p, 2.0, nd)
    n = p.shape[0]
    all_p = np.concatenate([p] * boxes)
    x, y, z = (all_p[:, k].copy() for k in range(3))
    ids = np.arange(n * boxes, dtype=np.int64)
    ctx = Context(nd=nd)
    ctx.build_many(np.arange(boxes + 1) * n, x, y, z, np.ones(n * boxes, np.float32),
                   np.zeros((boxes, 3)), np.full((boxes, 3), 2.0), ids=ids)
    nodes = ctx.nodes()
    m = ref.nodes.shape[0]
    for b in range(boxes):
        assert np.array_equal(ids[b * n:(b + 1) * n], ref.id + b * n)
        same(nodes[b * m:(b + 1) * m], ref.nodes)
    if boxes > 1:  # more nodes than the first launch has slots for
        assert boxes * (m - 1) > 5 * (boxes * n // nd) + 4 * boxes + 1024
    ctx.close()
