"""Builds with leaves of one to three particles on both sides of the lines
between which the passes over levels take them whole: bit-exact with the
oracle, and not slower than a build that has no subtrees (masses of 0.5)."""
import numpy as np
import pytest

from haccsr import Context
from test_gpu_subtree import oracle_tree, same

pytestmark = pytest.mark.gpu


def load(n):
    rng = np.random.default_rng(n)
    p = (rng.random((n, 3)) * 5).astype(np.float32)
    p[: n // 3] = 2.5 + 0.01 * rng.standard_normal((n // 3, 3))
    return p


@pytest.mark.parametrize("n,nd", [(512, 1), (513, 1), (1024, 2), (1025, 2), (1536, 3), (1537, 3), (1537, 4),
                                  (56000, 1), (56001, 1), (56001, 3)])
def test_around_the_lines(n, nd):
    print(f"case subtree rule n={n} nd={nd}", flush=True)
    p = load(n)
    ref = oracle_tree(p, 5.0, nd)
    ctx = Context(nd=nd)
    x, y, z = (p[:, k].copy() for k in range(3))
    ids = np.arange(n, dtype=np.int64)
    ctx.build(x, y, z, np.ones(n, np.float32), ids=ids, min_loc=(0, 0, 0), max_loc=(5, 5, 5))
    assert np.array_equal(ids, ref.id)
    same(ctx.nodes(), ref.nodes)
    for f in ("offset", "cl", "cr"):
        assert np.array_equal(ctx.nodes()[f], ref.nodes[f]), f
    ctx.close()


@pytest.mark.parametrize("n", [2000, 8000])
def test_small_leaves_cost(n):
    p = load(n)
    ms = []
    for mass in (1.0, 0.5):
        ctx = Context(nd=1)
        best = np.inf
        for _ in range(10):
            x, y, z = (p[:, k].copy() for k in range(3))
            ctx.build(x, y, z, np.full(n, mass, np.float32), min_loc=(0, 0, 0), max_loc=(5, 5, 5))
            best = min(best, ctx.stats().build_ms)
        ms.append(best)
        ctx.close()
    print(f"case subtree rule cost n={n} unit {ms[0]:.3f} other {ms[1]:.3f} ms", flush=True)
    # with subtrees 1.2 to 1.6 times the passes' time
    assert ms[0] < 1.15 * ms[1]
