"""Quadrupole masses of deep trees: bit-exact with the oracle with the nodes in
level order and with subtrees (few enough to pick a depth's out of all, or
bucketed by depth), and their cost beside the tree
build's where the tree is deep and has many nodes."""
import numpy as np
import pytest

from haccsr import Context
from test_gpu_quadrupole import check_ppm, run_q
from test_gpu_parity import check_tree

pytestmark = pytest.mark.gpu


def deep(n, chain):
    """n uniform particles and a geometric sequence on each axis, which makes
    the tree deep (68 levels with 95 particles an axis)."""
    rng = np.random.default_rng(n)
    k = np.arange(3 * chain)
    geo = np.stack([np.where(k % 3 == d, 0.3 ** (k // 3), 0.0) for d in range(3)], 1)
    p = np.concatenate([geo, 1.0 + 7.0 * rng.random((n, 3))]).astype(np.float32)
    return [p[:, d].copy() for d in range(3)]


@pytest.mark.parametrize("unit", [True, False])  # with subtrees, by levels alone
@pytest.mark.parametrize("n,chain,nd", [(0, 1, 4), (0, 40, 1), (5000, 95, 13), (30000, 40, 40), (30000, 95, 1)])
def test_masses(n, chain, nd, unit):
    print(f"case quadrupole depth n={n} chain={chain} nd={nd} unit={unit}", flush=True)
    x, y, z = deep(n, chain)
    m = np.ones(x.size, np.float32)
    if not unit:
        m[::3] = 0.5
    tp, tree, lists, ctx, arrs = run_q(x, y, z, m, [0] * 3, [8.0] * 3, [-1.0] * 3, [9.0] * 3, nd, 0.5)
    check_tree(tree, ctx, arrs)
    if x.size > nd and x.size > 12:
        check_ppm(tree, ctx)
    ctx.close()


def test_cost_is_not_nodes_times_depth():
    x, y, z = deep(1500000, 95)
    m = np.full(x.size, 0.5, np.float32)  # by levels alone
    ms = []
    for tdpts in (1, 12):
        ctx = Context(nd=1, tdpts=tdpts)
        best = np.inf
        for _ in range(8):
            ctx.build(x.copy(), y.copy(), z.copy(), m.copy(), min_loc=[0] * 3, max_loc=[8.0] * 3)
            best = min(best, ctx.stats().build_ms)
        ms.append(best)
        st = ctx.stats()
        print(f"case quadrupole cost tdpts={tdpts} nodes {st.nodes} depth {st.max_depth} build {best:.2f} ms", flush=True)
        ctx.close()
    # a visit of every node takes 1.2 ms, one for each of the 76 depths 5.5 ms,
    # beside a build of 26 ms
    assert ms[1] < 1.13 * ms[0]
