"""Leaf sizes at the edges of the pass rule (slots of a pass against targets
left): one leaf of n particles, forces and the fused adjoint against the
oracle."""
import numpy as np
import pytest

from haccsr import Context
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 7, 8, 9, 16, 17, 24, 25, 32, 33, 40, 41, 64, 65, 96, 97, 112, 113, 127, 128, 129,
         145, 200, 300]


@pytest.mark.parametrize("n", SIZES)
def test_one_leaf(n):
    print(f"case passes n={n}", flush=True)
    rng = np.random.default_rng(n)
    box = 3.0
    p = (rng.random((n, 3)) * box).astype(np.float32)
    x, y, z = (p[:, k].copy() for k in range(3))
    m = np.ones(n, np.float32)
    lo, hi = np.zeros(3, np.float32), np.full(3, box, np.float32)
    flo, fhi = np.full(3, -1, np.float32), np.full(3, box + 1, np.float32)
    tp = O.TreeParams(lo, hi, flo, fhi, nd=512)
    tree = O.build_tree(tp, x, y, z, m)
    R = np.stack(O.forces_step16(tp, tree, O.build_lists(tp, tree)), 1)
    ctx = Context(nd=512)
    ctx.build(x, y, z, m, min_loc=lo, max_loc=hi)
    ctx.lists(flo, fhi)
    F = np.stack(ctx.forces(), 1)
    # 1e-5: the force tolerance; n = 1 has no force at all
    assert np.sqrt(np.sum((F - R) ** 2)) <= 1e-5 * np.sqrt(np.sum(R ** 2))
    if n >= 7:
        lam = rng.standard_normal((n, 3)).astype(np.float32)
        lists = O.build_lists(tp, tree)
        ref = O.adjoint_f64(tp, tree, lists, lam.astype(np.float64))
        g = np.stack(ctx.adjoint(*(lam[:, k].copy() for k in range(3))), 1)
        # 1e-4: the adjoint's tolerance against FP64
        assert np.linalg.norm(g - ref) <= 1e-4 * np.linalg.norm(ref)
    ctx.close()
