"""The adjoint at the edges of its reductions' workgroup sizes (leaves of 64 and
128 particles), against the oracle, and its cost with small leaves: the
source reduction does not start waves that no particle of a leaf needs."""
import numpy as np
import pytest

from haccsr import Context
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nd", [1, 63, 64, 65, 127, 128, 129, 500])
@pytest.mark.parametrize("mode", [1, 2])  # fused, two passes
def test_adjoint(nd, mode):
    print(f"case leaf threads nd={nd} mode={mode}", flush=True)
    n, box = 3000 if nd > 1 else 700, 6.0
    rng = np.random.default_rng(nd)
    p = (rng.random((n, 3)) * box).astype(np.float32)
    x, y, z = (p[:, k].copy() for k in range(3))
    m = np.ones(n, np.float32)
    lo, hi = np.zeros(3, np.float32), np.full(3, box, np.float32)
    tp = O.TreeParams(lo, hi, lo - 1, hi + 1, nd=nd)
    tree = O.build_tree(tp, x, y, z, m)
    lam = rng.standard_normal((n, 3)).astype(np.float32)
    ref = O.adjoint_f64(tp, tree, O.build_lists(tp, tree), lam.astype(np.float64))
    ctx = Context(nd=nd)
    ctx.set_tuning(adjoint_mode=mode, chunk=256)  # lists in several items
    ctx.build(x, y, z, m, min_loc=lo, max_loc=hi)
    ctx.lists(lo - 1, hi + 1)
    ctx.forces()
    g = np.stack(ctx.adjoint(*(lam[:, k].copy() for k in range(3))), 1)
    # 1e-4: the adjoint's tolerance against FP64
    assert np.linalg.norm(g - ref) <= 1e-4 * np.linalg.norm(ref)
    ctx.close()


def test_cost_with_small_leaves():
    """Leaves of at most 8 particles on a lattice: 80 times the segments of
    leaves of up to 200, which the source reduction walks."""
    import torch
    side = 64
    g = torch.arange(side, dtype=torch.float32, device="cuda") * 0.5
    x, y, z = (t.reshape(-1).contiguous() for t in torch.meshgrid(g, g, g, indexing="ij"))
    n = x.numel()
    ms = {}
    for nd in (8, 200):
        a = [t.clone() for t in (x, y, z)] + [torch.ones(n, device="cuda")]
        out = [torch.empty(n, device="cuda") for _ in range(3)]
        lam = [torch.ones(n, device="cuda") for _ in range(3)]
        torch.cuda.synchronize()
        ctx = Context(nd=nd)
        ctx.build(*a, min_loc=(0, 0, 0), max_loc=(32, 32, 32), device_ptrs=True)
        ctx.lists((-1, -1, -1), (33, 33, 33))
        ctx.set_tuning(adjoint_mode=1)
        for _ in range(5):
            ctx.adjoint(*lam, *out, device_ptrs=True)
            ms[nd] = min(ms.get(nd, np.inf), ctx.stats().adjoint_ms)
        print(f"case small leaves nd={nd} segments {ctx.stats().segments} adjoint {ms[nd]:.3f} ms", flush=True)
        ctx.close()
    # 2.43 and 1.14 ms; 3.38 with four waves a leaf
    assert ms[8] < 2.5 * ms[200]
