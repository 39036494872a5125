"""The force phase's pair counts when the queue's waves outnumber the items
but its owners (half of the waves) do not: waves numbered past the items pop
items too, and what they evaluate counts."""
import numpy as np
import pytest

from haccsr import Context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wpc", [4, 10, 16])  # all waves of the grid fit on the chip at once
def test_pair_counts(wpc):
    import torch
    grid = torch.cuda.get_device_properties(0).multi_processor_count * wpc
    n, box = 25000 * wpc // 4, 9.0 * (wpc / 4) ** (1 / 3)
    rng = np.random.default_rng(wpc)
    p = (rng.random((n, 3)) * box).astype(np.float32)
    x, y, z = (p[:, k].copy() for k in range(3))
    ctx = Context(nd=128)
    ctx.set_tuning(waves_per_cu=wpc, cull_off=1)
    ctx.build(x, y, z, np.ones(n, np.float32), min_loc=(0, 0, 0), max_loc=(box,) * 3)
    ctx.lists((-1,) * 3, (box + 1,) * 3)
    ent = ctx.get_lists()[4]

    def items(chunk):
        return int(np.sum(-(-ent // chunk)))

    # the item length that puts their number halfway between owners and waves
    chunk = next(c for c in range(256, 1 << 20, 8) if items(c) <= 0.75 * grid)
    print(f"case counts waves/CU {wpc} grid {grid} leaves {ent.size} chunk {chunk} items {items(chunk)}", flush=True)
    assert 0.6 * grid < items(chunk)
    ctx.set_tuning(chunk=chunk)
    pairs = ctx.stats().pairs
    for _ in range(4):
        ctx.forces()
        # nothing is culled: every list pair is evaluated
        assert ctx.stats().evaluated_pairs == pairs
    # with culling: the same counts with twice the waves, when each item has an owner
    ctx.set_tuning(cull_off=0)
    ctx.forces()
    some = (ctx.stats().evaluated_pairs, ctx.stats().unmasked_pairs)
    ctx.set_tuning(waves_per_cu=2 * wpc)
    ctx.forces()
    assert some == (ctx.stats().evaluated_pairs, ctx.stats().unmasked_pairs)
    assert 0 < some[1] < some[0] < pairs
    ctx.close()
