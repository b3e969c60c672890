"""Probe batches on both sides of the line between a texel and four texels per wave,
with item sizes that do not divide their mips: equal to the filter's own calls to
the bit, run after run, and nothing written past a chain."""
import numpy as np
import pytest

from hellovulkan_amd import abi
from tests.helpers import to_dev

pytestmark = pytest.mark.gpu

FEW = [(16, 8, 4), (33, 21, 3)]  # 96 tiles
MANY = [(64, 60, 6), (20, 100, 4), (128, 64, 7), (5, 3, 2)]  # 2,406 tiles


@pytest.mark.parametrize("probes,samples", [(FEW, 10), (FEW, 11), (FEW, 100), (MANY, 100), (MANY[:1], 300)])
@pytest.mark.parametrize("tile,wgs", [(32, 1), (100, 3), (8192, 4)])
def test_batch_equals_calls(ctx, probes, samples, tile, wgs):
    import torch
    rng = np.random.default_rng(samples)
    cubes, outs, refs, specs = [], [], [], []
    for S, So, mips in probes:
        cubes.append(to_dev(rng.uniform(0, 9, 6 * S * S * 4).astype(np.float32)))
        floats = abi.cube_chain_floats(So, mips)
        refs.append(torch.full((floats + 8,), -1.0, dtype=torch.float32, device="cuda"))
        outs.append(torch.full_like(refs[-1], -1.0))
        ctx.filter(abi.FILTER_SPECULAR, cubes[-1], S, refs[-1], So, mips, samples)
        specs.append(abi.probe(cubes[-1], S, outs[-1], So, mips))
    b = abi.Batch(ctx, specs, samples, [])
    b.set_tuning(tile, wgs, 0, 8)
    for _ in range(2):
        for o in outs:
            o.fill_(-1.0)
        b.run()
        torch.cuda.synchronize()
        for o, r in zip(outs, refs):
            assert torch.equal(o.view(torch.int32), r.view(torch.int32))
    b.close()
