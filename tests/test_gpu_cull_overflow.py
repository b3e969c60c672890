"""Overflow counts of the packed lists: clusters of every remainder by four (the
counts before them shift the overflows' alignment), more of them than one pass of
the workgroup that sums them, most of them overflowing, and none."""
import numpy as np
import pytest

from hellovulkan_amd import abi
from oracle import hvx_oracle as O
from tests.helpers import camera, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [(1, 1, 1), (2, 1, 1), (3, 1, 1), (1, 5, 1), (16, 9, 24), (31, 11, 9), (26, 13, 21),
                                  (31, 17, 61), (32, 32, 32)])
@pytest.mark.parametrize("cap", [1, 7, 1024])
def test_overflow_equals_the_oracle(ctx, grid, cap):
    import torch
    _, _, ubo, _ = camera(800, 450, grid)
    n = grid[0] * grid[1] * grid[2]
    if n * cap > 1 << 22:
        cap = 3
    lights = abi.scene_lights(5, 900)
    boxes = O.build_aabbs(ubo)
    _, _, tot_ref, ov_ref = O.cull_lights(ubo, boxes, lights, cap)
    cells = torch.empty(2 * n, dtype=torch.int32, device="cuda")
    idx = torch.empty(n * cap, dtype=torch.int32, device="cuda")
    tot, ov = (torch.full((1,), -1, dtype=torch.int32, device="cuda") for _ in range(2))
    for call in (ctx.cull_lights, ctx.cull_lights_noalloc):
        ov.fill_(-1)
        call(ubo, to_dev(boxes), to_dev(lights.view(np.uint8)), 900, cap, cells, idx, n * cap, tot, ov)
        torch.cuda.synchronize()
        assert (int(tot.item()), int(ov.item())) == (tot_ref, ov_ref)
