"""Light lists at the sizes where the culling call takes another way: clusters
around a packing workgroup's 32, around the 32,768 up to which offsets and
lists are packed in one launch, and lights around the bound under which every
cluster block moves them to view space itself. Bit-exact against the oracle,
totals and overflow counts included, with and without asking for them."""
import numpy as np
import pytest

from hellovulkan_amd import abi
from oracle import hvx_oracle as O
from tests.helpers import camera, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid,n_lights,cap", [
    ((1, 1, 1), 1, 1), ((31, 1, 1), 40, 8), ((4, 8, 1), 100, 128), ((3, 11, 1), 300, 70), ((5, 13, 7), 2000, 150),
    ((32, 32, 32), 1500, 32), ((33, 31, 33), 1500, 16), ((16, 9, 24), 7281, 40), ((16, 9, 24), 7282, 40),
    ((16, 9, 24), 0, 16)])
@pytest.mark.parametrize("totals", [True, False])
def test_lists_at_the_dispatch_edges(ctx, grid, n_lights, cap, totals):
    import torch
    desc, cam, ubo, ivp = camera(800, 450, grid)
    n = grid[0] * grid[1] * grid[2]
    lights = abi.scene_lights(31 + n_lights, n_lights)
    boxes = O.build_aabbs(ubo)
    cells_ref, idx_ref, tot_ref, ov_ref = O.cull_lights(ubo, boxes, lights, cap)
    cells = torch.full((2 * n + 2,), -1, dtype=torch.int32, device="cuda")
    idx = torch.full((n * cap + 8,), -1, dtype=torch.int32, device="cuda")
    tot, ov = (torch.full((1,), -1, dtype=torch.int32, device="cuda") for _ in range(2))
    d_lights = to_dev(lights.view(np.uint8)) if n_lights else torch.zeros(48, dtype=torch.uint8, device="cuda")
    ctx.cull_lights(ubo, to_dev(boxes), d_lights, n_lights, cap, cells, idx, n * cap, tot if totals else None,
                    ov if totals else None)
    torch.cuda.synchronize()
    got = cells.cpu().numpy()
    assert np.array_equal(got[:2 * n].view(np.uint32), cells_ref.view(np.uint32).reshape(-1)) and np.all(got[2 * n:] == -1)
    host = idx.cpu().numpy()
    assert np.array_equal(host[:tot_ref].view(np.uint32), idx_ref) and np.all(host[tot_ref:] == -1)
    assert (int(tot.item()), int(ov.item())) == ((tot_ref, ov_ref) if totals else (-1, -1))
