"""Binning with the default (two roughness classes) and the exact variant at the sizes
where it takes another way: tiles past 16,384 pixels (counted twice), more tiles than
CUs (segments put together in LDS, the largest of them 64 KB), 2 x 512 bins, tiles
narrower and wider than a workgroup's step, one pixel. Every pixel of the frame."""
import numpy as np
import pytest

from hellovulkan_amd import abi
from oracle import hvx_oracle as O
from tests.helpers import camera, random_ibl_maps, to_dev
from tests.test_gpu_cf import SHADE_TOL, gpu_aabbs, gpu_cull

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["fast", "exact"])
@pytest.mark.parametrize("width,height,grid", [
    (1, 1, (1, 1, 1)), (130, 127, (1, 1, 4)), (2100, 9, (1, 1, 3)), (300, 260, (17, 16, 6)), (320, 200, (16, 16, 6)),
    (700, 130, (257, 1, 5)), (190, 340, (2, 1, 512)), (190, 340, (2, 1, 513)), (2142, 2142, (17, 17, 4))])
def test_every_pixel_is_shaded(ctx, width, height, grid, mode):
    import torch
    desc, cam, ubo, ivp = camera(width, height, grid)
    lights = abi.scene_lights(51, 60)
    fr = abi.scene_fragments(52, desc, ivp)
    maps = random_ibl_maps(np.random.default_rng(53))
    cells, idx, _, _, d_idx, d_lights, d_cells = gpu_cull(ctx, ubo, gpu_aabbs(ctx, ubo), lights, 32)
    dev = {k: to_dev(v) for k, v in fr.items()}
    dm = {k: to_dev(maps[k]) for k in ("spec", "diff", "lut")}
    m = abi.ibl_maps(dm["spec"], maps["spec_size"], maps["spec_mips"], dm["diff"], maps["diff_size"], dm["lut"],
                     maps["lut_w"], maps["lut_h"])
    F = width * height
    rgb = torch.full((3 * F + 8,), np.nan, dtype=torch.float32, device="cuda")
    ctx.set_option(abi.OPT_SHADE_EXACT, 1 if mode == "exact" else 0)
    try:
        ctx.shade(abi.frag_soa(dev, width, height, ivp), cam, ubo, abi.pbr_defaults(), d_lights, 60, d_cells, d_idx, m, rgb)
        torch.cuda.synchronize()
    finally:
        ctx.set_option(abi.OPT_SHADE_EXACT, 0)
    host = rgb.cpu().numpy()
    assert np.all(np.isfinite(host[:3 * F])) and np.all(np.isnan(host[3 * F:]))
    got = host[:3 * F].reshape(3, F).T
    ids = np.arange(F, dtype=np.uint32) if F <= 100000 else \
        np.unique(np.random.default_rng(5).integers(0, F, 60000)).astype(np.uint32)
    ref = O.shade(fr, width, height, ivp, cam, ubo, abi.pbr_defaults(), lights, cells, idx, maps, ids)
    if mode == "exact":
        assert np.array_equal(got[ids].view(np.uint32), ref.view(np.uint32))
    assert O.rel_err(got[ids], ref) <= SHADE_TOL
