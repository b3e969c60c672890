"""Lights whose term is NaN though they lie behind the surface: at the fragment's
own position (no direction), exactly opposite the viewer (no half vector), so
near that its attenuation overflows, of infinite colour. The default variant gives the oracle's NaN at the oracle's
fragments, whatever the rest of the wave does with the light, and the oracle's
value within the shading bound everywhere else."""
import numpy as np
import pytest

from hellovulkan_amd import abi
from oracle import hvx_oracle as O
from tests.helpers import camera, random_ibl_maps, to_dev
from tests.test_gpu_cf import SHADE_TOL

pytestmark = pytest.mark.gpu

W, H, Z0 = 64, 8, 0.25


@pytest.mark.parametrize("light,rough", [("own", 0.4), ("own", 0.9), ("opposite", 0.4), ("infinite", 0.4),
                                         ("infinite", 0.9), ("infinite_far", 0.4), ("near", 0.4)])
def test_nan_terms_behind_the_surface(ctx, light, rough):
    import torch
    # an identity matrix: fragment (x, y) lies at its own exact NDC position
    _, cam, ubo, _ = camera(W, H, (1, 1, 1))
    ivp = np.eye(4, dtype=np.float32).reshape(-1)
    px, py = 21, 3
    x0, y0 = (px + 0.5) / W * 2 - 1, (py + 0.5) / H * 2 - 1
    cam.position[:] = [x0, y0, Z0 + 4.0, 1.0]
    F = W * H
    fr = {k: np.full(F, v, np.float32) for k, v in
          dict(depth=Z0, nx=0.0, ny=0.0, nz=1.0, ar=0.5, ag=0.6, ab=0.7, rough=rough).items()}
    fr["metal"] = np.full(F, 64, np.uint8)
    lights = np.zeros(2, abi.LIGHT_DTYPE)
    lights["color"] = (1.0, 2.0, 3.0, 1.0)
    lights["radius"] = 16.0
    lights["position"][0] = (0.1, 0.2, Z0 + 1.0, 1.0)
    lights["position"][1] = (x0, y0, Z0 if light == "own" else Z0 - 0.5, 1.0)
    if light.startswith("infinite"):
        lights["color"][1, 0] = np.inf
        lights["position"][1] = (0.3, -0.2, Z0 - 0.5, 1.0)
    if light == "near":
        lights["position"][1] = (x0 + 2.0 ** -18, y0, Z0 - 2.0 ** -18, 1.0)
    if light == "infinite_far":  # its attenuation of 0 times its colour
        lights["radius"][1] = 0.05
    cells = np.zeros(1, abi.CELL_DTYPE)
    cells["count"] = 2
    idx = np.arange(2, dtype=np.uint32)
    maps = random_ibl_maps(np.random.default_rng(3))
    dm = {k: to_dev(maps[k]) for k in ("spec", "diff", "lut")}
    m = abi.ibl_maps(dm["spec"], maps["spec_size"], maps["spec_mips"], dm["diff"], maps["diff_size"], dm["lut"],
                     maps["lut_w"], maps["lut_h"])
    dev = {k: to_dev(v) for k, v in fr.items()}
    rgb = torch.full((3 * F,), -1.0, dtype=torch.float32, device="cuda")
    pc = abi.pbr_defaults()
    if light == "near":
        pc.light_falloff = 8.0
    ctx.shade(abi.frag_soa(dev, W, H, ivp), cam, ubo, pc, to_dev(lights.view(np.uint8)), 2,
              to_dev(cells.view(np.int32)), to_dev(idx.view(np.int32)), m, rgb)
    torch.cuda.synchronize()
    got = rgb.cpu().numpy().reshape(3, F).T
    ref = O.shade(fr, W, H, ivp, cam, ubo, pc, lights, cells, idx, maps, np.arange(F, dtype=np.uint32))
    nan = np.isnan(ref)
    want = np.zeros((F, 3), bool)
    if light.startswith("infinite"):
        want[:, 0] = True
    else:
        want[py * W + px] = True
    assert np.array_equal(nan, want)  # the case is what it says
    assert np.array_equal(np.isnan(got), nan)
    assert O.rel_err(got[~nan], ref[~nan]) <= SHADE_TOL
