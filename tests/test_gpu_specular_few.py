"""The specular filter on both sides of the line between a texel and four texels
per wave: samples around a ninth of the map's tiles, tiles around the 1,500 past
which a wave always takes four. Equal to the oracle to the bit."""
import numpy as np
import pytest

from hellovulkan_amd import abi
from oracle import hvx_oracle as O
from tests.helpers import to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,So,mips,n", [
    (64, 64, 2, 42), (64, 64, 2, 43),  # 384 tiles
    (80, 112, 2, 130), (80, 112, 2, 131),  # 1,176
    (64, 110, 4, 195), (64, 128, 2, 192)])  # 1,566 and 1,536
def test_lines_of_a_texel_per_wave(ctx, S, So, mips, n):
    import torch
    cube = np.random.default_rng(So + n).uniform(0, 30, 6 * S * S * 4).astype(np.float32)
    floats = abi.cube_chain_floats(So, mips)
    out = torch.full((floats + 16,), -1.0, dtype=torch.float32, device="cuda")
    ctx.filter(abi.FILTER_SPECULAR, to_dev(cube), S, out, So, mips, n)
    torch.cuda.synchronize()
    host = out.cpu().numpy()
    assert np.all(host[floats:] == -1.0)
    for m in range(1, mips):
        Sm, off = So >> m, abi.cube_level_offset_floats(So, m)
        ids = np.unique(np.random.default_rng(m).integers(0, 6 * Sm * Sm, 600)).astype(np.uint32)
        got = host[off:off + 6 * Sm * Sm * 4].reshape(-1, 4)[ids]
        ref = np.asarray(O.specular(cube, S, So, mips, m, n, ids), np.float32)
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), m
