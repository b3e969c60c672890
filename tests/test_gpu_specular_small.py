"""The specular filter of small maps (a texel per wave) and of maps just past the
size where a wave takes four: sample counts around a round's 64, faces of every
remainder of a tile, one mip's single texel. Equal to the oracle to the bit."""
import numpy as np
import pytest

from hellovulkan_amd import abi
from oracle import hvx_oracle as O
from tests.helpers import to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,So,mips,n", [(8, 2, 2, 1), (16, 5, 3, 63), (16, 6, 3, 64), (32, 11, 4, 65), (40, 24, 5, 200),
                                         (120, 110, 3, 70), (120, 116, 3, 70)])
def test_every_mip_is_the_oracles(ctx, S, So, mips, n):
    import torch
    cube = np.random.default_rng(So).uniform(0, 30, 6 * S * S * 4).astype(np.float32)
    floats = abi.cube_chain_floats(So, mips)
    out = torch.full((floats + 16,), -1.0, dtype=torch.float32, device="cuda")
    ctx.filter(abi.FILTER_SPECULAR, to_dev(cube), S, out, So, mips, n)
    torch.cuda.synchronize()
    host = out.cpu().numpy()
    assert np.all(host[floats:] == -1.0)
    for m in range(mips):
        Sm = max(So >> m, 1)
        off = abi.cube_level_offset_floats(So, m)
        got = host[off:off + 6 * Sm * Sm * 4].reshape(-1, 4)
        ids = np.arange(6 * Sm * Sm, dtype=np.uint32)
        if ids.size > 800:
            ids = np.unique(np.concatenate([ids[:50], np.random.default_rng(m).integers(0, ids.size, 500), ids[-50:]])).astype(np.uint32)
        ref = np.asarray(O.specular(cube, S, So, mips, m, n, ids), np.float32)
        sub, nan = got[ids], np.isnan(ref)
        assert np.array_equal(np.isnan(sub), nan)
        assert np.array_equal(sub[~nan].view(np.uint32), ref[~nan].view(np.uint32)), m
