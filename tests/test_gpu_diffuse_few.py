"""The diffuse filter on both sides of the lines up to which a workgroup takes one
texel: 640 texels from any face, and up to 2,048 where texels times face stay within
2^18. Equal to the oracle to the bit, nothing written past the map."""
import numpy as np
import pytest

from hellovulkan_amd import abi
from oracle import hvx_oracle as O
from tests.helpers import to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,Sd", [(420, 10), (430, 11), (20, 18), (20, 19), (140, 17), (151, 17), (152, 17)])
def test_lines_of_a_texel_per_workgroup(ctx, S, Sd):
    import torch
    n = 6 * Sd * Sd
    cube = np.random.default_rng(S + Sd).uniform(0, 40, 6 * S * S * 4).astype(np.float32)
    out = torch.full((4 * n + 16,), -1.0, dtype=torch.float32, device="cuda")
    ctx.filter(abi.FILTER_DIFFUSE, to_dev(cube), S, out, Sd, 1, 0)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert np.all(got[4 * n:] == -1.0)
    ids = np.unique(np.concatenate([np.arange(20), np.random.default_rng(1).integers(0, n, 200), np.arange(n - 20, n)]))
    ref = np.asarray(O.diffuse(cube, S, Sd, ids.astype(np.uint32)), np.float32)
    sub, nan = got[:4 * n].reshape(-1, 4)[ids], np.isnan(ref)
    assert np.array_equal(np.isnan(sub), nan)
    assert np.array_equal(sub[~nan].view(np.uint32), ref[~nan].view(np.uint32))
