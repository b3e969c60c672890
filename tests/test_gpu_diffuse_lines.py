"""The diffuse filter's staged lines hold four footprints each: faces whose rows
end at every place in a line equal the oracle to the bit, edges and corners
included."""
import numpy as np
import pytest

from hellovulkan_amd import abi
from oracle import hvx_oracle as O
from tests.helpers import to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S", [1, 2, 3, 4, 5, 7, 8, 30])
def test_rows_ending_anywhere_in_a_line(ctx, S):
    import torch
    Sd = 5
    cube = np.random.default_rng(S).uniform(0, 40, 6 * S * S * 4).astype(np.float32)
    out = torch.full((6 * Sd * Sd * 4,), np.nan, dtype=torch.float32, device="cuda")
    ctx.filter(abi.FILTER_DIFFUSE, to_dev(cube), S, out, Sd, 1, 0)
    torch.cuda.synchronize()
    ids = np.arange(6 * Sd * Sd, dtype=np.uint32)
    ref = np.asarray(O.diffuse(cube, S, Sd, ids), np.float32).reshape(-1)
    got = out.cpu().numpy()
    # the middle texels of the two Y faces look along the frame's up axis: their
    # frame is 0 / 0, and a NaN's bits are nobody's
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(got), nan) and int(nan.sum()) <= 6
    assert np.array_equal(got[~nan].view(np.uint32), ref[~nan].view(np.uint32))


@pytest.mark.parametrize("S,Sd", [(30, 9), (30, 10), (24, 26), (20, 27), (520, 10)])
def test_texels_per_workgroup(ctx, S, Sd):
    """Output maps on both sides of the sizes where a workgroup takes another
    number of texels, whole and with a last workgroup that is not full."""
    import torch
    cube = np.random.default_rng(S + Sd).uniform(0, 40, 6 * S * S * 4).astype(np.float32)
    out = torch.full((6 * Sd * Sd * 4 + 16,), -1.0, dtype=torch.float32, device="cuda")
    ctx.filter(abi.FILTER_DIFFUSE, to_dev(cube), S, out, Sd, 1, 0)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert np.all(got[6 * Sd * Sd * 4:] == -1.0)
    ids = np.unique(np.concatenate([np.arange(40), np.random.default_rng(1).integers(0, 6 * Sd * Sd, 300),
                                    np.arange(6 * Sd * Sd - 40, 6 * Sd * Sd)])).astype(np.uint32)
    ref = np.asarray(O.diffuse(cube, S, Sd, ids), np.float32)
    sub = got[:6 * Sd * Sd * 4].reshape(-1, 4)[ids]
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(sub), nan)
    assert np.array_equal(sub[~nan].view(np.uint32), ref[~nan].view(np.uint32))
