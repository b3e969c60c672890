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
