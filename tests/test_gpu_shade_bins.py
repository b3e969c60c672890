"""Binning of the fragments at the sizes where it takes another way: tiles of
up to 16,384 pixels (counted once) and beyond, more tiles than CUs (segments put
together in LDS) and fewer, tiles narrower and wider than a workgroup's step,
one pixel. The exact variant equals the oracle to the bit at every pixel."""
import numpy as np
import pytest

from hellovulkan_amd import abi
from tests.test_gpu_cf import _shade_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height,grid", [
    (1, 1, (1, 1, 1)), (128, 128, (1, 1, 4)), (130, 127, (1, 1, 4)), (2100, 9, (1, 1, 3)), (300, 260, (17, 16, 6)),
    (700, 130, (257, 1, 5)), (190, 340, (2, 1, 512))])
def test_every_pixel_of_every_tile(ctx, width, height, grid):
    ctx.set_option(abi.OPT_SHADE_EXACT, 1)
    try:
        got, ref, _ = _shade_case(ctx, width, height, grid, 60, 32, 51, None)
    finally:
        ctx.set_option(abi.OPT_SHADE_EXACT, 0)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
