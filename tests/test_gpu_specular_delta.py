"""The roughness-0 mip at the sample counts where its equal terms are summed in
another way (430 one by one, 431 a binade at a time) and around the first of them,
by the filter and in a batch: equal to the oracle to the bit, dark and bright texels."""
import numpy as np
import pytest

from hellovulkan_amd import abi
from oracle import hvx_oracle as O
from tests.helpers import to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 430, 431, 1023])
def test_roughness_zero_sums(ctx, n):
    import torch
    S, So = 24, 13
    rng = np.random.default_rng(n)
    cube = (rng.uniform(0, 1, 6 * S * S * 4) * 10.0 ** rng.integers(-6, 7, 6 * S * S * 4)).astype(np.float32)
    d = to_dev(cube)
    out, again = (torch.full((6 * So * So * 4,), -1.0, dtype=torch.float32, device="cuda") for _ in range(2))
    ctx.filter(abi.FILTER_SPECULAR, d, S, out, So, 1, n)
    b = abi.Batch(ctx, [abi.probe(d, S, again, So, 1)], n, [])
    b.run()
    torch.cuda.synchronize()
    b.close()
    ids = np.arange(6 * So * So, dtype=np.uint32)
    ref = np.asarray(O.specular(cube, S, So, 1, 0, n, ids), np.float32)
    for o in (out, again):
        assert np.array_equal(o.cpu().numpy().reshape(-1, 4).view(np.uint32), ref.view(np.uint32))
