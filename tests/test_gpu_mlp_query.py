"""Queries of the network around the tiles (16), steps (128) and full launches of
its kernel: the results do not depend on how many samples the call holds, so a
call equals the same samples asked for in pieces, to the bit, and nothing is
written past the last."""
import numpy as np
import pytest
import torch

from hellovulkan_amd import abi

pytestmark = pytest.mark.gpu

FULL = 128 * 4 * 256  # samples of the largest call with one step per workgroup


@pytest.mark.parametrize("n", [1, 15, 64, 129, 1000, FULL - 1, FULL, FULL + 1, 2 * FULL + 97])
def test_query_does_not_depend_on_the_call(ctx, n):
    gen = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn(n, 4, generator=gen, device="cuda")
    x[:, :3] /= x[:, :3].norm(dim=1, keepdim=True)
    x[:, 3] = torch.rand(n, generator=gen, device="cuda") * 6.0
    mlp = abi.Mlp(ctx, 6.0, 5)
    out = torch.full((3 * n + 8,), np.nan, device="cuda")
    mlp.eval(x, n, out)
    parts = torch.full((3 * n + 8,), np.nan, device="cuda")
    step = 777 if n > 64 else 7
    for a in range(0, n, step * max(1, n // (20 * step))):
        m = min(step * max(1, n // (20 * step)), n - a)
        mlp.eval(x[a:].contiguous(), m, parts[3 * a:])
    torch.cuda.synchronize()
    mlp.close()
    assert torch.equal(out.view(torch.int32), parts.view(torch.int32))
    assert bool(torch.isfinite(out[:3 * n]).all()) and bool(torch.isnan(out[3 * n:]).all())
