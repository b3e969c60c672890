"""The training step's block kernel at the sizes where its slices change: one
block per slice up to 32,768 samples, then 256 slices of any number of steps of 32
(33,024: four or five, across blocks; 66,048; 2 x 256 blocks). Gradient, loss and
parameters after steps equal the separate launches bit for bit (both sum the
same products over the same slices in the same order)."""
import numpy as np
import pytest
import torch

from hellovulkan_amd import abi

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.asarray(a).view(np.uint32)


@pytest.mark.parametrize("batch", [256, 768, 32768, 33024, 65536, 66048])
def test_slices_equal_separate_launches(ctx, batch):
    gen = torch.Generator(device="cuda").manual_seed(batch)
    n = 2 * batch + 77
    x = torch.randn(n, 4, generator=gen, device="cuda")
    x[:, :3] /= x[:, :3].norm(dim=1, keepdim=True)
    x[:, 3] = torch.rand(n, generator=gen, device="cuda") * 5.0
    y = torch.randn(n, 4, generator=gen, device="cuda")
    out = {}
    for separate in (1, 0):
        ctx.set_option(abi.OPT_MLP_SEPARATE_LAUNCHES, separate)
        try:
            mlp = abi.Mlp(ctx, 5.0, 3)
            g = torch.zeros(abi.MLP_PARAMS, dtype=torch.float32, device="cuda")
            loss, curve = torch.zeros(1, device="cuda"), torch.zeros(5, device="cuda")
            mlp.gradient(x, y, batch, g, loss)
            mlp.train(x, y, n, batch, 5, 2e-3, curve)
            g2 = torch.zeros_like(g)
            mlp.gradient(x, y, 256, g2, None)  # a smaller batch after a larger one
            torch.cuda.synchronize()
            out[separate] = (g.cpu(), loss.cpu(), curve.cpu(), g2.cpu(), mlp.params())
            mlp.close()
        finally:
            ctx.set_option(abi.OPT_MLP_SEPARATE_LAUNCHES, 0)
    for a, b in zip(out[0], out[1]):
        assert np.array_equal(_bits(a), _bits(b))
    assert np.all(np.isfinite(out[0][4]))
