"""Training that changes between the fused step and the separate launches from call
to call, and parameters set between them: the separate launches' transposed weights
and encodings follow, so the parameters equal those of fused steps alone bit for
bit, whether a call revisits its samples (encoded once) or not."""
import numpy as np
import pytest

from hellovulkan_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,epochs", [(256, 3), (1024, 1), (33024, 2)])
def test_changing_between_the_two_ways(ctx, batch, epochs):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(batch)
    n = epochs * batch + 19
    x = torch.randn(n, 4, generator=gen, device="cuda")
    x[:, :3] /= x[:, :3].norm(dim=1, keepdim=True)
    x[:, 3] = torch.rand(n, generator=gen, device="cuda") * 5.0
    y = torch.randn(n, 4, generator=gen, device="cuda")
    out = []
    for ways in ((0, 0, 0, 0, 0), (1, 0, 1, 1, 0), (0, 1, 0, 1, 1)):
        mlp = abi.Mlp(ctx, 5.0, 3)
        try:
            for k, separate in enumerate(ways):
                ctx.set_option(abi.OPT_MLP_SEPARATE_LAUNCHES, separate)
                if k == 3:
                    mlp.set_params(mlp.params() * np.float32(0.5))
                # one step less than an epoch, then several epochs
                mlp.train(x, y, n, batch, 1 if k % 2 else 2 * epochs + 1, 2e-3, None)
            g = torch.zeros(abi.MLP_PARAMS, device="cuda")
            mlp.gradient(x, y, batch, g, None)
            out.append((mlp.params(), g.cpu().numpy()))
        finally:
            ctx.set_option(abi.OPT_MLP_SEPARATE_LAUNCHES, 0)
            mlp.close()
    assert np.all(np.isfinite(out[0][0]))
    for o in out[1:]:
        for a, b in zip(out[0], o):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
