"""Many probes of small outputs: from 8,192 units over all probes on, the GEMM's
workgroups stage levels that one block of rows sums each themselves. Every probe's
result equals its single call's to the bit, on both sides of that line, on faces
down to 4 texels, in both precisions, and for plans that are never taken that way."""
import numpy as np
import pytest

from hellovulkan_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ftype,S,So,mips,precision,probes", [
    (abi.FILTER_SPECULAR, 4, 4, 3, 0, 690), (abi.FILTER_SPECULAR, 8, 8, 4, 0, 171), (abi.FILTER_SPECULAR, 16, 8, 4, 0, 42),
    (abi.FILTER_SPECULAR, 16, 8, 4, 0, 43), (abi.FILTER_SPECULAR, 16, 8, 4, 1, 100), (abi.FILTER_SPECULAR, 32, 16, 5, 1, 11),
    (abi.FILTER_SPECULAR, 64, 32, 6, 0, 7), (abi.FILTER_SPECULAR, 1024, 16, 5, 0, 3), (abi.FILTER_SPECULAR, 32, 16, 2, 0, 90),
    (abi.FILTER_DIFFUSE, 8, 1, 1, 0, 200), (abi.FILTER_DIFFUSE, 64, 16, 1, 0, 37),
    # never: two blocks of rows, a near and far field, roughness 0 alone
    (abi.FILTER_SPECULAR, 64, 64, 2, 0, 12), (abi.FILTER_SPECULAR, 256, 128, 8, 1, 5), (abi.FILTER_SPECULAR, 16, 16, 1, 0, 50)])
def test_many_probes_equal_single_calls(ctx, ftype, S, So, mips, precision, probes):
    import torch
    levels = abi.mip_count(S)
    plan = abi.ContractPlan(ctx, ftype, S, So, mips, precision)
    plan.reserve(probes)
    gen = torch.Generator(device="cuda").manual_seed(S + So)
    L, O = abi.cube_chain_floats(S, levels), abi.cube_chain_floats(So, mips)
    chains = torch.rand(probes, (L + 63) // 64 * 64, generator=gen, device="cuda")
    chains *= torch.logspace(-3, 3, probes, device="cuda")[:, None]  # scales of their own
    for p in range(probes):
        ctx.cube_mips(chains[p], S, levels)
    outs = torch.full((probes, (O + 63) // 64 * 64), np.nan, device="cuda")
    plan.filter_multi(probes, torch.tensor([chains[p].data_ptr() for p in range(probes)], device="cuda"), levels,
                      torch.tensor([outs[p].data_ptr() for p in range(probes)], device="cuda"))
    ref = torch.full_like(outs, np.nan)
    for p in range(probes):
        plan.filter(chains[p], levels, ref[p])
    torch.cuda.synchronize()
    plan.close()
    assert torch.equal(outs.view(torch.int32), ref.view(torch.int32))
    assert bool(torch.isfinite(outs[:, :O]).all())
