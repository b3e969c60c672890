"""Per-probe scratch where the card's memory is short: a reserve that does not fit
as a whole takes fewer copies, and the calls run in passes with the same results."""
import pytest

from hellovulkan_amd import abi

pytestmark = pytest.mark.gpu


def test_reserve_with_little_memory(ctx):
    import torch
    S, So, mips, n = 1024, 512, 10, 3
    levels = abi.mip_count(S)
    plan = abi.ContractPlan(ctx, abi.FILTER_SPECULAR, S, So, mips)
    gen = torch.Generator(device="cuda").manual_seed(1)
    chains = [torch.rand(abi.cube_chain_floats(S, levels), generator=gen, device="cuda") for _ in range(n)]
    outs = [torch.full((abi.cube_chain_floats(So, mips),), -1.0, device="cuda") for _ in range(n)]
    ref = torch.full_like(outs[0], -2.0)
    for c in chains:
        ctx.cube_mips(c, S, levels)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    # 200 probes' scratch is more than 9 GiB
    filler = torch.empty(torch.cuda.mem_get_info()[0] - int(8.9 * 2 ** 30), dtype=torch.uint8, device="cuda")
    try:
        plan.reserve(200)
        plan.filter_multi(n, torch.tensor([c.data_ptr() for c in chains], device="cuda"), levels,
                          torch.tensor([o.data_ptr() for o in outs], device="cuda"))
        for c, o in zip(chains, outs):
            plan.filter(c, levels, ref)
            torch.cuda.synchronize()
            assert torch.equal(o.view(torch.int32), ref.view(torch.int32))
    finally:
        del filler
        plan.close()
        torch.cuda.empty_cache()
