"""The contraction filter's rows are the texels of one octant of a face, each
serving its images under the square's eight symmetries on all six faces: every
output texel of a cube without any symmetry of its own against the FP64 twin,
at the sizes where the images coincide (faces of 1, 2 and 4 texels, diagonal
rows), where units are shorter than a row of the level (input faces of 4), and
where row blocks and K steps are partly filled."""
import numpy as np
import pytest

from hellovulkan_amd import abi
from oracle import hvx_oracle as O
from tests.helpers import to_dev

pytestmark = pytest.mark.gpu

# FP16 weights and radiance, each rounded once (2^-11 relative): a positive sum's
# relative error is at most the sum of the two, about 1e-3
TOL = 1e-3


@pytest.mark.parametrize("ftype,S,So,mips,probes", [
    (abi.FILTER_SPECULAR, 4, 4, 3, 1), (abi.FILTER_SPECULAR, 8, 2, 2, 3), (abi.FILTER_SPECULAR, 16, 16, 5, 1),
    (abi.FILTER_SPECULAR, 64, 8, 4, 5), (abi.FILTER_SPECULAR, 256, 64, 6, 2), (abi.FILTER_DIFFUSE, 4, 1, 1, 1),
    (abi.FILTER_DIFFUSE, 8, 2, 1, 1), (abi.FILTER_DIFFUSE, 32, 32, 1, 2), (abi.FILTER_DIFFUSE, 16, 64, 1, 1)])
def test_every_image_matches_the_twin(ctx, ftype, S, So, mips, probes):
    import torch
    levels = abi.mip_count(S)
    rng = np.random.default_rng(S * 131 + So)
    plan = abi.ContractPlan(ctx, ftype, S, So, mips)
    cubes, chains, outs = [], [], []
    for _ in range(probes):
        c = rng.uniform(0.1, 4.0, 6 * S * S * 4).astype(np.float32)
        chain = torch.empty(abi.cube_chain_floats(S, levels), dtype=torch.float32, device="cuda")
        chain[:c.size].copy_(to_dev(c))
        ctx.cube_mips(chain, S, levels)
        cubes.append(c)
        chains.append(chain)
        outs.append(torch.full((abi.cube_chain_floats(So, mips),), np.nan, dtype=torch.float32, device="cuda"))
    if probes == 1:
        plan.filter(chains[0], levels, outs[0])
    else:
        plan.reserve(probes)
        plan.filter_multi(probes, torch.tensor([t.data_ptr() for t in chains], dtype=torch.int64, device="cuda"),
                          levels, torch.tensor([t.data_ptr() for t in outs], dtype=torch.int64, device="cuda"))
    torch.cuda.synchronize()
    for c, o in zip(cubes, outs):
        host = o.cpu().numpy()
        for m in range(mips):
            Sm, off = max(So >> m, 1), abi.cube_level_offset_floats(So, m)
            got = host[off: off + 6 * Sm * Sm * 4].reshape(-1, 4)
            ids = np.arange(6 * Sm * Sm, dtype=np.uint32)
            if ids.size > 3000:
                ids = np.unique(rng.integers(0, ids.size, 3000)).astype(np.uint32)
            ref = O.contract(ftype, c, S, So, mips, m, ids)
            assert np.all(got[:, 3] == 1.0)
            assert O.rel_err(got[ids, :3], ref) <= TOL, (m, Sm)
    plan.close()
