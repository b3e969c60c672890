"""Near and far fields under the eight symmetries of a face: every one of the 48
images of rows on the octant's corners, edges and diagonal, and of some inside it,
against the FP64 twin on a cube without any symmetry of its own, in both precisions,
for one probe and for several. Faces with a narrow and a wide near level, windows
that reach past a face's edge from its own edge texels included."""
import numpy as np
import pytest

from hellovulkan_amd import abi
from oracle import hvx_oracle as O
from tests.helpers import to_dev

pytestmark = pytest.mark.gpu

# weights and radiance each rounded once to FP16: 2 x 2^-11; split BF16: each lost
# past hi + lo (2^-18), and lo * lo left out (2^-18)
TOL = {0: 1e-3, 1: 2e-5}


def _images(So, x, y):
    """Texel ids of the images of (x, y) under the square's maps on all faces."""
    ids = set()
    for a, b in ((x, y), (y, x)):
        for u in (a, So - 1 - a):
            for v in (b, So - 1 - b):
                ids.update((f * So + v) * So + u for f in range(6))
    return sorted(ids)


@pytest.mark.parametrize("precision", [abi.PRECISION_FP16_SCALED, abi.PRECISION_BF16_SPLIT])
@pytest.mark.parametrize("S,So,mips,probes", [(256, 128, 8, 1), (256, 128, 8, 3), (128, 256, 4, 1)])
def test_all_images_of_edge_and_diagonal_rows(ctx, precision, S, So, mips, probes):
    import torch
    levels = abi.mip_count(S)
    plan = abi.ContractPlan(ctx, abi.FILTER_SPECULAR, S, So, mips, precision)
    split = [m for m in range(mips) if plan.info(m).kind == abi.CONTRACT_SPLIT]
    assert split  # the case has a near and a far field
    cubes, chains, outs = [], [], []
    for p in range(probes):
        c = np.random.default_rng(S + So + p).uniform(0.1, 4.0, 6 * S * S * 4).astype(np.float32)
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
        plan.filter_multi(probes, torch.tensor([t.data_ptr() for t in chains], device="cuda"), levels,
                          torch.tensor([t.data_ptr() for t in outs], device="cuda"))
    torch.cuda.synchronize()
    plan.close()
    for p in {0, probes - 1}:
        host = outs[p].cpu().numpy()
        assert np.all(np.isfinite(host))
        for m in split:
            Sm, off = So >> m, abi.cube_level_offset_floats(So, m)
            h = Sm // 2
            rows = [(0, 0), (h - 1, h - 1), (0, h - 1), (0, 1), (h // 3, h // 3), (h // 5, h - 1), (0, h // 2), (3, h // 2)]
            ids = np.unique(np.concatenate([_images(Sm, x, y) for x, y in rows])).astype(np.uint32)
            got = host[off: off + 6 * Sm * Sm * 4].reshape(-1, 4)[ids]
            ref = O.contract(abi.FILTER_SPECULAR, cubes[p], S, So, mips, m, ids)
            assert np.all(got[:, 3] == 1.0)
            err = np.abs(got[:, :3] - ref) / np.abs(ref)
            assert err.max() <= TOL[precision], (p, m, ids[np.argmax(err.max(1))])
