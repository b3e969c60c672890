"""The short forms behind the environment stages: atan2 and acos equal the
double-precision functions to the bit (unit directions, every quadrant, axes,
zeros of both signs, the ends of acos' range and past them); a cube's mip chain
equals the oracle's at the sizes where a launch takes another number of levels
or tiles, alone and when only some levels are asked for; the equirect conversion
equals the oracle's at odd faces and at images narrower than a footprint."""
import ctypes as C

import numpy as np
import pytest

from hellovulkan_amd import abi
from oracle import hvx_oracle as O
from tests.helpers import to_dev
from tests.test_gpu_fastmath import LIB

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["directions", "near_axes", "ends"])
def test_angles_equal_the_double_functions(gpu, kind):
    import torch
    lib = C.CDLL(LIB)
    lib.hvxt_angles_check.argtypes = [C.c_void_p, C.c_void_p, C.c_uint32, C.c_void_p]
    g = torch.Generator(device="cuda").manual_seed(11)
    n = 1 << 24
    v = torch.randn(2, n, generator=g, device="cuda")
    if kind == "directions":
        v = v / torch.sqrt((v * v).sum(0) + torch.randn(n, generator=g, device="cuda") ** 2)
    elif kind == "near_axes":
        v[0] = v[0] * torch.exp2(-20.0 * torch.rand(n, generator=g, device="cuda"))
        v = v / torch.sqrt((v * v).sum(0))
        v[:, ::4] = v[:, ::4].flip(0)
    else:
        v = torch.tanh(8.0 * v)
        edge = torch.tensor([0.0, -0.0, 1.0, -1.0, 1.5, 0.26794919, -0.57735026, 1e-30, 0.99999994], device="cuda")
        k = torch.randint(0, 9, (2, n // 2), generator=g, device="cuda")
        v[:, : n // 2] = edge[k]
    bad = torch.zeros(2, dtype=torch.int64, device="cuda")
    y, x = v[0].contiguous(), v[1].contiguous()
    assert lib.hvxt_angles_check(y.data_ptr(), x.data_ptr(), n, bad.data_ptr()) == 0
    torch.cuda.synchronize()
    assert bad.tolist() == [0, 0]


@pytest.mark.parametrize("S,levels", [(1, 1), (2, 2), (4, 3), (16, 5), (32, 6), (32, 2), (64, 7), (128, 4), (256, 9)])
def test_mip_chain_levels(ctx, S, levels):
    import torch
    full = abi.cube_chain_floats(S, levels)
    chain = np.full(full, np.nan, np.float32)
    chain[: 6 * S * S * 4] = np.random.default_rng(S).uniform(-3, 100, 6 * S * S * 4)
    d = to_dev(np.concatenate([chain, np.full(64, 7.0, np.float32)]))
    ctx.cube_mips(d, S, levels)
    torch.cuda.synchronize()
    got = d.cpu().numpy()
    assert np.array_equal(got[:full].view(np.uint32), np.asarray(O.cube_mips(chain, S, levels)).view(np.uint32))
    assert np.all(got[full:] == 7.0)


@pytest.mark.parametrize("w,h,S", [(1, 1, 1), (2, 1, 5), (3, 2, 63), (64, 32, 64), (37, 19, 65), (256, 128, 33)])
def test_equirect_edges(ctx, w, h, S):
    import torch
    eq = np.random.default_rng(w * h).uniform(0, 50, (h, w, 4)).astype(np.float32)
    d = torch.full((6 * S * S * 4 + 16,), -1.0, dtype=torch.float32, device="cuda")
    ctx.equirect_to_cube(to_dev(eq), w, h, d, S)
    torch.cuda.synchronize()
    got = d.cpu().numpy()
    ref = np.asarray(O.equirect_to_cube(eq, S), np.float32).reshape(-1)
    assert np.array_equal(got[: 6 * S * S * 4].view(np.uint32), ref.view(np.uint32)) and np.all(got[6 * S * S * 4:] == -1.0)
