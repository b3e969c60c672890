"""The exact fast paths of hvx_device.h that rely on their argument's range:
1 / sqrt of near-unit squared lengths from the bit pattern (every float around
1, past both ends of the pattern's range) and the correctly rounded quotient
(significands spread evenly and drawn near each other, over the exponents the
BRDF table meets) equal the compiler's IEEE operations bit for bit; and the
table itself equals the oracle's at widths around its lane counts."""
import ctypes as C

import numpy as np
import pytest

from oracle import hvx_oracle as O
from tests.test_gpu_fastmath import LIB

pytestmark = pytest.mark.gpu


def test_inv_unit_length_every_float_near_one(gpu):
    import torch
    lib = C.CDLL(LIB)
    lib.hvxt_unit_length_check.argtypes = [C.c_uint32, C.c_uint32, C.c_void_p]
    bad = torch.zeros(1, dtype=torch.int64, device="cuda")
    first = int(np.float32(0.25).view(np.uint32))
    n = int(np.float32(4.0).view(np.uint32)) - first
    assert lib.hvxt_unit_length_check(first, n, bad.data_ptr()) == 0
    torch.cuda.synchronize()
    assert int(bad.item()) == 0


def test_div_rn_normal(gpu):
    import torch
    lib = C.CDLL(LIB)
    lib.hvxt_div_check.argtypes = [C.c_void_p, C.c_void_p, C.c_uint32, C.c_void_p]
    g = torch.Generator(device="cuda").manual_seed(5)
    n = 1 << 26
    bad = torch.zeros(1, dtype=torch.int64, device="cuda")
    for k in range(4):
        sig = torch.randint(1 << 23, 1 << 24, (2, n), generator=g, device="cuda")
        if k % 2:  # quotients next to 1, where a residual is smallest
            sig[1] = (sig[0] + torch.randint(-64, 65, (n,), generator=g, device="cuda")).clamp(1 << 23, (1 << 24) - 1)
        e = torch.randint(-40, 8, (2, n), generator=g, device="cuda")
        a, b = torch.ldexp(sig.double(), e - 23).float()
        assert lib.hvxt_div_check(a.data_ptr(), b.data_ptr(), n, bad.data_ptr()) == 0
    torch.cuda.synchronize()
    assert int(bad.item()) == 0


@pytest.mark.parametrize("W,H,n", [(1, 3, 5), (63, 2, 64), (64, 5, 1025), (65, 1, 33), (256, 7, 100), (257, 3, 64),
                                   (513, 2, 128), (1024, 3, 77)])
def test_brdf_lut_is_the_oracles_to_the_bit(ctx, W, H, n):
    import torch
    d = torch.full((W * H * 2,), np.nan, dtype=torch.float32, device="cuda")
    ctx.brdf_lut(W, H, n, d)
    torch.cuda.synchronize()
    ids = np.arange(W * H, dtype=np.uint32)
    ref = np.asarray(O.brdf_lut(W, H, n, ids), np.float32).reshape(-1)
    assert np.array_equal(d.cpu().numpy().view(np.uint32), ref.view(np.uint32))
