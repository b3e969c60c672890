"""The sum of n equal floats by whole binades equals the n additions bit for
bit: terms of every exponent and sign (zeros, subnormals, the largest, infinite
and NaN among them), short significands and ones that lie halfway between two
multiples of a binade's spacing, counts around the first additions and to 4,096."""
import ctypes as C

import pytest

from tests.test_gpu_fastmath import LIB

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["any", "unit", "subnormal", "largest", "short", "halfway"])
def test_repeat_sum_equals_the_additions(gpu, kind):
    import torch
    lib = C.CDLL(LIB)
    lib.hvxt_repeat_sum_check.argtypes = [C.c_void_p, C.c_void_p, C.c_uint32, C.c_void_p]
    g = torch.Generator(device="cuda").manual_seed(7)
    n = 1 << 20
    u = torch.randint(0, 1 << 32, (n,), generator=g, device="cuda")
    sign = u & 0x80000000
    if kind == "unit":
        u = sign | 0x3F800000 | (u & 0x7FFFFF)
    elif kind == "subnormal":
        u = sign | (u % 4096)
    elif kind == "largest":
        u = sign | 0x7E000000 | (u & 0x1FFFFFF)
    elif kind == "short":
        u = u & 0xFFF00000
    elif kind == "halfway":
        u = (u & 0xFF800000) | ((1 << (u % 23)) + (u >> 9) % 3 - 1)
    counts = torch.randint(0, 4097, (n,), generator=g, device="cuda")
    counts[: n // 4] %= 40
    bad = torch.zeros(1, dtype=torch.int64, device="cuda")
    terms, counts = u.to(torch.uint32), counts.to(torch.uint32)
    assert lib.hvxt_repeat_sum_check(terms.data_ptr(), counts.data_ptr(), n, bad.data_ptr()) == 0
    torch.cuda.synchronize()
    assert int(bad.item()) == 0
