"""Work items of a probe batch: every texel of mip 0 and every tile of the other
mips exactly once, and every XCD the same share (to an item) of every mip, so that
mips of different cost keep none of the XCDs waiting."""
import ctypes as C
import os

import numpy as np
import pytest

from hellovulkan_amd.build import TEST_KERNELS_LIB


def _items(faces, mips, samples, texels, slots):
    if not os.path.exists(TEST_KERNELS_LIB):
        pytest.skip("test kernels not built")
    lib = C.CDLL(TEST_KERNELS_LIB)
    lib.hvxt_probe_items.restype = C.c_uint32
    cap = 1 << 20
    buf = np.zeros((cap, 4), np.uint32)
    begin, one = np.zeros(9, np.uint32), np.zeros(1, np.uint32)
    f, m = np.asarray(faces, np.uint32), np.asarray(mips, np.uint32)
    p = lambda a: a.ctypes.data_as(C.c_void_p)
    n = lib.hvxt_probe_items(p(f), p(m), len(faces), samples, texels, slots, p(buf), cap, p(begin), p(one))
    assert n <= cap and begin[0] == 0 and begin[8] == n and np.all(np.diff(begin.astype(np.int64)) >= 0)
    return buf[:n].astype(np.int64), begin.astype(np.int64), bool(one[0])


@pytest.mark.parametrize("faces,mips,samples,texels,slots", [
    ([256], [9], 1024, 256, 1024), ([512], [10], 1024, 8192, 256), ([16], [5], 1024, 256, 1024),
    ([1], [1], 1, 32, 256), ([32, 64, 128, 256], [6, 7, 8, 9], 1024, 64, 2048), ([50, 7, 300], [6, 3, 9], 100, 100, 1024),
    ([8] * 37, [4] * 37, 64, 256, 1024), ([110], [3], 1024, 256, 1024)])
def test_items_cover_and_balance(faces, mips, samples, texels, slots):
    items, begin, one = _items(faces, mips, samples, texels, slots)
    tw, th = (1, 4) if one else (4, 4)
    tiles4 = sum(6 * ((max(f >> m, 1) + 3) // 4) ** 2 for f, k in zip(faces, mips) for m in range(1, k))
    assert one == (tiles4 <= 1500 and 9 * samples >= tiles4)
    xcd = np.searchsorted(begin[1:], np.arange(len(items)), side="right")
    for kind in (0, 1):  # what is left over of the mips goes round the XCDs
        per = np.bincount(xcd[(items[:, 1] > 0) == kind], minlength=8)
        assert per.max() - per.min() <= 1
    for p, (f, k) in enumerate(zip(faces, mips)):
        for m in range(k):
            s = max(f >> m, 1)
            total = 6 * s * s if m == 0 else 6 * ((s + tw - 1) // tw) * ((s + th - 1) // th)
            mine = (items[:, 0] == p) & (items[:, 1] == m)
            it = items[mine]
            order = np.argsort(it[:, 2])
            ends = np.concatenate([[0], (it[order, 2] + it[order, 3])])
            assert np.array_equal(it[order, 2], ends[:-1]) and ends[-1] == total and np.all(it[:, 3] > 0)
            assert it[:, 3].max() * (1 if m == 0 else tw * th) <= max(texels, tw * th)
            per = np.bincount(xcd[mine], minlength=8)
            assert per.max() - per.min() <= 1
