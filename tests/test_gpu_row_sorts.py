"""The row sorts of the contraction against the oracle, bit for bit: rows at the
borders of the sorting kernels' sizes, coarse ids of one digit (up to 12 or 14
bits), just more, and three, with the smallest and the largest id in a row.
(reference: hunyuangraph_GPU_contraction.h:715-1247)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LENGTHS = [9, 33, 63, 64, 65, 128, 129, 256, 257, 512, 513, 1024, 1025, 2048, 2049, 4095, 4096, 4097, 8192, 8193, 16384]


@pytest.mark.parametrize("n", [4095, 4096, 16383, 16384, 65537, (1 << 21) + 3, (1 << 22) + 1])
@pytest.mark.parametrize("paired", [False, True])
def test_rows(hgp, orc, n, paired):
    rng = np.random.default_rng(n)
    nh = len(LENGTHS)
    src, dst = [], []
    for h, d in enumerate(LENGTHS):
        d = min(d, n - nh)
        u = nh + rng.choice(n - nh, size=d, replace=False)
        u[:2] = (nh, n - 1)
        u = np.unique(u)
        src.append(np.full(len(u), h))
        dst.append(u)
    s, t = np.concatenate(src), np.concatenate(dst)
    w = rng.integers(1, 9, size=len(s))
    s, t, w = np.concatenate([s, t]), np.concatenate([t, s]), np.concatenate([w, w])
    o = np.lexsort((t, s))
    s, a, aw = s[o], t[o].astype(np.int32), w[o].astype(np.int32)
    x = np.concatenate([[0], np.cumsum(np.bincount(s, minlength=n))]).astype(np.int64)
    vw = np.ones(n, np.int32)
    match = np.full(n, -1, np.int32)
    if paired:   # the far ends in pairs across the id range, so the concatenated rows are unsorted
        free = np.arange(nh, n)
        lo, hi = free[:len(free) // 2], free[::-1][:len(free) // 2]
        match[lo], match[hi] = hi, lo
    got, exp = hgp.contract(x, a, aw, vw, match), orc.contract(x, a, aw, vw, match)
    for g_arr, e_arr, what in zip(got, exp, ["match", "cmap", "cxadj", "cadjncy", "cadjwgt", "cvwgt"]):
        np.testing.assert_array_equal(g_arr, e_arr, err_msg=what)
