"""The rebalancing step against the oracle, bit for bit, at the edges of its
paths: one block with 4, 8 and 16 rows a wave (4096, 8192 and 16384 vertices),
tiles that sum the digit counts themselves and past 64 tiles (262144 vertices),
parts that need one, two and three digit passes, k past 1024 (no block path),
weights that make the slices of the evicted list short and long.
(reference: hunyuangraph_GPU_krefine.h:2515-2766, 3243-3366)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(hgp, orc, n_side, k, wmax, heavy, seed):
    x, a, vw, aw = hgp.gen_grid2d(*n_side)
    n = len(x) - 1
    rng = np.random.default_rng(seed)
    vw = rng.integers(1, wmax + 1, n).astype(np.int32)
    aw = aw.copy()
    # a few parts hold most of the graph: RW and RS iterations from the start
    where = np.minimum(np.arange(n, dtype=np.int64) * k // n, k - 1).astype(np.int32)
    over = rng.random(n) < heavy
    where[over] = rng.integers(0, max(1, k // 8), int(over.sum()))
    tv = int(vw.sum())
    cut = orc.edge_cut(x, a, aw, where)
    for finest in (0, 1):
        g = hgp.refine(x, a, vw, aw, k, tv, finest, where, cut)
        o = orc.dga_refine(x, a, vw, aw, k, tv, finest, where, cut)
        np.testing.assert_array_equal(g[0], o[0], err_msg=f"n={n} k={k} wmax={wmax} finest={finest}")
        assert g[1] == o[1] and g[2] == o[2]


# (513..): just above the levels that one block refines whole
@pytest.mark.parametrize("side", [(27, 19), (64, 64), (17, 241), (64, 128), (8193, 1), (128, 128), (5462, 3), (400, 655),
                                  (512, 512), (262145, 1)])
@pytest.mark.parametrize("k", [3, 40])
def test_sizes(hgp, orc, side, k):
    _check(hgp, orc, side, k, 4, 0.5, side[0] * side[1] + k)


@pytest.mark.parametrize("k,side", [(5, (100, 100)), (6, (100, 100)), (1024, (120, 130)), (1025, (120, 130)),
                                    (1400, (150, 150)), (4096, (200, 210))])
def test_parts(hgp, orc, k, side):
    _check(hgp, orc, side, k, 3, 0.4, k)


@pytest.mark.parametrize("wmax,heavy", [(1, 0.9), (1000, 0.9), (100000, 0.3), (2, 0.05)])
@pytest.mark.parametrize("side", [(60, 60), (300, 310)])
def test_weights(hgp, orc, side, wmax, heavy):
    _check(hgp, orc, side, 17, wmax, heavy, wmax)
