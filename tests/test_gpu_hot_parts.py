"""Refinement of large levels against the oracle, bit for bit, where the
selection keeps part ids in LDS (classes of at least 4M entries): levels held whole (up to 65536 byte ids, 32768
of 16 bits), larger ones in the order with the heaviest vertices first, k
whose LDS rows leave room for four rows a wave, for one, and for none.
(reference: hunyuangraph_GPU_krefine.h:1995-2135, 2515-2556, 3184-3241)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale,nedges,k", [(15, 1 << 21, 40), (15, 1 << 23, 1000), (15, 1 << 23, 1500),
                                            (16, 1 << 24, 40), (17, 1 << 24, 256), (17, 1 << 24, 257)])
def test_selection(hgp, orc, scale, nedges, k):
    x, a, vw, aw = hgp.gen_rmat(scale, nedges, seed=scale + k)
    n = len(x) - 1
    rng = np.random.default_rng(k)
    aw = np.ones(len(a), np.int32)
    vw = np.ones(n, np.int32) if vw is None else vw
    for heavy in (0.0, 0.3):   # balanced: LP iterations first; overweight parts: RW and RS
        where = (np.arange(n, dtype=np.int64) * k // n).astype(np.int32)
        over = rng.random(n) < heavy
        where[over] = rng.integers(0, max(1, k // 8), int(over.sum()))
        cut = orc.edge_cut(x, a, aw, where)
        g = hgp.refine(x, a, vw, aw, k, int(vw.sum()), 0, where, cut)
        o = orc.dga_refine(x, a, vw, aw, k, int(vw.sum()), 0, where, cut)
        np.testing.assert_array_equal(g[0], o[0])
        assert g[1] == o[1] and g[2] == o[2]
