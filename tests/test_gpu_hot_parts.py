"""Refinement of large levels against the oracle, bit for bit, where the
selection keeps part ids in LDS (classes of at least 4M entries): levels held
whole (up to 65536 byte ids, 32768 of 16 bits), larger ones in the order with
the heaviest vertices first, k whose LDS rows leave room for four rows a wave,
for one, and for none.  Each case names the launches that have to be among
those of the refinement, so that none of them passes on other kernels.
(reference: hunyuangraph_GPU_krefine.h:1995-2135, 2515-2556, 3184-3241)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

HOT = {"k_hot_codes", "k_jet_select_seg_hot", "k_jet_select_w_hot", "k_jet_select_few_hot"}
SEG, W, ORDER, FEW = {"k_jet_select_seg_hot"}, {"k_jet_select_w_hot"}, {"k_hot_codes"}, {"k_jet_select_few_hot"}


def _check(hgp, orc, x, a, vw, k, hot):
    n = len(x) - 1
    rng = np.random.default_rng(k)
    aw = np.ones(len(a), np.int32)
    vw = np.ones(n, np.int32) if vw is None else vw
    ran = set()
    for heavy in (0.0, 0.3):   # balanced: LP iterations first; overweight parts: RW and RS
        where = (np.arange(n, dtype=np.int64) * k // n).astype(np.int32)
        over = rng.random(n) < heavy
        where[over] = rng.integers(0, max(1, k // 8), int(over.sum()))
        cut = orc.edge_cut(x, a, aw, where)
        hgp.ktimer_enable(True)
        g = hgp.refine(x, a, vw, aw, k, int(vw.sum()), 0, where, cut)
        ran |= set(hgp.ktimer_report())
        hgp.ktimer_enable(False)
        o = orc.dga_refine(x, a, vw, aw, k, int(vw.sum()), 0, where, cut)
        np.testing.assert_array_equal(g[0], o[0])
        assert g[1] == o[1] and g[2] == o[2]
    assert ran & HOT == hot


# (2^21 edges: no class of 4M entries)
@pytest.mark.parametrize("scale,nedges,k,hot", [
    (15, 1 << 21, 40, set()), (15, 1 << 22, 40, SEG), (15, 1 << 23, 1000, SEG), (15, 1 << 23, 1500, SEG),
    (15, 1 << 23, 1600, set()), (16, 1 << 24, 40, SEG), (17, 1 << 24, 256, ORDER | SEG | W),
    (17, 1 << 24, 257, ORDER | SEG | W), (17, 1 << 24, 400, ORDER | SEG | W), (17, 1 << 24, 1000, ORDER | SEG | W),
    (17, 1 << 24, 1400, ORDER | SEG)])
def test_selection(hgp, orc, scale, nedges, k, hot):
    x, a, vw, aw = hgp.gen_rmat(scale, nedges, seed=scale + k)
    _check(hgp, orc, x, a, vw, k, hot)


@pytest.mark.parametrize("n,degree,k,hot", [
    (65536, 90, 40, W), (32768, 190, 400, W), (32768, 190, 1000, W), (16000, 380, 40, FEW)])
def test_selection_of_middle_rows_held_whole(hgp, orc, n, degree, k, hot):
    """Rows of 33..512 entries with 4M entries or more, and hubs with at least
    an eighth of all entries but fewer than 4M."""
    rng = np.random.default_rng(n + k)
    hubs = 1000
    u = np.concatenate([rng.integers(0, n, n * degree // 2), rng.integers(0, hubs, 1500 * hubs)])
    v = rng.integers(0, n, len(u))
    u, v = u[u != v], v[u != v]
    key = np.unique(np.concatenate([u * n + v, v * n + u]))
    x = np.concatenate([[0], np.cumsum(np.bincount(key // n, minlength=n))]).astype(np.int64)
    a = (key % n).astype(np.int32)
    d = np.diff(x)
    assert int(d[d <= 512].sum()) >= 1 << 22 and len(a) // 8 <= int(d[d > 512].sum()) < 1 << 22
    _check(hgp, orc, x, a, None, k, hot)
