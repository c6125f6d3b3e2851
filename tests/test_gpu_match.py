"""The proposals of the handshake matching against the oracle, bit for bit:
rows at the borders of the degree classes and of the segments, where the best
entries of a row lead to neighbours that are too heavy or taken, so that a
group's lone lookups fail and its lanes look their entries up.
(reference: hunyuangraph_GPU_match.h:454-510, 800-861)"""
import numpy as np
import pytest

from conftest import csr_from_edges

pytestmark = pytest.mark.gpu

DEGREES = [1, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 129, 511, 512, 513, 1023, 1025, 2047, 2048, 2049, 4097]


@pytest.mark.parametrize("wmax", [1, 3, 20000])
@pytest.mark.parametrize("heavy", [0.0, 0.5, 0.97])
def test_rows_with_refused_neighbours(hgp, orc, wmax, heavy):
    rng = np.random.default_rng(wmax % 1000 + int(100 * heavy))
    n = 6000
    edges = {}
    for v, d in enumerate(DEGREES):
        for u in rng.choice(np.arange(len(DEGREES), n), size=d, replace=False):
            edges[(v, int(u))] = int(rng.integers(1, wmax + 1)) if wmax > 1 else 1
    x, a, w = csr_from_edges(n, list(edges), list(edges.values()))
    vw = np.where(rng.random(n) < heavy, 99, rng.integers(1, 3, size=n)).astype(np.int32)
    for rounds in (1, 2, 8):
        m_g, c_g = hgp.match(x, a, vw, w, 100, 5, 1, rounds)
        m_o, c_o = orc.dga_match(x, a, vw, w, 100, 5, 1, rounds)
        np.testing.assert_array_equal(m_g, m_o)
        assert c_g == c_o
