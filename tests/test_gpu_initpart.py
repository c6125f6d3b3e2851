"""The bisection trials' paths against the oracle, bit for bit: the dense
trials at the edges of their thread layouts (one wave up to 256 vertices of a
node, 256 threads up to 2048, 512 threads up to 4096; one and two bit-matrix
words per lane), and the list trials past 4096 vertices and for rows that do
not ascend.  (reference: hunyuangraph_GPU_initialpartition.h:2426-3659)"""
import numpy as np
import pytest

from conftest import csr_from_edges

pytestmark = pytest.mark.gpu


def _graph(n, seed, clusters=True):
    """Sparse random edges and a dense cluster, isolated vertices and a second
    component, weights 1..9."""
    rng = np.random.default_rng(seed)
    e = {(int(a), int(b)) for a, b in np.sort(rng.integers(0, max(2, n - 3), (3 * n, 2)), axis=1) if a != b}
    if clusters:
        c = rng.choice(n, min(n, 40), replace=False)
        e |= {(int(min(a, b)), int(max(a, b))) for a in c for b in c if a != b and rng.random() < 0.5}
    edges = sorted(e)
    x, a, aw = csr_from_edges(n, edges, rng.integers(1, 10, len(edges)))[:3]
    return x, a, rng.integers(1, 5, n).astype(np.int32), aw


@pytest.mark.parametrize("n", [2, 5, 31, 64, 65, 255, 256, 257, 1023, 1024, 1025, 2047, 2048, 2049, 4095, 4096, 4097])
def test_trials_by_size(hgp, orc, n):
    x, a, vw, aw = _graph(n, n)
    for k, trials in ((2, 6), (7, 3)):
        w = hgp.initpart(x, a, vw, aw, k, seed=5, trials=trials)
        o = orc.dga_initpart(x, a, vw, aw, k, seed=5, trials=trials)
        np.testing.assert_array_equal(w, o, err_msg=f"n={n} k={k}")


@pytest.mark.parametrize("n", [60, 300, 1500])
def test_trials_of_rows_out_of_order(hgp, orc, n):
    x, a, vw, aw = _graph(n, n + 1)
    a, aw = a.copy(), aw.copy()
    for v in range(n):   # every row reversed
        a[x[v]:x[v + 1]] = a[x[v]:x[v + 1]][::-1]
        aw[x[v]:x[v + 1]] = aw[x[v]:x[v + 1]][::-1]
    w = hgp.initpart(x, a, vw, aw, 5, seed=2, trials=8)
    o = orc.dga_initpart(x, a, vw, aw, 5, seed=2, trials=8)
    np.testing.assert_array_equal(w, o)
