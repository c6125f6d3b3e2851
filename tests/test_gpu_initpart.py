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


def test_dense_trials_run(hgp):
    """The stage entry point has room for the matrices of up to 4096 vertices."""
    for n, dense in ((2, True), (4096, True), (4097, False)):
        x, a, vw, aw = _graph(n, n, clusters=False)
        hgp.ktimer_enable(True)
        hgp.initpart(x, a, vw, aw, 2, seed=5, trials=3)
        ran = hgp.ktimer_report()
        hgp.ktimer_enable(False)
        assert ("k_ip_dense" in ran) == dense, n


def test_matrices_yield_to_the_memory_there_is(hgp, orc):
    """The dense trials' matrices (68 MB here) are taken only where the arena
    has the room: a graph whose coarsening stops after one step, at 4050
    vertices, is served within a budget that its lists need a few MB of, and
    with its matrices, at the first go, where the budget has the room."""
    n = 8100
    pairs, links = [(v, v + 1) for v in range(0, n, 2)], [(v + 1, v + 2) for v in range(0, 3600, 4)]
    x, a, aw = csr_from_edges(n, pairs + links, [5] * len(pairs) + [1] * len(links))
    vw = np.ones(n, np.int32)
    ref, _ = orc.dga_partition(x, a, 2, vw, aw, seed=3)
    for budget, dense in ((71_000_000, False), (1 << 30, True)):
        hgp.ktimer_enable(True)
        with hgp.Server(slots=1, budget_bytes=budget) as s:
            part, st, _ = s.wait(s.submit(x, a, 2, vw, aw, seed=3))
        ran = hgp.ktimer_report()
        hgp.ktimer_enable(False)
        assert st["coarsest_n"] == 4050
        np.testing.assert_array_equal(part, ref)
        assert ran.get("k_ip_dense", (0,))[0] == int(dense)
        assert ran["k_ip_trials"][0] == 1 and st["arena_bytes"] < 90_000_000


def test_list_trials_within_a_budget(hgp):
    """A thousand trials on the lists of a coarsest graph of 15600 vertices take
    226 MB of scratch, 14 B a vertex and trial: served within 262 MB."""
    n = 31200
    pairs, links = [(v, v + 1) for v in range(0, n, 2)], [(v + 1, v + 2) for v in range(0, 14000, 4)]
    x, a, aw = csr_from_edges(n, pairs + links, [5] * len(pairs) + [1] * len(links))
    vw = np.ones(n, np.int32)
    ref, _ = hgp.partition(x, a, 2, vw, aw, seed=3)
    with hgp.Server(slots=1, budget_bytes=262_000_000) as s:
        part, st, _ = s.wait(s.submit(x, a, 2, vw, aw, seed=3))
    assert st["coarsest_n"] == 15600
    np.testing.assert_array_equal(part, ref)
