"""Hop distances of the multi-source search at the edges of its launch rules: every row width
(64 sources per word, up to 16 words, several passes beyond), light, medium and heavy rows (a
hub of more than one chunk), rows that are done early, and searches longer than one batch of
levels. Distances are whole numbers: equal to the oracle's."""
import numpy as np
import pytest

from gpugraphlayout_amd import Engine, coo_to_csr

pytestmark = pytest.mark.gpu


def hub_graph(n):
    """Node 0 next to most nodes, node 1 to 300, a sparse rest, the last 5 nodes on their own."""
    rng = np.random.default_rng(4)
    s = [np.zeros(n - 400, np.int64), np.ones(300, np.int64), rng.integers(0, n - 5, n // 2), [n - 4]]
    t = [np.arange(2, n - 398), np.arange(n - 400, n - 100), rng.integers(0, n - 5, n // 2), [n - 3]]
    s, t = np.concatenate(s), np.concatenate(t)
    key = np.unique(np.minimum(s, t)[s != t] * n + np.maximum(s, t)[s != t])
    return n, (key // n).astype(np.int32), (key % n).astype(np.int32)


def path_graph(n):
    return n, np.arange(n - 1, dtype=np.int32), np.arange(1, n, dtype=np.int32)


@pytest.mark.parametrize("graph,sources", [(hub_graph(6000), k) for k in (1, 64, 65, 200, 400, 1000, 1024, 1500)]
                         + [(path_graph(50), 50), (hub_graph(2600), 4000)])
def test_hop_distances(oracle, graph, sources):
    n, s, t = graph
    print(f"case bfs n={n} sources={sources}", flush=True)
    eng = Engine(n, s, t)
    npairs = eng.stress_setup(sources, 40, seed=sources)
    a, b, d = eng.stress_pairs()
    assert len(a) == 40 * min(sources, n) and npairs == int((d > 0).sum())
    src = a[::40]
    assert len(np.unique(src)) == len(src) and np.all(a != b)
    rowptr, col = coo_to_csr(n, s, t)
    step = max(1, len(src) // 60)
    for k in sorted(set(range(0, len(src), step)) | {len(src) - 1}):
        ref = oracle.bfs(rowptr, col, int(src[k]))
        sel = slice(40 * k, 40 * k + 40)
        np.testing.assert_array_equal(d[sel], np.maximum(ref[b[sel]], 0))
    eng.close()
