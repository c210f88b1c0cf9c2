"""A network handle's graphs share memory one after another: graphs added, released and added again
in blocks that are kept, too small, less than half used or another graph's give what a fresh handle
gives, with and without a target; an engine's graph, whose row lists are the engine's, gives the
bits of the same graph from the host."""
import numpy as np
import pytest

from gpugraphlayout_amd import Engine, Mpnn, graphs

pytestmark = pytest.mark.gpu


def csr(n, hub):
    """A ring with a hub of the given length and rows of 33 to 40 entries beside it."""
    i = np.arange(n)
    a, b = [i], [(i + 1) % n]
    a.append(np.zeros(hub, np.int64))
    b.append(2 + np.arange(hub))
    for k in range(8):
        a.append(np.full(31 + k, 5 + 60 * k))
        b.append((5 + 60 * k + 2 + np.arange(31 + k)) % n)
    return graphs.edges_to_graph(np.concatenate(a), np.concatenate(b))


def outcome(m, g, seed, target):
    rowptr, col = g.csr()
    T = np.random.default_rng(seed).normal(size=(g.n, 2)).astype(np.float32) if target else None
    gid = m.add_graph(g.n, rowptr, col, target=T, feature_seed=seed, steps=1)
    out = [m.features(gid), m.infer(gid, 10.0)]
    if target:
        out += [np.array(x) for x in m.loss_grad(gid, [1, 3])]
    return gid, out


def test_blocks_kept_and_grown():
    print("case mpnn blocks", flush=True)
    m, held = Mpnn(seed=1), []
    for k, (n, hub) in enumerate([(3000, 2500), (3000, 2500), (2000, 100), (600, 0), (9000, 6000), (600, 40), (9000, 8998)]):
        g = csr(n, hub)
        gid, got = outcome(m, g, k, k % 2 == 1)
        fresh = Mpnn(seed=1)
        _, want = outcome(fresh, g, k, k % 2 == 1)
        for x, y in zip(got, want):
            np.testing.assert_array_equal(x, y, err_msg=f"graph {k}")
        fresh.close()
        held.append((gid, got[0]))
        if k in (2, 4):          # two graphs stay while others take blocks
            for kept, X in held[-1:]:
                np.testing.assert_array_equal(m.features(kept), X)
        else:
            m.release_graph(gid)
    for k in (2, 4):
        np.testing.assert_array_equal(m.features(held[k][0]), held[k][1])
    m.close()


@pytest.mark.parametrize("n,hub", [(700, 0), (700, 600), (3000, 2046), (3000, 2049), (9000, 8900)])
def test_engine_rows_are_the_host_rows(n, hub):
    print(f"case mpnn engine rows n={n} hub={hub}", flush=True)
    g = csr(n, hub)
    m, eng = Mpnn(seed=2), Engine(g.n, g.src, g.dst)
    rowptr, col = g.csr()
    a = m.add_graph(g.n, rowptr, col, feature_seed=9, steps=2)
    b = m.add_engine_graph(eng, feature_seed=9, steps=2)
    eng.close()                  # the graph holds copies
    np.testing.assert_array_equal(m.features(a), m.features(b))
    np.testing.assert_array_equal(m.infer(a, 5.0), m.infer(b, 5.0))
    m.close()
