"""A network handle after a graph too large for the device: the error is reported once, the graphs
that were there give what they gave, and new ones fit."""
import numpy as np
import pytest

from gpugraphlayout_amd import Engine, GFA2Error, Mpnn, graphs

pytestmark = pytest.mark.gpu


def test_handle_survives_a_graph_that_does_not_fit():
    """300M nodes need 485 GB of scratch; the device has 288."""
    print("case mpnn out of memory", flush=True)
    s, t = graphs.barabasi_albert(3000, 4, 1)
    g = graphs.edges_to_graph(s, t)
    rowptr, col = g.csr()
    target = graphs.uniform_positions(g.n, 50.0, 2)
    m, eng = Mpnn(seed=3), Engine(g.n, g.src, g.dst)

    def results(gid):
        loss, grad = m.loss_grad(gid, [1, 5])
        m.infer_to_engine(gid, 10.0, eng)
        return [np.array(loss), grad, m.infer(gid, 10.0), eng.positions()]

    first = m.add_graph(g.n, rowptr, col, target=target, feature_seed=4, steps=1)
    want = results(first)
    with pytest.raises(GFA2Error) as ei:
        m.add_graph(300_000_000, np.zeros(300_000_001, np.int64), np.zeros(0, np.int32), feature_seed=1, steps=0)
    assert ei.value.code == -2
    second = m.add_graph(g.n, rowptr, col, target=target, feature_seed=4, steps=1)
    for gid in (first, second):
        for x, y in zip(results(gid), want):
            np.testing.assert_array_equal(x, y)
    m.train(3, 1e-3, 2, 1)
    # the scratch gone, the first graph's use brings it back
    with pytest.raises(GFA2Error):
        m.add_graph(300_000_000, np.zeros(300_000_001, np.int64), np.zeros(0, np.int32), feature_seed=1, steps=0)
    assert np.isfinite(m.infer(first, 10.0)).all()
    m.close()
    eng.close()
