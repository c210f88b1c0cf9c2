"""Keys and attraction in one launch against the two launches that timing asks for: positions and
forces equal bit for bit over several iterations, for sizes on either side of the sort's forms, rows of
every class, weights and logarithmic attraction, graph capture, and batches."""
import numpy as np
import pytest

from gpugraphlayout_amd import GFA2_FORCE_ATTRACTION_GRAVITY, BatchEngine, Engine, graphs

pytestmark = pytest.mark.gpu


def edges(n, hub, seed):
    rng = np.random.default_rng(seed)
    s, t = rng.integers(0, n, (2, 3 * n))
    s, t = np.concatenate([s, np.zeros(hub, np.int64)]), np.concatenate([t, rng.permutation(n)[:hub]])
    s, t = np.concatenate([s, np.full(min(n, 60), 1)]), np.concatenate([t, rng.permutation(n)[:60]])
    key = np.unique(np.minimum(s, t)[s != t] * n + np.maximum(s, t)[s != t])
    return (key // n).astype(np.int32), (key % n).astype(np.int32)


def run(eng, pos, timing, capture=False):
    eng.set_graph_capture(capture)
    eng.set_timing(timing)
    eng.set_positions(pos)
    eng.reset()
    out = []
    for _ in range(3):
        eng.step(2)
        eng.sync()
        out.append((eng.positions(), eng.forces(), eng.forces(GFA2_FORCE_ATTRACTION_GRAVITY)))
    return out


def compare(make, pos, captured):
    eng = make()
    want = run(eng, pos, True)
    for capture in ((False, True) if captured else (False,)):
        for a, b in zip(run(eng, pos, False, capture), want):
            for x, y in zip(a, b):
                np.testing.assert_array_equal(x, y)
    eng.close()


@pytest.mark.parametrize("n,hub,linlog,weighted", [(4097, 0, 0, False), (5000, 4500, 1, True), (33_000, 9000, 0, True),
                                                   (70_000, 2100, 0, False), (263_000, 2100, 1, False)])
def test_one_graph(n, hub, linlog, weighted):
    print(f"case keys and attraction n={n} hub={hub} linlog={linlog} weighted={weighted}", flush=True)
    s, t = edges(n, hub, n)
    w = np.random.default_rng(1).uniform(0.25, 4.0, len(s)).astype(np.float32) if weighted else None
    compare(lambda: Engine(n, s, t, weights=w, scale=2.0, linlog=linlog, edge_weight_influence=1.0, strong_gravity=1),
            graphs.uniform_positions(n, 2 * np.sqrt(n), 3), n < 100_000)


@pytest.mark.parametrize("sizes", [[5000, 1, 300, 2], [34_000, 40, 1]])
def test_batch(sizes):
    print(f"case keys and attraction batch {sizes}", flush=True)
    gs = [(n, *edges(n, min(n - 1, 2500), n)) if n > 60 else (n, np.arange(n - 1, dtype=np.int32), np.arange(1, n, dtype=np.int32))
          for n in sizes]
    pos = np.concatenate([graphs.uniform_positions(n, 2 * np.sqrt(n), k) for k, n in enumerate(sizes)])
    compare(lambda: BatchEngine(gs, scale=2.0, strong_gravity=1), pos, True)
