"""The tied-run fix-up of the path-key sort on graphs too large for the one-block tree: runs within
a block's window, across its border, of exactly and past the 64 bodies its halo holds, alone and
per graph of a batch. Clumps of bodies contract until whole clumps share the digits the previous
tree's cells left to sort; every body order equals a numpy sort of the restated keys."""
import numpy as np
import pytest

from gpugraphlayout_amd import BatchEngine, Engine
from test_gpu_parity import FULL_SORTS_AFTER_NEW, expected_order, sorted_passes

pytestmark = pytest.mark.gpu

SIZES = [2, 3, 17, 40, 63, 64, 65, 66, 130, 300]


def clumps(count, seed):
    """`count` stars of cycling sizes, each around its own centre: (positions, src, dst)."""
    rng = np.random.default_rng(seed)
    pos, src, dst, at = [], [], [], 0
    for k in range(count):
        m = SIZES[k % len(SIZES)]
        c = rng.uniform(-300, 300, 2)
        pos.append(c + np.concatenate([[[0, 0]], rng.normal(size=(m - 1, 2)) * 0.5]))
        src.append(np.full(m - 1, at))
        dst.append(np.arange(at + 1, at + m))
        at += m
    return np.concatenate(pos).astype(np.float32), np.concatenate(src), np.concatenate(dst)


def longest_tie(order, key, bits):
    k = key[order] >> np.uint64(64 - bits)
    edge = np.flatnonzero(np.concatenate([[True], k[1:] != k[:-1], [True]]))
    return int(np.diff(edge).max())


@pytest.mark.parametrize("weight,least", [(1.0, 2), (1e7, 17), (1e9, 65), (1e14, 500)])
def test_one_graph(weight, least):
    """After the full sorts one edge gets the given weight: the bodies it flings away widen the
    root box, and the others share digits that the previous tree's cells had left to the sort."""
    print(f"case fix-up, one graph, weight {weight}", flush=True)
    pos, src, dst = clumps(90, 1)
    eng = Engine(len(pos), src, dst, scale=1e-6, gravity=0.0, strong_gravity=1, cell_factor=40,
                 edge_weight_influence=1.0)
    eng.set_edge_weights(np.ones(2 * len(src), np.float32))
    eng.set_positions(pos)
    prev, longest = None, 0
    for it in range(10):
        if it == 6:
            w = np.ones(2 * len(src), np.float32)
            w[0] = weight             # node 0's first entry
            eng.set_edge_weights(w)
        p = eng.positions()
        eng.step(1)
        eng.sync()
        tree = eng.tree()
        order, key = expected_order(p)
        np.testing.assert_array_equal(tree["perm"], order, err_msg=f"iteration {it}")
        if prev is not None and it > FULL_SORTS_AFTER_NEW:
            longest = max(longest, longest_tie(order, key, 8 * sorted_passes(prev)))
        prev = tree
    assert longest >= least
    eng.close()


def test_batch():
    print("case fix-up, batch", flush=True)
    made = [clumps(c, c) for c in (30, 10, 25, 40)]
    eng = BatchEngine([(len(p), s, t) for p, s, t in made], scale=1e-6, gravity=0.0, strong_gravity=1, cell_factor=40)
    eng.set_positions(np.concatenate([p for p, _, _ in made]))
    for it in range(14):
        p = eng.split(eng.positions())
        eng.step(1)
        eng.sync()
        perm = eng.tree()["perm"]
        for g, q in enumerate(p):
            a = eng.node_off[g]
            np.testing.assert_array_equal(perm[a:a + len(q)] - a, expected_order(q)[0], err_msg=f"iteration {it}")
    eng.close()
