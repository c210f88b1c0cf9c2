"""The attraction's kernels round alike: with unit edge weights (the general form) a node gets the
bits it gets without weights, under weak gravity strong enough to show in the last place, whatever
kernel takes its row: the small graph's one launch, keys and attraction in one launch, the launch of
its own on one stream or beside others, a batch."""
import numpy as np
import pytest

from gpugraphlayout_amd import GFA2_FORCE_ATTRACTION_GRAVITY, BatchEngine, Engine, graphs

pytestmark = pytest.mark.gpu


def forces(eng, pos):
    eng.set_positions(pos)
    eng.step(1)
    eng.sync()
    return eng.forces(GFA2_FORCE_ATTRACTION_GRAVITY)


@pytest.mark.parametrize("n", [600, 3000, 20000])
def test_unit_weights_change_no_bit(n):
    print(f"case attraction rounding n={n}", flush=True)
    hub = 5000 if n == 20000 else 40            # a heavy row beside the light and medium ones
    s, t = graphs.barabasi_albert(n, 4, 3)
    g = graphs.edges_to_graph(np.concatenate([s, np.full(hub, n - 1)]), np.concatenate([t, np.arange(hub)]))
    pos = graphs.uniform_positions(g.n, 2 * np.sqrt(g.n), 4)
    params = dict(scale=2.0, gravity=50.0, edge_weight_influence=1.0)
    ones = np.ones(g.m, np.float32)
    want = None
    for weights in (None, ones):
        for mode in (0, 2):
            eng = Engine(g.n, g.src, g.dst, weights=weights, **params)
            eng.set_launch_config(256, 4, mode, mode)
            got = forces(eng, pos)
            eng.set_timing(True)                # the attraction in a launch of its own
            eng.reset()
            np.testing.assert_array_equal(forces(eng, pos).view(np.uint32), got.view(np.uint32))
            eng.close()
            if want is None:
                want = got
            np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
    eng = BatchEngine([(g.n, g.src, g.dst)] * 2, **params)
    both = forces(eng, np.concatenate([pos, pos]))
    eng.close()
    np.testing.assert_array_equal(both.view(np.uint32), np.concatenate([want, want]).view(np.uint32))
