"""What the autotuner records for graphs whose launch shape does not place the attraction (small
graphs, all pairs): the place that others of the bucket measured, or the default, never one of
several equal ones."""
import ctypes

import numpy as np
import pytest

from gpugraphlayout_amd import Engine, LaunchConfig, graphs, lib

pytestmark = pytest.mark.gpu


def recorded(n):
    c = LaunchConfig()
    rc = lib().gfa2_tuned_config(n, ctypes.byref(c))
    return None if rc else (c.attraction_stream, c.attraction_blocks_per_cu)


def tune(n, **params):
    s, t = graphs.barabasi_albert(n, 3, n)
    eng = Engine(n, s, t, scale=2.0, **params)
    eng.set_positions(graphs.uniform_positions(n, 2 * np.sqrt(n), 1))
    best = eng.autotune(2)
    shape = eng.launch_config()
    assert all(shape[k] == best[k] for k in ("walk_block", "blocks_per_cu", "attraction_stream",
                                             "attraction_blocks_per_cu"))
    eng.close()
    return best["attraction_stream"], best["attraction_blocks_per_cu"]


def test_small_graphs_place_no_attraction():
    print("case tuned shapes", flush=True)
    for n in (5, 70, 140, 300, 600, 1100, 2100):
        before = recorded(n)
        got = tune(n)
        assert recorded(n) == (before or (0, 0)) and got == (before or (0, 0)), n
    # 4,096 nodes are one launch, 5,000 of the same bucket are not
    place = tune(5000)
    assert recorded(5000) == place
    for _ in range(3):
        tune(4096)
        assert recorded(5000) == place
    # all pairs leave what the tree's runs measured
    tune(9000)
    place = recorded(9000)
    tune(9000, use_barneshut=0)
    assert recorded(9000) == place
