"""An allocation that finds no device memory is reported by the call that asked for it and by no
later one."""
import ctypes

import numpy as np
import pytest

from gpugraphlayout_amd import Engine, GFA2Error, Mpnn, lib

pytestmark = pytest.mark.gpu


def free_memory():
    free, total = ctypes.c_size_t(0), ctypes.c_size_t(0)
    assert lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0     # of the runtime the library runs on
    return free.value


def test_engine_out_of_memory_is_reported_once():
    print("case engine out of memory", flush=True)
    # all but 4 GB held by a network handle's scratch (1,616 bytes a node) and graph (136)
    n = int((free_memory() - 4e9) // 1752)
    m = Mpnn(seed=1)
    m.add_graph(n, np.zeros(n + 1, np.int64), np.zeros(0, np.int32), feature_seed=1, steps=0)
    big = np.arange(20_000_000, dtype=np.int32)
    with pytest.raises(GFA2Error) as ei:
        Engine(len(big), big[:-1], big[1:])          # needs over 5 GB
    assert ei.value.code == -2
    pos = np.array([[0, 0], [3, 4], [5, 1]], np.float32)
    eng = Engine(3, np.array([0, 1], np.int32), np.array([1, 2], np.int32))
    eng.set_positions(pos)
    eng.step(1)
    eng.sync()
    assert np.isfinite(eng.positions()).all() and eng.bbox().shape == (4,)
    eng.close()
    m.close()
