"""An allocation that finds no device memory is reported by the call that asked for it and by no
later one."""
import numpy as np
import pytest

from gpugraphlayout_amd import Engine, GFA2Error, Mpnn

pytestmark = pytest.mark.gpu


def test_engine_out_of_memory_is_reported_once():
    import torch
    print("case engine out of memory", flush=True)
    # all but 4 GB held by a network handle's scratch (1,616 bytes a node) and graph (136)
    n = int((torch.cuda.mem_get_info()[0] - 4e9) // 1752)
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
