"""The sort's pass of one launch at the edges of its tiles (2,048 and 4,096 pairs), of its rounds
over earlier tiles (8 and 16 of them), of its two tile sizes (32,768 pairs) and of its range
(262,144), on full sorts and on ones that skip low passes, one key digit shared by almost all
bodies among them: body orders equal a numpy sort of the restated keys; and in a batch with a graph
over the per-graph sort's limit."""
import numpy as np
import pytest

from gpugraphlayout_amd import BatchEngine, Engine
from test_gpu_parity import expected_order

pytestmark = pytest.mark.gpu


def positions(n, clumped):
    rng = np.random.default_rng(n)
    p = rng.uniform(-1000, 1000, size=(n, 2))
    p[: n // 10] *= 1e-3
    if clumped:                  # nearly all top digits alike
        p[2:] = p[2:] * 2.0 ** -9 + 300
    return p.astype(np.float32)


@pytest.mark.parametrize("n,clumped", [(4097, 0), (16_384, 0), (16_385, 1), (18_433, 0), (32_768, 1), (32_769, 0),
                                       (36_865, 1), (69_633, 0), (262_144, 1), (262_145, 0)])
def test_orders(n, clumped):
    print(f"case sort pass n={n} clumped={clumped}", flush=True)
    src = np.arange(0, n - 1, 2)
    eng = Engine(n, src, src + 1, scale=1.0, gravity=1.0)
    eng.set_positions(positions(n, clumped))
    for it in range(5):          # full sorts, then by the previous tree's depth
        p = eng.positions()
        eng.step(1)
        eng.sync()
        np.testing.assert_array_equal(eng.tree()["perm"], expected_order(p)[0], err_msg=f"iteration {it}")
    eng.close()


def test_batch_over_the_per_graph_limit():
    print("case sort pass batch", flush=True)
    sizes = [40_000, 1, 300, 7000]
    chain = [(n, np.arange(n - 1, dtype=np.int32), np.arange(1, n, dtype=np.int32)) for n in sizes]
    eng = BatchEngine(chain, scale=1.0, gravity=1.0)
    eng.set_positions(np.concatenate([positions(n, 0) for n in sizes]))
    off = np.concatenate([[0], np.cumsum(sizes)])
    for it in range(3):
        p = eng.positions()
        eng.step(1)
        eng.sync()
        perm = eng.tree()["perm"]
        for a, b in zip(off, off[1:]):
            np.testing.assert_array_equal(perm[a:b] - a, expected_order(p[a:b])[0], err_msg=f"iteration {it}")
    eng.close()
