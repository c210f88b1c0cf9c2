"""The sort's pass of one launch at the edges of its tiles (2,048 and 4,096 pairs), of its rounds
over earlier tiles (8 and 16 of them), of its two tile sizes (32,768 pairs) and of its range
(262,144), on full sorts and on ones that skip low passes, one key digit shared by almost all
bodies among them: body orders equal a numpy sort of the restated keys. The same of batches, at the
edges of the per-graph sort's forms (2,048, 4,096, 8,192 and 32,768 bodies) and past them."""
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


@pytest.mark.parametrize("sizes", [
    [40_000, 1, 300, 7000],                                               # over the per-graph sort's limit
    [1, 2, 2047, 2048, 500, 64, 65],                                      # a block of 256 threads each
    [4096, 2049, 1, 4095, 100],                                           # of 512
    [8192, 4097, 2048, 2049, 1, 700, 511, 64, 300],                       # of 1,024, or a quarter of one
    [32_768, 8193, 16_384, 16_385, 2048, 2, 100, 30],                     # and tile by tile
])
def test_batches(sizes):
    print(f"case sort pass batch {sizes}", flush=True)
    chain = [(n, np.arange(n - 1, dtype=np.int32), np.arange(1, n, dtype=np.int32)) for n in sizes]
    eng = BatchEngine(chain, scale=1.0, gravity=1.0)
    eng.set_positions(np.concatenate([positions(n, 0) for n in sizes]))
    off = np.concatenate([[0], np.cumsum(sizes)])
    for it in range(5):
        p = eng.positions()
        eng.step(1)
        eng.sync()
        perm = eng.tree()["perm"]
        for a, b in zip(off, off[1:]):
            np.testing.assert_array_equal(perm[a:b] - a, expected_order(p[a:b])[0], err_msg=f"iteration {it}")
    eng.close()
