"""The network's matrix-instruction kernels at the edges of their tiles (16 nodes per wave, runs of
64 nodes per gradient partial) and past one round of their grids (16,384, 65,536 and 131,072
nodes), and the aggregation at the borders of its row classes: features, loss, gradient and placed
positions against the FP64 oracle."""
import numpy as np
import pytest

from gpugraphlayout_amd import Mpnn
from oracle import mpnn_oracle as mo

pytestmark = pytest.mark.gpu


def sparse_csr(n, seed):
    """About 1.5 random edges per node, some nodes with none."""
    rng = np.random.default_rng(seed)
    a, b = rng.integers(0, n, (2, 3 * n // 2 + 1))
    key = np.unique(np.concatenate([a[a != b] * n + b[a != b], b[a != b] * n + a[a != b]]))
    rowptr = np.zeros(n + 1, np.int64)
    rowptr[1:] = np.cumsum(np.bincount(key // n, minlength=n))
    return rowptr, (key % n).astype(np.int32)


@pytest.mark.parametrize("n", [3, 15, 16, 17, 63, 64, 65, 1000, 16_385, 65_600, 131_090])
def test_gradient_and_positions(n):
    print(f"case mpnn sizes n={n}", flush=True)
    rowptr, col = sparse_csr(n, n)
    rng = np.random.default_rng(n + 1)
    T = rng.normal(size=(n, 2)).astype(np.float32)
    m = Mpnn(seed=3)
    gid = m.add_graph(n, rowptr, col, target=T, feature_seed=n, steps=1)
    X = m.features(gid)
    offsets = sorted({1, n // 2, n - 1} - {0})
    loss, grad = m.loss_grad(gid, offsets)
    t = T.astype(np.float64) - T.mean(0, dtype=np.float64)
    t /= np.sqrt((t ** 2).sum(1).mean())
    p = m.params().astype(np.float64)
    L, G = mo.loss_grad(p, rowptr, col, X, t, offsets, round_bf16=True)
    # the bars of the other gradient tests (float32 products against the FP64 network)
    assert loss == pytest.approx(L, rel=1e-5)
    assert np.linalg.norm(grad - G) < 1e-4 * np.linalg.norm(G)
    Y, _ = mo.forward(p, rowptr, col, X)
    Y -= Y.mean(0)
    want = Y * (25.0 / np.sqrt((Y ** 2).sum(1).mean()))
    got = m.infer(gid, 25.0)
    assert np.linalg.norm(got - want) < 1e-4 * np.linalg.norm(want)
    m.close()


def rows_csr(degrees):
    """Rows of the given lengths over leaves of at most a few entries, numbered in random order."""
    leaves = max(degrees) + 3
    n = len(degrees) + leaves
    new = np.random.default_rng(n).permutation(n)
    a = np.repeat(np.arange(len(degrees)), degrees)
    b = len(degrees) + np.concatenate([(np.arange(d) * 7 + 11 * k) % leaves for k, d in enumerate(degrees)])
    a, b = new[a], new[b]
    key = np.unique(np.concatenate([a * n + b, b * n + a]))
    rowptr = np.zeros(n + 1, np.int64)
    rowptr[1:] = np.cumsum(np.bincount(key // n, minlength=n))
    return rowptr, (key % n).astype(np.int32)


@pytest.mark.parametrize("degrees", [(1, 3, 4, 5, 31, 32, 33, 64, 65, 127, 128, 129), (512, 513, 1023, 1024, 2047, 2048),
                                     (2049, 3072, 3073, 4096, 4097, 5121, 9000), (8191, 8192, 8193, 70_000)])
def test_row_lengths(degrees):
    """Rows at the borders of the aggregation's classes (32, 2,048), of its batches and of its
    chunks and their quarters (4,096, 1,024)."""
    print(f"case mpnn rows {degrees}", flush=True)
    rowptr, col = rows_csr(degrees)
    n = len(rowptr) - 1
    T = np.random.default_rng(n).normal(size=(n, 2)).astype(np.float32)
    m = Mpnn(seed=3)
    gid = m.add_graph(n, rowptr, col, target=T, feature_seed=n, steps=2)
    X = m.features(gid)
    assert np.max(np.abs(X - mo.features(rowptr, col, n, 2))) < 1e-4      # the bar of the other feature tests
    loss, grad = m.loss_grad(gid, [1, 7])
    t = T.astype(np.float64) - T.mean(0, dtype=np.float64)
    t /= np.sqrt((t ** 2).sum(1).mean())
    L, G = mo.loss_grad(m.params().astype(np.float64), rowptr, col, X, t, [1, 7], round_bf16=True)
    assert loss == pytest.approx(L, rel=1e-5)
    assert np.linalg.norm(grad - G) < 1e-4 * np.linalg.norm(G)
    m.close()


@pytest.mark.parametrize("n", [2, 3, 127, 128, 129, 57_344, 57_345, 115_000])
def test_feature_columns(n):
    """One to all blocks of the columns' sums (128 rows each, 448 blocks), and past one round."""
    print(f"case mpnn feature columns n={n}", flush=True)
    rowptr, col = sparse_csr(n, n)
    m = Mpnn(seed=3)
    X = m.features(m.add_graph(n, rowptr, col, feature_seed=n, steps=1))
    assert np.max(np.abs(X - mo.features(rowptr, col, n, 1))) < 1e-4      # the bar of the other feature tests
    m.close()
