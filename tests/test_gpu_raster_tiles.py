"""The tiled rasteriser at its edges: pictures of one pixel, of less and more than a tile (256 x
128) in each direction, zoomed frames whose lines end far outside, lines of no length, nodes on
tile borders, graphs without edges, more lines than one slice or one list. The picture is bytes:
equal to the CPU rasteriser's, and to the allocation-free entry point's where that takes it."""
import numpy as np
import pytest

from gpugraphlayout_amd import Engine, Raster, graphs
from gpugraphlayout_amd.host import HostGraph, png_frame, render_gray

pytestmark = pytest.mark.gpu


def scene(n, m, seed):
    s, t = graphs.barabasi_albert(n, m, seed)
    hg = HostGraph.from_edges(s, t)
    g = hg.arrays()
    rng = np.random.default_rng(seed)
    pos = (rng.normal(size=(g.n, 2)) * 300).astype(np.float32)
    pos[:: 7] = np.round(pos[:: 7])           # on pixel grids
    pos[3] = pos[4] = pos[5]                  # lines of no length
    return hg, g, pos


@pytest.mark.parametrize("w,h", [(1, 1), (255, 127), (256, 128), (257, 129), (700, 33), (31, 500)])
@pytest.mark.parametrize("n", [40, 6000])
def test_fitted_pictures(n, w, h):
    print(f"case raster tiles n={n} {w}x{h}", flush=True)
    hg, g, pos = scene(n, 3, 5)
    eng = Engine(g.n, g.src, g.dst)
    eng.set_positions(pos)
    f = png_frame(eng.bbox(), w, h, g.n, g.m)
    got = eng.render(f)
    np.testing.assert_array_equal(got, render_gray(hg, pos, f))
    np.testing.assert_array_equal(got, eng.render_noalloc(f))
    eng.close()


@pytest.mark.parametrize("zoom", [0.01, 3.0, 900.0, 30000.0])
def test_zoomed_frames(zoom):
    """Most ends outside; at the largest zoom the coordinates pass 2^22 pixels."""
    print(f"case raster zoom {zoom}", flush=True)
    hg, g, pos = scene(12, 2, 6)
    eng = Engine(g.n, g.src, g.dst)
    eng.set_positions(pos)
    f = Raster(float(pos[9, 0]) - 150 / zoom, float(pos[9, 1]) - 90 / zoom, zoom, zoom, 0.3, 0.2, 300, 180)
    np.testing.assert_array_equal(eng.render(f), render_gray(hg, pos, f))
    eng.close()


def test_no_edges_and_several_lists():
    print("case raster lists", flush=True)
    eng = Engine(5, np.zeros(0, np.int32), np.zeros(0, np.int32))
    pos = np.array([[0, 0], [10, 0], [10, 10], [3, 4], [-5, 2]], np.float32)
    eng.set_positions(pos)
    f = png_frame(eng.bbox(), 90, 60, 5, 0)
    np.testing.assert_array_equal(eng.render(f), eng.render_noalloc(f))
    eng.close()
    # 2.6M edges: 5.2M CSR entries, more than one list of 4M
    n, m = 20_000, 2_600_000
    rng = np.random.default_rng(1)
    key = np.unique(rng.integers(0, n * n, 2 * m))
    a, b = key // n, key % n
    keep = a < b
    a, b = a[keep].astype(np.int32), b[keep].astype(np.int32)
    assert 2 * len(a) > 4 << 20
    eng = Engine(n, a, b)
    eng.set_positions(graphs.uniform_positions(n, 50.0, 2))
    f = png_frame(eng.bbox(), 64, 48, n, len(a))
    f.node_alpha, f.edge_alpha = 1e-4, 1e-6     # neither the nodes nor the lines saturate
    got = eng.render(f)
    np.testing.assert_array_equal(got, eng.render_noalloc(f))
    assert 0 < got.min() < got.max() < 255
    eng.close()
