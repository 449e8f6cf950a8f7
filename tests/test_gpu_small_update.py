"""The one-block window update at the edges of its sizes (64, 256 and 1024
stride keys, 1024-position rounds, the largest window and stride it takes, and
the first sizes past them): labels and ids against the CPU oracle (integers),
and the window it leaves behind."""
import numpy as np
import pytest

from tests.refcheck import window_at

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (2, 1), (3, 3), (64, 64), (65, 65), (130, 65), (256, 256), (257, 257), (514, 257), (1000, 10),
         (1023, 341), (1024, 1024), (1025, 205), (2048, 1024), (2050, 1025), (3072, 1024), (4095, 1365), (4095, 819),
         (4096, 512), (4096, 1024), (4097, 241), (7168, 1024), (8191, 1), (8192, 1024), (8192, 8), (8193, 2731),
         (9216, 1024)]


def _data(dim, W, S, slides):
    rng = np.random.default_rng(W * 7 + S + dim)
    n = W + slides * S
    d = rng.normal(0, {1: W / 40.0, 2: W ** 0.5 / 4, 3: W ** (1 / 3.0)}[dim], (n, dim)).astype(np.float32)
    d[::3] *= np.float32(0.01)  # a third of the points in few cells
    d[n // 2:n // 2 + n // 8] = d[:n // 8]
    if W > 100:
        d[rng.integers(0, n, 5), 0] = np.nan
        d[rng.integers(0, n, 5), dim - 1] = 1e30  # clamped into a border cell
    return d


@pytest.mark.parametrize("W,S", SIZES)
@pytest.mark.parametrize("dim", [1, 2, 3])
def test_sizes(engine, oracle, dim, W, S):
    slides = min(W // S + 2, 5)
    d = _data(dim, W, S, slides)
    eps, mp = 0.25, 4
    rl, rc = oracle.stream(d, W, S, eps, mp, slides, method="bruteforce")
    s = engine.Stream(dim, W, S, eps, mp, lo=[-50.0] * dim, hi=[50.0] * dim)
    s.init(d[:W])
    for t in range(slides):
        l, c = s.slide(d[W + t * S: W + (t + 1) * S])
        assert np.array_equal(l, rl[t]) and np.array_equal(c, rc[t]), t
    assert np.array_equal(s.window().reshape(W, dim).view(np.uint32), window_at(d, W, S, slides - 1).view(np.uint32))
    s.close()


@pytest.mark.parametrize("sizes", [[(1000, 10), (4096, 1024), (512, 512)], [(1000, 10), (4097, 241), (512, 512)]])
@pytest.mark.parametrize("graph", [False, True])
def test_batches(engine, oracle, sizes, graph):
    """All members small, and a member past the limit among small ones."""
    slides, eps, mp = 4, 0.25, 4
    data = [_data(2, W, S, slides) for W, S in sizes]
    ref = [oracle.stream(d, W, S, eps, mp, slides, method="bruteforce") for d, (W, S) in zip(data, sizes)]
    st = [engine.Stream(2, W, S, eps, mp, lo=[-50.0] * 2, hi=[50.0] * 2) for W, S in sizes]
    for s, d in zip(st, data):
        s.init(d[:s.W])
    b = engine.Batch(st, use_graph=graph)
    for t in range(slides):
        out = b.slide([d[W + t * S: W + (t + 1) * S] for d, (W, S) in zip(data, sizes)])
        for i, (l, c) in enumerate(zip(*out)):
            assert np.array_equal(l, ref[i][0][t]) and np.array_equal(c, ref[i][1][t]), (i, t)
    b.close()
    for s in st:
        s.close()


# host slides of a small stream read and write pinned memory from the kernels:
# the caller's buffers where they are pinned, else the engine's staging
@pytest.mark.parametrize("pinned", [(0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 1)])
@pytest.mark.parametrize("shift", [0, 2])  # bytes off a word
def test_host_buffers(engine, oracle, pinned, shift):
    W, S, slides, eps, mp = 1500, 300, 6, 0.25, 4
    d = _data(2, W, S, slides)
    rl, rc = oracle.stream(d, W, S, eps, mp, slides, method="bruteforce")
    s = engine.Stream(2, W, S, eps, mp, lo=[-50.0] * 2, hi=[50.0] * 2)
    s.init(d[:W])
    hb = engine.HostBuffer(S * 8 + W * 8 + shift)
    x = hb.array(np.float32, S * 2, offset=shift) if pinned[0] else np.empty(S * 2, np.float32)
    l = hb.array(np.int32, W, offset=S * 8 + shift) if pinned[1] else np.empty(W, np.int32)
    c = hb.array(np.int32, W, offset=S * 8 + W * 4 + shift) if pinned[2] else np.empty(W, np.int32)
    for t in range(slides):
        x[:] = d[W + t * S: W + (t + 1) * S].reshape(-1)
        l[:] = -7
        c[:] = -7
        s.slide(x, l, c)
        assert np.array_equal(l, rl[t]) and np.array_equal(c, rc[t]), t
    s.close()
