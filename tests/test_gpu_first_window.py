"""The first window's sort at the edges of its runs (2048 keys), merge tiles
(512 outputs) and pass counts: the window read back bit for bit, and labels and
ids of the slides after it against the CPU oracle (integers)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,S", [(1, 1), (2, 1), (511, 73), (512, 256), (513, 171), (2047, 89), (2048, 512), (2049, 683),
                                 (4096, 4096), (4097, 241), (6150, 1025), (8193, 2731), (16389, 5463), (40000, 4000)])
@pytest.mark.parametrize("dim", [1, 2, 3])
def test_sizes(engine, oracle, dim, W, S):
    rng = np.random.default_rng(W + dim)
    n = W + 2 * S
    # a third of the points share a cell, some coordinates twice
    data = rng.normal(0, {1: W / 40.0, 2: W ** 0.5 / 4, 3: W ** (1 / 3.0)}[dim], (n, dim)).astype(np.float32)
    data[::3] *= np.float32(0.001)
    data[n // 2:n // 2 + n // 8] = data[:n // 8]
    eps, mp = 0.25, 4
    rl, rc = oracle.stream(data, W, S, eps, mp, 2, method="grid")
    s = engine.Stream(dim, W, S, eps, mp)
    for again in range(2):  # a stream may be given a first window twice
        s.init(data[:W])
        assert np.array_equal(s.window().reshape(W, dim).view(np.uint32), data[:W].view(np.uint32)), (again, W)
        for t in range(2):
            l, c = s.slide(data[W + t * S: W + (t + 1) * S])
            assert np.array_equal(l, rl[t]) and np.array_equal(c, rc[t]), (again, t)
    s.close()


# bounds of the first window, as the grid's origin shows them: extremes in the
# first, last and every other place of the scan (32,768 points a turn), NaNs
# passed over, an axis of NaNs alone taken as zero
@pytest.mark.parametrize("W", [1, 2, 63, 257, 32768, 32769, 70001])
@pytest.mark.parametrize("dim", [1, 2, 3])
@pytest.mark.parametrize("nans", ["none", "some", "axis"])
def test_bounds(engine, dim, W, nans):
    rng = np.random.default_rng(W)
    eps = 0.5
    for place in sorted({0, W // 2, W - 1}):
        x = rng.uniform(-1, 1, (W, dim)).astype(np.float32)
        x[place] = -3.25
        x[W - 1 - place] = 7.5
        if nans == "some":
            x[rng.integers(0, W, W // 3)] = np.nan
        elif nans == "axis":
            x[:, dim - 1] = np.nan
        s = engine.Stream(dim, W, W, eps, 3)
        s.init(x)
        info = s.info()
        for a in range(dim):
            v = x[:, a][~np.isnan(x[:, a])].astype(np.float64)
            mn, mx = (v.min(), v.max()) if v.size else (0.0, 0.0)
            lo = float(np.float32(mn - 2.0 * (mx - mn) - eps))
            assert info["lo"][a] == lo, (place, a)
            assert info["grid"][a] == int((mx + 2.0 * (mx - mn) + eps - lo) * (1.0 / info["cell_side"])) + 1, (place, a)
        assert np.array_equal(s.window().reshape(W, dim).view(np.uint32), x.view(np.uint32))
        s.close()
