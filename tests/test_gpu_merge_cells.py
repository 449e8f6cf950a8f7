"""The merge of safe cells by links and joins, at the edges of its tiles and of
the sizes that pick a pair's lanes: bit-exact labels and ids against the CPU
oracle (integers)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _clumps(n, dim, seed, clumps, sigma, box, noise=0.2):
    rng = np.random.default_rng(seed)
    c = rng.uniform(0, box, (clumps, dim))
    p = c[rng.integers(0, clumps, n)] + rng.normal(0, sigma, (n, dim))
    m = rng.random(n) < noise
    p[m] = rng.uniform(0, box, (int(m.sum()), dim))
    return p.astype(np.float32)


def _check(engine, oracle, data, dim, W, S, eps, mp, slides, what, **kw):
    rl, rc = oracle.stream(data, W, S, eps, mp, slides, method="grid")
    s = engine.Stream(dim, W, S, eps, mp, **kw)
    s.init(data[:W])
    for t in range(slides):
        l, c = s.slide(data[W + t * S: W + (t + 1) * S])
        assert np.array_equal(l, rl[t]), "%s slide %d labels" % (what, t)
        assert np.array_equal(c, rc[t]), "%s slide %d ids" % (what, t)
    s.close()


@pytest.mark.parametrize("mode", ["1", "2"])
@pytest.mark.parametrize("tile", ["1", "7", "8", "32", "64"])
@pytest.mark.parametrize("dim,k", [(1, 2), (1, 3), (2, 2), (2, 3), (3, 2), (3, 3)])
def test_tiles(engine, oracle, monkeypatch, dim, k, tile, mode):
    monkeypatch.setenv("RTDBS_CELL_TILE", tile)
    monkeypatch.setenv("RTDBS_NEIGHBOR_MODE", mode)
    W, S, slides = 2000, 500, 3
    data = _clumps(W + slides * S, dim, 10 * dim + k, 25, 0.4, {1: 60, 2: 16, 3: 9}[dim])
    eps = {1: 0.05, 2: 0.4, 3: 0.7}[dim]
    _check(engine, oracle, data, dim, W, S, eps, 5, slides, "dim %d k %d" % (dim, k), cell_div=k)


# two clumps a little more or a little less than eps apart, of sizes around what
# a lane (4 points), 8 lanes (32), 16 lanes (64) and a wave (256) hold
@pytest.mark.parametrize("n", [1, 4, 5, 32, 33, 64, 65, 256, 257, 600])
@pytest.mark.parametrize("apart", [0.99, 1.01])
def test_pairs_near_eps(engine, oracle, n, apart):
    rng = np.random.default_rng(n)
    eps, W = 1.0, 2 * n + 40
    a = rng.uniform(0, 0.05, (n, 3))
    b = rng.uniform(0, 0.05, (n, 3)) + np.array([apart + 0.02, 0.03, 0.0])
    pts = np.concatenate([a, b, rng.uniform(6, 30, (40, 3))])[rng.permutation(W)].astype(np.float32)
    _check(engine, oracle, np.concatenate([pts, pts]), 3, W, W // 2, eps, max(1, n // 2), 2, "n %d" % n)


# grid bounds inside the data: border cells hold clamped points, every core of
# theirs is an element of its own
@pytest.mark.parametrize("mode", ["1", "2"])
@pytest.mark.parametrize("dim", [1, 2, 3])
def test_unsafe_cells(engine, oracle, monkeypatch, dim, mode):
    monkeypatch.setenv("RTDBS_NEIGHBOR_MODE", mode)
    W, S, slides = 1500, 300, 3
    data = _clumps(W + slides * S, dim, 70 + dim, 12, 0.5, 8)
    _check(engine, oracle, data, dim, W, S, {1: 0.03, 2: 0.3, 3: 0.6}[dim], 4, slides, "dim %d" % dim,
           lo=[2.0] * dim, hi=[6.0] * dim)


def test_batch_of_safe_and_unsafe_streams(engine, oracle):
    # reach 1 has no safe cell: its merge kernel runs beside the links and joins
    W, S, slides = 1200, 300, 3
    specs = [(2, 1, 0.4), (2, 2, 0.4), (3, 3, 0.7), (3, 1, 0.7), (1, 2, 0.05)]
    datas = [_clumps(W + slides * S, d, 90 + i, 20, 0.4, {1: 60, 2: 16, 3: 9}[d]) for i, (d, _, _) in enumerate(specs)]
    refs = [oracle.stream(x, W, S, e, 5, slides, method="grid") for x, (_, _, e) in zip(datas, specs)]
    streams = []
    for x, (d, k, e) in zip(datas, specs):
        s = engine.Stream(d, W, S, e, 5, cell_div=k)
        s.init(x[:W])
        streams.append(s)
    b = engine.Batch(streams)
    for t in range(slides):
        ls, cs = b.slide([x[W + t * S: W + (t + 1) * S] for x in datas])
        for i, (rl, rc) in enumerate(refs):
            assert np.array_equal(ls[i], rl[t]) and np.array_equal(cs[i], rc[t]), (i, t)
    b.close()
    for s in streams:
        s.close()
