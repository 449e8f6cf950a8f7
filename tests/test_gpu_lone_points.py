"""Points whose count finds no neighbour are noise without a look at their
stencil: isolated points, pairs below min_pts, border points whose only
neighbour is a core, coordinates that are not numbers, and an eps whose square
is zero, in every form of the count and of the outputs, against the CPU oracle;
the work counters, which cover every point's stencil, change nothing."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _data(dim, n, seed):
    rng = np.random.default_rng(seed)
    d = rng.uniform(-60.0, 60.0, (n, dim)).astype(np.float32)  # mostly alone
    kind = rng.integers(0, 8, n)
    at = np.zeros((n, dim), np.float32)
    at[:, 0] = 80.0 + 4.0 * rng.integers(0, 6, n)
    d[kind == 0] = at[kind == 0] + rng.normal(0, 0.05, ((kind == 0).sum(), dim))  # cores
    ring = kind == 1  # one neighbour or few: at the edge of a cluster's reach
    d[ring] = at[ring]
    d[ring, 0] += rng.uniform(0.85, 1.15, ring.sum()).astype(np.float32)
    pair = np.flatnonzero(kind == 2)[: 2 * ((kind == 2).sum() // 2)]
    d[pair[1::2]] = d[pair[::2]]  # two points, no core
    odd = np.flatnonzero(kind == 3)[:6]
    for i, v in zip(odd, [np.nan, np.inf, -np.inf, 3e38, np.nan, np.inf]):
        d[i, i % dim] = v
    return d


@pytest.mark.parametrize("form", ["", "cell", "point1", "point4", "cell-regroup"])
@pytest.mark.parametrize("dim,eps,mp", [(1, 1.0, 3), (2, 1.0, 4), (3, 1.0, 4), (3, 1.0, 1), (2, 1.0, 2), (2, 1e-23, 2)])
def test_lone_points(engine, oracle, monkeypatch, form, dim, eps, mp):
    if form:
        monkeypatch.setenv("RTDBS_NEIGHBOR_MODE", "1" if form == "cell" else "2")
        if form.startswith("point"):
            monkeypatch.setenv("RTDBS_BORDER_LPQ", form[5:])
            monkeypatch.setenv("RTDBS_BORDER_REGROUP", "0")
        if form == "cell-regroup":
            monkeypatch.setenv("RTDBS_COUNT_MODE", "1")
    W, S, slides = 2600, 650, 5
    d = _data(dim, W + slides * S, 10 * dim + mp)
    lim = dict(lo=[-70.0] * dim, hi=[110.0] * dim)
    rl, rc = oracle.stream(d, W, S, eps, mp, slides, method="bruteforce")
    for stats in (False, True):
        s = engine.Stream(dim, W, S, eps, mp, **lim)
        s.init(d[:W])
        if stats:
            s.set_stats(True)
        for t in range(slides):
            l, c = s.slide(d[W + t * S: W + (t + 1) * S])
            assert np.array_equal(l, rl[t]) and np.array_equal(c, rc[t]), (t, stats)
        s.close()
