"""The validator's pass layout at the sizes where it changes: around a wave's
and a wave group's queries, a candidate chunk and the switch from one to four
queries per lane. Exact integers against the CPU oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _points(n, dim, seed):
    rng = np.random.default_rng(seed)
    c = rng.uniform(0, 5, (7, dim))
    p = c[rng.integers(0, 7, n)] + rng.normal(0, 0.3, (n, dim))
    p[rng.random(n) < 0.3] = rng.uniform(0, 5, dim)  # repeated points
    out = rng.random(n) < 0.2
    p[out] = rng.uniform(-20, 20, (int(out.sum()), dim))
    return p.astype(np.float32)


@pytest.mark.parametrize("dim", [1, 2, 3])
@pytest.mark.parametrize("n", [2, 31, 33, 64, 65, 127, 129, 255, 257, 1025, 8192, 8193, 9001])
def test_validator_sizes(engine, oracle, n, dim):
    pts = _points(n, dim, 100 * n + dim)
    eps, mp = (0.004, 3) if dim == 1 else (0.15, 4)
    label, cid, nn = engine.bruteforce(pts, eps, mp)
    ol, oc = oracle.grid(pts, eps, mp)
    assert np.array_equal(nn, oracle.neighbor_counts(pts, eps))
    assert np.array_equal(label, ol)
    assert np.array_equal(cid, oc)
