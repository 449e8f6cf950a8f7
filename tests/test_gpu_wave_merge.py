"""The merge by a wave per cell of streams with safe cells, which small single
streams take by size and every stream here is forced into (or out of): few and
many candidates, border cells whose cores are elements of their own, and the
sizes where the choice changes, against the CPU oracle."""
import numpy as np
import pytest

from test_gpu_merge_cells import _check, _clumps

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wave", ["0", "1"])
@pytest.mark.parametrize("mode", ["1", "2"])
@pytest.mark.parametrize("dim,k", [(1, 2), (2, 2), (2, 3), (3, 2), (3, 3), (3, 1)])
@pytest.mark.parametrize("clumps,sigma", [(25, 0.4), (3, 0.25)])  # the second: cells past 192 candidates
def test_forms(engine, oracle, monkeypatch, wave, mode, dim, k, clumps, sigma):
    monkeypatch.setenv("RTDBS_WAVE_MERGE", wave)
    monkeypatch.setenv("RTDBS_NEIGHBOR_MODE", mode)
    W, S, slides = 2000, 500, 3
    data = _clumps(W + slides * S, dim, 10 * dim + k, clumps, sigma, {1: 60, 2: 16, 3: 9}[dim])
    eps = {1: 0.05, 2: 0.4, 3: 0.7}[dim]
    _check(engine, oracle, data, dim, W, S, eps, 5, slides, "dim %d k %d" % (dim, k), cell_div=k)


@pytest.mark.parametrize("wave", ["0", "1"])
@pytest.mark.parametrize("dim", [1, 2, 3])
def test_border_cells(engine, oracle, monkeypatch, wave, dim):
    monkeypatch.setenv("RTDBS_WAVE_MERGE", wave)
    W, S, slides = 1500, 300, 3
    data = _clumps(W + slides * S, dim, 70 + dim, 12, 0.5, 8)
    _check(engine, oracle, data, dim, W, S, {1: 0.03, 2: 0.3, 3: 0.6}[dim], 4, slides, "dim %d" % dim,
           lo=[2.0] * dim, hi=[6.0] * dim)


@pytest.mark.parametrize("wave", ["0", "1"])
@pytest.mark.parametrize("n", [1, 4, 64, 65, 192, 193, 600])
@pytest.mark.parametrize("apart", [0.99, 1.01])
def test_pairs_near_eps(engine, oracle, monkeypatch, wave, n, apart):
    monkeypatch.setenv("RTDBS_WAVE_MERGE", wave)
    rng = np.random.default_rng(n)
    W = 2 * n + 40
    a = rng.uniform(0, 0.05, (n, 3))
    b = rng.uniform(0, 0.05, (n, 3)) + np.array([apart + 0.02, 0.03, 0.0])
    pts = np.concatenate([a, b, rng.uniform(6, 30, (40, 3))])[rng.permutation(W)].astype(np.float32)
    _check(engine, oracle, np.concatenate([pts, pts]), 3, W, W // 2, 1.0, max(1, n // 2), 2, "n %d" % n)


@pytest.mark.parametrize("dim,W,k", [(2, 2048, 2), (2, 2050, 2), (3, 90000, 2), (3, 90002, 3)])
def test_choice_by_size(engine, oracle, dim, W, k):
    S = W // 2
    data = _clumps(W + S, dim, W, W // 40, 0.4, 3.0 * W ** (1.0 / dim) / 2)
    _check(engine, oracle, data, dim, W, S, 0.5, 5, 1, "W %d" % W, cell_div=k)
