"""The stride's rank against the oracle where its chunks of 64 keys and runs of
512 end, and where one run's keys span the others'."""
import numpy as np
import pytest

from test_gpu_parity import assert_parity, engine_slides

pytestmark = pytest.mark.gpu


def _points(kind, n, S, dim, seed):
    rng = np.random.default_rng(seed)
    x = rng.normal(0.0, 1.0, (n, dim))
    at = np.arange(n) % S
    if kind == "rising":  # the runs hold disjoint key ranges
        x[:, 0] = at * (8.0 / S) + rng.normal(0.0, 0.01, n)
    elif kind == "spanning":  # the first run's keys lie on either side of all others
        first = at < 512
        x[first, 0] = np.where(rng.random(first.sum()) < 0.5, -20.0, 20.0)
    elif kind == "repeated":  # whole runs in one cell: ranks by slot alone
        x = np.round(x)
    return x.astype(np.float32)


@pytest.mark.parametrize("split", ["0", "1"])
@pytest.mark.parametrize("kind", ["mixed", "rising", "spanning", "repeated"])
@pytest.mark.parametrize("S,dim", [(1, 2), (63, 2), (64, 3), (65, 1), (511, 3), (513, 2), (577, 1), (1025, 3),
                                   (8191, 2), (17000, 3)])
def test_stride_rank_sizes(engine, oracle, monkeypatch, split, kind, S, dim):
    monkeypatch.setenv("RTDBS_RANK_SPLIT", split)
    monkeypatch.setenv("RTDBS_SMALL_UPDATE", "0")  # small strides too go through the rank kernel
    W, slides = 3 * S, 3
    eps = 4.0 / max(2.0, W ** (1.0 / dim))
    data = _points(kind, W + slides * S, S, dim, 17 * S + dim)
    ref_l, ref_c = oracle.stream(data, W, S, eps, 4, slides, method="grid")
    got = engine_slides(engine, data, dim, W, S, eps, 4, slides)
    assert_parity(got, ref_l, ref_c, "split %s %s S%d dim%d" % (split, kind, S, dim))
