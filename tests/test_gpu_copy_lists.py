"""Host-buffer slides whose pinned buffers do not abut: the copies of a slide
run as one launch over a list. Every result equals the plain path's, for
buffers apart by gaps, of one point up to several blocks of words."""
import numpy as np
import pytest

from rtdbstream_amd import workloads as WL

pytestmark = pytest.mark.gpu

SPECS = [(1, 3, 1), (2, 64, 64), (3, 341, 11), (2, 4096, 1024), (3, 9000, 1500), (1, 2047, 89), (2, 2, 1)]


def _data(dim, n, seed):
    if dim == 1:
        return np.random.default_rng(seed).normal(0, 3, (n, 1)).astype(np.float32)
    return WL.blobs2d(n, seed=seed) if dim == 2 else WL.walks3d(n, seed=seed, n_walks=40, box=(20.0, 20.0, 5.0))


@pytest.mark.parametrize("pipelined", [False, True])
@pytest.mark.parametrize("use_graph", [False, True])
def test_scattered_pinned_buffers(engine, pipelined, use_graph):
    R, slides = engine, 5
    datas = [_data(d, W + slides * S, 30 + i) for i, (d, W, S) in enumerate(SPECS)]
    plain = []
    for x, (d, W, S) in zip(datas, SPECS):
        s = R.Stream(d, W, S, 0.5, 4)
        s.init(x[:W])
        plain.append([s.slide(x[W + t * S: W + (t + 1) * S]) for t in range(slides)])
        s.close()
    buf = R.HostBuffer(1 << 20)
    at = [0]

    def view(dtype, n):
        v = buf.array(dtype, n, offset=at[0])
        at[0] += 4 * n + 4 * (1 + n % 5)  # a gap, of no multiple of 16 bytes
        return v

    streams, ins, labels, cids = [], [], [], []
    for x, (d, W, S) in zip(datas, SPECS):
        s = R.Stream(d, W, S, 0.5, 4)
        s.init(x[:W])
        streams.append(s)
        row = []
        for t in range(slides):
            v = view(np.float32, S * d)
            v[:] = x[W + t * S: W + (t + 1) * S].reshape(-1)
            row.append(v)
        ins.append(row)
        labels.append([view(np.int32, W) for _ in range(2)])
        cids.append([view(np.int32, W) for _ in range(2)])
    b = R.Batch(streams, use_graph=use_graph)

    def check(t):
        for i in range(len(SPECS)):
            assert np.array_equal(labels[i][t & 1], plain[i][t][0]), (i, t)
            assert np.array_equal(cids[i][t & 1], plain[i][t][1]), (i, t)

    for t in range(slides):
        args = [r[t] for r in ins], [v[t & 1] for v in labels], [v[t & 1] for v in cids]
        if pipelined:
            b.slide_pipelined(*args)
            if t:
                check(t - 1)
        else:
            b.slide(*args)
            check(t)
    if pipelined:
        b.drain()
        check(slides - 1)
    b.close()
    for s in streams:
        s.close()
    buf.free()
