"""Additions of data far from uniform -- one far point, a heavy tail, many equal
points, points on a line, non-finite coordinates: the results of the CPU oracle,
and no multiple of the time that uniform points take to add (a cut of the extents
into equal cells put nearly all points into one bucket: 50 to 130 times)."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
N = 300_000


def data(kind, metric, dim):
    rng = np.random.default_rng(17)
    x = rng.uniform(-3, 3, (N, dim)).astype(np.float32)
    t = dim
    if metric == 1:
        t, q = 3, rng.normal(size=(N, 4))
        x[:, 3:] = q / np.linalg.norm(q, axis=1, keepdims=True)
    if kind == "far point":
        x[N // 2, :t] = 1e6
    elif kind == "heavy tail":
        x[:, :t] = rng.standard_cauchy((N, t))
    elif kind == "half equal":
        x[:N // 2] = x[0]
    elif kind == "all equal":
        x[:] = x[0]
    elif kind == "nearly constant":  # in one coordinate
        x[:, 0] = 0.0
        x[::50, 0] = np.linspace(-1e6, 1e6, N // 50)
    elif kind == "nearly equal":
        x[::50] += 1.0
        x[np.arange(N) % 50 > 0] = x[1]
    elif kind == "line":
        x[:, :t] = x[:, :1] + np.linspace(0, 1, t)
    elif kind == "not finite":
        x[rng.choice(N, N // 20, replace=False), rng.integers(0, t, N // 20)] = np.nan
    return x


def add_us(nn, pts):
    import torch

    us = []
    for _ in range(7):
        nn.clear()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        nn.add(pts)
        us.append(1e6 * (time.perf_counter() - t0))
    return sorted(us)[3]


@pytest.mark.parametrize("kind", ["far point", "heavy tail", "half equal", "all equal", "line", "not finite",
                                  "nearly constant", "nearly equal"])
@pytest.mark.parametrize("metric,dim", [(0, 1), (0, 3), (0, 7), (1, 7)])
def test_skewed_points(gpu, oracle, kind, metric, dim):
    import torch
    from ompl_amd.nn import NearestNeighborsGPU

    x = data(kind, metric, dim)
    nn = NearestNeighborsGPU(metric, dim)
    even, skewed = (add_us(nn, torch.from_numpy(p).cuda()) for p in (data("", metric, dim), x))
    q = x[:: N // 12][:12].copy()
    q[np.isnan(q)] = 0.0
    ids = np.flatnonzero(~np.isnan(x).any(axis=1))  # a point that is not finite is in no result
    gi, gd = nn.knn_batch(q, 10)
    oi, od = oracle.knn(metric, x[ids], q, 10)
    assert np.array_equal(gi, ids[oi]) and np.array_equal(gd, od)
    print(f"{kind} {metric} {dim}: {skewed:.0f} us against {even:.0f}", flush=True)
    assert skewed < 10 * even
