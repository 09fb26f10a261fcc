"""GPU parity of the nearest-neighbour structure's spatial index (kept from
2,048 points on, L2 up to 7 dimensions and SE3) with the CPU oracle's full
scan: sizes at the edges of tiles (64 points), nodes (4,096) and supernodes
(262,144), points added after a build, removals, duplicates, degenerate data,
and every number of waves a query is given."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def points(gpu, metric, dim, seed, n):
    if metric == 1:
        return gpu.workload.se3(seed, n)
    return np.random.default_rng(seed).uniform(-np.pi, np.pi, (n, dim)).astype(np.float32)


def index(metric, dim, *parts):
    from ompl_amd.nn import NearestNeighborsGPU

    nn = NearestNeighborsGPU(metric, dim)
    for p in parts:
        nn.add(p)
    return nn


def same_knn(nn, oracle, metric, data, q, k):
    gi, gd = nn.knn_batch(q, k)
    oi, od = oracle.knn(metric, data, q, k)
    assert np.array_equal(gi, oi) and np.array_equal(gd, od)


def same_radius(nn, oracle, metric, data, q, r):
    off, gi, gd = nn.radius_batch(q, r)
    for j, (oi, od) in enumerate(oracle.radius(metric, data, q, r)):
        assert np.array_equal(gi[off[j]:off[j + 1]], oi) and np.array_equal(gd[off[j]:off[j + 1]], od)


@pytest.mark.parametrize("metric,dim", [(0, d) for d in range(1, 8)] + [(1, 7)])
@pytest.mark.parametrize("n", [2047, 2048, 2049, 4096, 4097, 9999])
def test_tile_and_node_edges(gpu, oracle, metric, dim, n):
    data = points(gpu, metric, dim, 100 + n, n)
    q = points(gpu, metric, dim, 7, 33)
    nn = index(metric, dim, data)
    for k in (1, 10, 64):
        same_knn(nn, oracle, metric, data, q, k)
    r = float(np.median(oracle.knn(metric, data, q, 20)[1][:, -1]))
    same_radius(nn, oracle, metric, data, q, r)
    same_radius(nn, oracle, metric, data, q, 0.0)


@pytest.mark.parametrize("metric,dim", [(0, 2), (1, 7)])
def test_supernodes(gpu, oracle, metric, dim):
    data = points(gpu, metric, dim, 3, 262_144 * 2 + 65)
    q = points(gpu, metric, dim, 4, 40)
    nn = index(metric, dim, data)
    same_knn(nn, oracle, metric, data, q, 16)
    same_radius(nn, oracle, metric, data, q, 0.3)


@pytest.mark.parametrize("nq", [1, 128, 129, 2049, 6145])
def test_waves_per_query(gpu, oracle, nq):
    data = points(gpu, 0, 5, 11, 8000)
    q = points(gpu, 0, 5, 12, nq)
    nn = index(0, 5, data)
    gi, gd = nn.knn_batch(q, 11)
    sel = np.linspace(0, nq - 1, min(nq, 64)).astype(int)
    oi, od = oracle.knn(0, data, q[sel], 11)
    assert np.array_equal(gi[sel], oi) and np.array_equal(gd[sel], od)


def test_ordered_radius_batch(gpu, oracle):
    """A batch large enough to be searched in Morton order (results stay in the caller's)."""
    data = points(gpu, 1, 7, 21, 200_000)
    q = points(gpu, 1, 7, 22, 20_000)
    off, gi, gd = index(1, 7, data).radius_batch(q, 1.2)
    sel = np.linspace(0, len(q) - 1, 40).astype(int)
    for j, (oi, od) in zip(sel, oracle.radius(1, data, q[sel], 1.2)):
        assert np.array_equal(gi[off[j]:off[j + 1]], oi) and np.array_equal(gd[off[j]:off[j + 1]], od)


def test_tail_rebuild_removal_and_clear(gpu, oracle):
    data = points(gpu, 0, 7, 31, 6000)
    q = points(gpu, 0, 7, 32, 20)
    nn = index(0, 7, data[:4000], data[4000:4300], data[4300:4301])  # built, then a tail of 301
    same_knn(nn, oracle, 0, data[:4301], q, 10)
    nn.add(data[4301:])  # built again
    rng = np.random.default_rng(5)
    gone = rng.choice(6000, 900, replace=False)
    for i in gone:
        assert nn.remove(int(i))
    keep = np.setdiff1d(np.arange(6000), gone)

    def check(ids, pts):
        gi, gd = nn.knn_batch(q, 12)
        oi, od = oracle.knn(0, pts, q, 12)
        assert np.array_equal(gi, ids[oi]) and np.array_equal(gd, od)

    check(keep, data[keep])
    more = points(gpu, 0, 7, 33, 1000)
    nn.add(more)  # a build after removals
    check(np.concatenate([keep, 6000 + np.arange(1000)]), np.concatenate([data[keep], more]))
    nn.clear()
    nn.add(more)  # below the size an index is kept for
    same_knn(nn, oracle, 0, more, q, 12)
    nn.add(data)
    same_knn(nn, oracle, 0, np.concatenate([more, data]), q, 12)


@pytest.mark.parametrize("kind", ["same", "line", "copies", "far", "skewed"])
def test_degenerate_data(gpu, oracle, kind):
    rng = np.random.default_rng(41)
    data = rng.uniform(-1, 1, (5000, 3)).astype(np.float32)
    if kind == "same":
        data[:] = data[0]
    elif kind == "line":
        data[:, 1:] = 0.5
    elif kind == "copies":
        data[100:] = data[np.arange(4900) % 100]
    elif kind == "far":
        data[7] = 1e18
    else:
        data[:, 0] = np.exp(12 * data[:, 0])
    q = np.concatenate([data[:20], rng.uniform(-3, 3, (20, 3)).astype(np.float32)])
    nn = index(0, 3, data)
    for k in (1, 40):
        same_knn(nn, oracle, 0, data, q, k)


def test_packed_batches(gpu, oracle):
    import torch

    data = points(gpu, 1, 7, 51, 5000)
    q = points(gpu, 1, 7, 52, 70)
    nn = index(1, 7, data)
    k = (np.arange(70) % 18 - 1).astype(np.int32)  # -1 .. 16
    off, gi, gd = nn.knn_packed_dev(torch.from_numpy(q).cuda(), torch.from_numpy(k).cuda(), 16)
    off, gi, gd = off.cpu().numpy(), gi.cpu().numpy(), gd.cpu().numpy()
    oi, od = oracle.knn(1, data, q, 16)
    for j in range(70):
        m = max(int(k[j]), 0)
        assert off[j + 1] - off[j] == m
        assert np.array_equal(gi[off[j]:off[j + 1]], oi[j, :m]) and np.array_equal(gd[off[j]:off[j + 1]], od[j, :m])
    r = np.linspace(-1.0, 4.0, 70).astype(np.float32)
    r[5] = np.nan
    off, gi, gd = nn.radius_packed_dev(torch.from_numpy(q).cuda(), torch.from_numpy(r).cuda())
    off, gi, gd = off.cpu().numpy(), gi.cpu().numpy(), gd.cpu().numpy()
    for j in range(70):
        if not r[j] >= 0:
            assert off[j + 1] == off[j]
            continue
        (oi, od), = oracle.radius(1, data, q[j:j + 1], float(r[j]))
        assert np.array_equal(gi[off[j]:off[j + 1]], oi) and np.array_equal(gd[off[j]:off[j + 1]], od)
