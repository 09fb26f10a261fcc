"""A k-NN search captured into a graph and replayed while the structure goes on:
additions that build the index again, removals, a clear, with eager searches
between the replays.  Every replay against the CPU oracle over the ids that were
there at the capture.  (9 dimensions: the full scan, whose working space the
eager searches of more points outgrow.)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("metric,dim", [(0, 3), (0, 7), (0, 9), (1, 7)])
@pytest.mark.parametrize("nq", [30, 7000])
def test_replays(gpu, oracle, metric, dim, nq):
    import torch
    from ompl_amd.nn import NearestNeighborsGPU

    k, n, all_ = 9, 5000, 7900  # within the capacity of 8,192
    rng = np.random.default_rng(dim)
    draw = (lambda m, s: gpu.workload.se3(s, m)) if metric else \
        (lambda m, s: rng.uniform(-3, 3, (m, dim)).astype(np.float32))
    data, q = draw(all_, 1), draw(nq, 2)
    dev = torch.from_numpy(q).cuda()
    out_i = torch.empty((nq, k), dtype=torch.int32, device="cuda")
    out_d = torch.empty((nq, k), dtype=torch.float32, device="cuda")
    nn = NearestNeighborsGPU(metric, dim)
    nn.add(data[:n])
    side = torch.cuda.Stream()
    nn.knn_dev(dev, k, out_i, out_d, stream=side.cuda_stream)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        nn.knn_dev(dev, k, out_i, out_d, stream=side.cuda_stream)
    some = np.unique(np.linspace(0, nq - 1, 30).astype(int))

    def same(i, d, pts, ids):
        oi, od = oracle.knn(metric, pts[ids], q[some], k)
        assert np.array_equal(i[some], ids[oi]) and np.array_equal(d[some], od)

    def replay(pts, ids, total):
        out_i.fill_(-7)
        graph.replay()
        torch.cuda.synchronize()
        same(out_i.cpu().numpy(), out_d.cpu().numpy(), pts, ids)
        same(*nn.knn_batch(q, k), pts, total)  # the eager search sees all points

    ids = np.arange(n)
    replay(data, ids, ids)
    replay(data, ids, ids)
    gone = np.zeros(0, int)
    for m in (5300, 6000, all_):  # a tail, then builds
        nn.add(data[nn.size() + len(gone):m])
        replay(data, ids, np.setdiff1d(np.arange(m), gone))
        new = np.setdiff1d(rng.choice(m, 60, replace=False), gone)
        for i in new:
            assert nn.remove(int(i))
        gone = np.concatenate([gone, new])
        ids = np.setdiff1d(np.arange(n), gone)
        replay(data, ids, np.setdiff1d(np.arange(m), gone))
    nn.clear()
    other = draw(6000, 3)
    nn.add(other)
    replay(other, np.arange(n), np.arange(6000))
