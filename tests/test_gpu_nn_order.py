"""Calls that follow an asynchronous ompl_amd_nn_add_dev at once, while the
build of the spatial index that it starts is still waiting on its own stream:
removals, a clear, and additions on another stream.  Results against the CPU
oracle."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def add_dev(nn, pts, stream):
    from ompl_amd._lib import call

    first = C.c_int64()
    call("ompl_amd_nn_add_dev", nn.handle, C.c_void_p(pts.data_ptr()), pts.shape[0], C.byref(first),
         C.c_void_p(stream.cuda_stream))
    return first.value


def busy(torch, stream):
    """Some milliseconds of work in front of what the stream gets next."""
    with torch.cuda.stream(stream):
        a = torch.ones((2048, 2048), device="cuda")
        for _ in range(20):
            a = a @ a * 1e-4
    return a


def expect(nn, oracle, data, ids, q, k=12):
    gi, gd = nn.knn_batch(q, k)
    oi, od = oracle.knn(0, data[ids], q, k)
    assert np.array_equal(gi, ids[oi]) and np.array_equal(gd, od)


@pytest.mark.parametrize("room", [False, True])
def test_remove_behind_a_pending_build(gpu, oracle, room):
    import torch
    from ompl_amd.nn import NearestNeighborsGPU

    rng = np.random.default_rng(3)
    data = rng.uniform(-3, 3, (12_000, 3)).astype(np.float32)
    q = rng.uniform(-3, 3, (50, 3)).astype(np.float32)
    nn = NearestNeighborsGPU(0, 3)
    if room:  # the arrays hold all points already
        nn.add(data)
        nn.clear()
    nn.add(data[:3000])
    dev = torch.from_numpy(data).cuda()
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    keep = [busy(torch, side)]
    assert add_dev(nn, dev[3000:], side) == 3000
    gone = np.concatenate([rng.choice(3000, 40, replace=False), 3000 + rng.choice(9000, 40, replace=False)])
    for i in gone:
        assert nn.remove(int(i))
    torch.cuda.synchronize()
    del keep
    expect(nn, oracle, data, np.setdiff1d(np.arange(12_000), gone), q)


def test_clear_and_add_on_another_stream(gpu, oracle):
    import torch
    from ompl_amd.nn import NearestNeighborsGPU

    rng = np.random.default_rng(4)
    data = rng.uniform(-3, 3, (20_000, 7)).astype(np.float32)
    q = rng.uniform(-3, 3, (50, 7)).astype(np.float32)
    nn = NearestNeighborsGPU(0, 7)
    nn.add(data)
    nn.clear()
    dev = torch.from_numpy(data).cuda()
    one, two = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    keep = [busy(torch, one)]
    add_dev(nn, dev[:10_000], one)
    nn.clear()
    assert add_dev(nn, dev[10_000:], two) == 0
    torch.cuda.synchronize()
    del keep
    expect(nn, oracle, data[10_000:], np.arange(10_000), q)
