"""A device that is nearly full: memory that the library keeps of destroyed
structures is there for any of its allocations, and points are added where there
is room for them but not for their spatial index."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
MIB = 1 << 20


class Fill:
    """Takes what is left of the device in ever smaller pieces, down to `rest` bytes each."""

    def __init__(self, rest):
        import torch

        torch.cuda.empty_cache()
        self.hip = C.CDLL(next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line))
        self.held = []
        size = 1 << 36
        while size >= rest:
            p = C.c_void_p()
            if self.hip.hipMalloc(C.byref(p), C.c_size_t(size)) == 0:
                self.held.append(p)
            else:
                self.hip.hipGetLastError()
                size //= 2

    def free(self):
        for p in self.held:
            self.hip.hipFree(p)
        self.held = []


def kept_blocks(gpu, n):
    """Builds and destroys a structure; the library keeps its blocks (at most 768 MiB)."""
    import torch
    from ompl_amd.nn import NearestNeighborsGPU

    nn = NearestNeighborsGPU(1, 7)
    nn.add(torch.rand((n, 7), device="cuda"))
    nn.close()


def test_kept_blocks_serve_every_allocation(gpu):
    from ompl_amd._lib import call
    from ompl_amd.serve import Server

    kept_blocks(gpu, 4_000_000)  # 460 MB
    fill = Fill(16 * MIB)
    try:
        p = C.c_void_p()
        call("ompl_amd_malloc", C.byref(p), C.c_size_t(150 * MIB))
        call("ompl_amd_free", p)
    finally:
        fill.free()
    kept_blocks(gpu, 4_000_000)
    fill = Fill(16 * MIB)
    try:
        srv = Server(hbm_budget_bytes=150 * MIB, max_active=2, max_nodes=64)
        srv.close()
    finally:
        fill.free()


def test_points_without_room_for_the_index(gpu, oracle):
    import torch
    from ompl_amd._lib import OmplAmdError
    from ompl_amd.nn import NearestNeighborsGPU

    n = 4_000_000  # arrays of 290 MB, an index of 245
    rng = np.random.default_rng(8)
    data = rng.uniform(-3, 3, (n, 7)).astype(np.float32)
    pts, q = torch.from_numpy(data).cuda(), data[::1_000_000] + np.float32(0.01)
    nn = NearestNeighborsGPU(0, 7)
    room = Fill(1 << 62)  # (nothing held)
    p = C.c_void_p()
    assert room.hip.hipMalloc(C.byref(p), C.c_size_t(330 * MIB)) == 0
    fill = Fill(16 * MIB)
    room.hip.hipFree(p)
    try:
        nn.add(pts)
        gi, gd = nn.knn_batch(q, 5)
        oi, od = oracle.knn(0, data, q, 5)
        assert np.array_equal(gi, oi) and np.array_equal(gd, od)
        with pytest.raises(OmplAmdError):  # no room for the points: the structure is as it was
            nn.add(pts)
        gi, gd = nn.knn_batch(q, 5)
        assert np.array_equal(gi, oi) and np.array_equal(gd, od)
    finally:
        fill.free()
    nn.add(data[:10])  # (not grown yet: still the scan)
    assert nn.size() == n + 10
    nn.add(pts)
    gi, gd = nn.knn_batch(q, 5)
    oi, od = oracle.knn(0, np.concatenate([data, data[:10], data]), q, 5)
    assert np.array_equal(gi, oi) and np.array_equal(gd, od)
