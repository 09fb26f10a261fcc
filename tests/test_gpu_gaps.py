"""Walks that leave out the positions which the clearance of their neighbours
proves valid, against the oracle (validity, checked counts, lastValid): small obstacles
that an edge may touch between the positions looked at first, resolutions from a
few positions an edge to thousands, the sizes at which a walk changes shape (31,
32, 33 positions), coordinates at and beyond the range that clearances hold for."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
N = 4600  # most are survivors: more than the blocks of a launch


def dev(x):
    import torch

    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


@pytest.fixture(autouse=True)
def own_shape(gpu):
    saved = gpu.get_tuning()
    gpu.set_tuning(validity_lanes_per_state=8, validity_obstacle_parts=2, validity_shared_fk=0,
                   motion_lanes_per_state=8, motion_obstacle_parts=1, motion_strategy=3)
    yield
    gpu.set_tuning(**saved)


def points(seed, n):
    """Obstacles of no size, spread where the arm moves."""
    rng = np.random.default_rng(seed)
    c = rng.normal(size=(n, 3))
    c *= rng.uniform(0.5, 2.1, (n, 1)) / np.linalg.norm(c, axis=1, keepdims=True)
    return np.concatenate([c, np.zeros((n, 1))], 1).astype(np.float32)


@pytest.mark.parametrize("lvs,lo,hi", [(0.3, 0.5, 9.5), (0.05, 1.5, 1.7), (0.01, 0.05, 6.0), (0.0006, 0.02, 0.6)])
@pytest.mark.parametrize("n_obs,offset", [(6, 0.0), (40, 0.0), (12, 13.0), (12, 400.0)])
def test_edges_between_points(gpu, oracle, lvs, lo, hi, n_obs, offset):
    s, none = points(n_obs, n_obs), np.zeros((0, 6), np.float32)
    env, oenv = gpu.Env(s, none), oracle.OracleEnv(s, none)
    rng = np.random.default_rng(int(1e5 * lvs) + n_obs)
    a = rng.uniform(-3, 3, (N, 7)) + offset
    d = rng.normal(size=(N, 7))
    b = a + d * rng.uniform(lo, hi, (N, 1)) / np.linalg.norm(d, axis=1, keepdims=True)
    rv, rc = oracle.check_motions(oenv, a, b, lvs, threads=8)
    A, B = dev(a.T), dev(b.T)
    v, c = gpu.check_motions(env, A, B, lvs, exact_count=True)
    assert np.array_equal(v.cpu().numpy(), rv) and np.array_equal(c.cpu().numpy(), rc)
    assert np.array_equal(gpu.check_motions(env, A, B, lvs).cpu().numpy(), rv)
    assert 0 < rv.sum() < N
    lv, lt = gpu.check_motions_last_valid(env, A, B, lvs)
    lv, lt = lv.cpu().numpy(), lt.cpu().numpy()
    assert np.array_equal(lv, rv) and np.isnan(lt[rv == 1]).all()
    for i in np.flatnonzero(rv == 0)[:400]:
        assert lt[i] == oracle.check_motion_last_valid(oenv, a[i], b[i], lvs)[1], i
