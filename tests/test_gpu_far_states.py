"""States beyond the sine's range are tested against every obstacle: in scenes
of one to three obstacles, where a scan's length is that of a cell that names
its obstacles, and in scenes none of whose obstacles is within the arm's reach.
GPU parity with the CPU oracle in both lane mappings and through motions,
lastValid and state lists."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
PI = np.pi
SCENES = {
    "sphere": ([[0.7, 0.1, 0.6, 0.1]], []),
    "two spheres": ([[0.3, 0.0, 0.2, 0.01], [0.9, 0.3, 0.8, 0.4]], []),
    "sphere and box": ([[0.3, 0.0, 0.2, 0.01]], [[0.9, 0.3, 0.8, 0.4, 0.4, 0.3]]),
    "two boxes": ([], [[0.3, 0.0, 0.2, 0.01, 0.01, 0.01], [-0.9, 0.3, 0.8, 0.4, 0.4, 0.3]]),
    "three": ([[0.3, 0.0, 0.2, 0.01], [0.5, -0.6, 0.9, 0.02]], [[0.9, 0.3, 0.8, 0.4, 0.4, 0.3]]),
}


def dev(x):
    import torch

    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


def arrays(name):
    s, b = SCENES[name]
    return np.array(s, np.float32).reshape(-1, 4), np.array(b, np.float32).reshape(-1, 6)


def far_states(n, seed):
    q = np.random.default_rng(seed).uniform(-PI, PI, (7, n)).astype(np.float32)
    q[0] = np.random.default_rng(seed + 1).uniform(6001.0, 6500.0, n)
    q[6, ::5] = np.inf  # the links before it have finite centres
    return q


@pytest.mark.parametrize("name", SCENES)
@pytest.mark.parametrize("n", [2000, 140_000])
def test_few_obstacles(gpu, oracle, name, n):
    s, b = arrays(name)
    env, oenv = gpu.Env(s, b), oracle.OracleEnv(s, b)
    q = far_states(n, 5)
    want = oracle.validate_states_mt(oenv, q, 8)
    last = (s[:-1], b) if not len(b) else (s, b[:-1])
    if len(s) + len(b) > 1:  # most collisions are with the last obstacle
        without = oracle.validate_states_mt(oracle.OracleEnv(*last), q, 8)
        assert ((want == 0) & (without == 1)).sum() > 50
    assert np.array_equal(gpu.validate_states(env, dev(q)).cpu().numpy(), want)
    assert np.array_equal(gpu.validate_states(env, dev(q.astype(np.float64))).cpu().numpy(), want)


@pytest.mark.parametrize("name", ["two spheres", "sphere and box"])
@pytest.mark.parametrize("n", [40, 3000])
def test_walks_of_few_obstacles(gpu, oracle, name, n):
    s, b = arrays(name)
    env, oenv = gpu.Env(s, b), oracle.OracleEnv(s, b)
    rng = np.random.default_rng(n)
    a_ = rng.uniform(-PI, PI, (n, 7))
    a_[:, 0] += 6100.0
    b_ = a_ + rng.normal(0, 0.3, (n, 7))
    rv, rc = oracle.check_motions(oenv, a_, b_, 0.05, threads=8)
    assert 0 < rv.sum() < n
    v, c = gpu.check_motions(env, dev(a_.T), dev(b_.T), 0.05, exact_count=True)
    assert np.array_equal(v.cpu().numpy(), rv) and np.array_equal(c.cpu().numpy(), rc)
    lv, lt = gpu.check_motions_last_valid(env, dev(a_.T), dev(b_.T), 0.05)
    lv, lt = lv.cpu().numpy(), lt.cpu().numpy()
    for i in np.unique(np.linspace(0, n - 1, 200).astype(int)):
        ov, ot, _ = oracle.check_motion_last_valid(oenv, a_[i], b_[i], 0.05)
        assert lv[i] == ov and (np.isnan(lt[i]) if ov else lt[i] == ot)
    ok = oracle.validate_states(oenv, b_.astype(np.float32).T.copy()) == 1
    v, f = gpu.check_state_lists(env, dev(b_.T), dev(np.array([0, n // 2, n], np.int64)))
    for i, part in enumerate((ok[:n // 2], ok[n // 2:])):
        assert v.cpu().numpy()[i] == part.all() and f.cpu().numpy()[i] == (-1 if part.all() else np.argmin(part))


@pytest.mark.parametrize("n", [500, 140_000])
def test_nothing_in_reach(gpu, oracle, n):
    """Beyond 1e8 rad the polynomial's centres leave the workspace, and may
    meet an obstacle that no arm can reach."""
    s = np.array([[0, 0, 300.0, 290.0]], np.float32)
    b = np.array([[-900.0, 0, 0, 890.0, 890.0, 890.0]], np.float32)
    env, oenv = gpu.Env(s, b), oracle.OracleEnv(s, b)
    rng = np.random.default_rng(n)
    q = rng.uniform(-PI, PI, (7, n)).astype(np.float32)
    far = rng.choice(n, n // 4, replace=False)
    q[rng.integers(1, 6, n // 4), far] = rng.uniform(1e8, 9e8, n // 4).astype(np.float32)
    want = oracle.validate_states_mt(oenv, q, 8)
    assert (want == 0).sum() > 10 and want[np.setdiff1d(np.arange(n), far)].all()
    assert np.array_equal(gpu.validate_states(env, dev(q)).cpu().numpy(), want)
