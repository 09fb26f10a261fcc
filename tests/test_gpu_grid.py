"""GPU parity of the checks over the environment's cell grid (the library's own
choice of shape) with the CPU oracle: scenes at the edges of what a cell can
say (nothing in reach, cells with long lists or none that fits, obstacles
across the border of the workspace, contact within a rounding), states beyond
the range of the sine, batches at the edges of the lane mappings and of the
one-launch form, and walks past what one block takes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
PI = np.pi
LVS = 0.01


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


def scene(gpu, kind):
    rng = np.random.default_rng(3)
    none_s, none_b = np.zeros((0, 4), np.float32), np.zeros((0, 6), np.float32)
    if kind == "mixed":
        return gpu.workload.obstacles(1001, 40, 30)
    if kind == "one point":
        return np.array([[0.6, 0.1, 0.5, 0.0]], np.float32), none_b
    if kind == "out of reach":
        return np.array([[30.0, 0, 0, 2.0]], np.float32), np.array([[0, -9.0, 0, 1, 1, 1]], np.float32)
    if kind == "huge":  # most of each obstacle is outside the workspace
        return (np.array([[1000.0, 0, 0, 998.9], [0, 0, -60.0, 59.2]], np.float32),
                np.array([[0, 40.0, 0, 500, 38.8, 500], [-1.9, 0, 0, 0.0, 3, 3]], np.float32))
    if kind == "cluster":  # dozens of surfaces through the same cells
        c = np.array([0.7, 0.2, 0.6]) + rng.normal(0, 0.01, (300, 3))
        s = np.concatenate([c, rng.uniform(0.0, 0.05, (300, 1))], 1).astype(np.float32)
        b = np.concatenate([c[:120] + 0.3, rng.uniform(0, 0.03, (120, 3))], 1).astype(np.float32)
        return s, b
    if kind == "beyond lists":  # more surfaces in a cell than a list holds, and than a brick keeps
        c = np.array([0.7, 0.2, 0.6]) + rng.normal(0, 0.004, (700, 3))
        return np.concatenate([c, rng.uniform(0.01, 0.03, (700, 1))], 1).astype(np.float32), none_b
    if kind == "base":  # touches the base link
        return np.array([[0.05, 0.0, 0.2, 0.02]], np.float32), none_b
    return none_s, none_b


KINDS = ["mixed", "none", "one point", "out of reach", "huge", "cluster", "beyond lists", "base"]


@pytest.mark.parametrize("kind", KINDS)
def test_validity_scenes(gpu, oracle, kind):
    s, b = scene(gpu, kind)
    env, oenv = gpu.Env(s, b), oracle.OracleEnv(s, b)
    q = np.random.default_rng(5).uniform(-PI, PI, (6000, 7)).astype(np.float32)
    q[:200] = 0.0
    q[:200, 1] = np.linspace(-PI, PI, 200)
    qs = q.T.copy()
    ref = oracle.validate_states(oenv, qs)
    assert np.array_equal(gpu.validate_states(env, dev(qs)).cpu().numpy(), ref)
    big = np.tile(qs, (1, 22))[:, :131_072]  # one lane per state
    got = gpu.validate_states(env, dev(big)).cpu().numpy()
    assert np.array_equal(got, np.tile(ref, 22)[:131_072])


@pytest.mark.parametrize("n", [1, 31, 32, 33, 131_071, 131_073])
@pytest.mark.parametrize("f64", [False, True])
def test_validity_sizes(gpu, oracle, n, f64):
    s, b = scene(gpu, "mixed")
    env, oenv = gpu.Env(s, b), oracle.OracleEnv(s, b)
    q = np.random.default_rng(n).uniform(-PI, PI, (7, n)).astype(np.float64 if f64 else np.float32)
    got = gpu.validate_states(env, dev(q)).cpu().numpy()
    sel = np.unique(np.linspace(0, n - 1, min(n, 3000)).astype(int))
    assert np.array_equal(got[sel], oracle.validate_states(oenv, q[:, sel].astype(np.float32)))


def test_contact_within_a_rounding(gpu, oracle):
    """Point obstacles at the contact distance of robot spheres, give or take 1e-7 m."""
    rng = np.random.default_rng(9)
    q = rng.uniform(-PI, PI, (400, 7)).astype(np.float32)
    c = np.stack([oracle.arm_spheres(x) for x in q])
    i = rng.integers(8, 28, 400)
    d = rng.normal(size=(400, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    at = c[np.arange(400), i] + d * (0.08 + rng.uniform(-2e-7, 2e-7, (400, 1)))
    for k in range(0, 400, 50):
        s = np.concatenate([at[k:k + 50], np.full((50, 1), 0.03)], 1).astype(np.float32)
        env, oenv = gpu.Env(s, None), oracle.OracleEnv(s, np.zeros((0, 6), np.float32))
        qs = np.tile(q[k:k + 50].T, (1, 4)).copy()
        assert np.array_equal(gpu.validate_states(env, dev(qs)).cpu().numpy(), oracle.validate_states(oenv, qs))


@pytest.mark.parametrize("kind", ["mixed", "huge"])
@pytest.mark.parametrize("n", [500, 140_000])
def test_states_beyond_the_sine(gpu, oracle, kind, n):
    s, b = scene(gpu, kind)
    env, oenv = gpu.Env(s, b), oracle.OracleEnv(s, b)
    rng = np.random.default_rng(2)
    q = rng.uniform(-PI, PI, (7, n)).astype(np.float32)
    odd = rng.choice(n, 120, replace=False)
    vals = np.array([np.nan, np.inf, -np.inf, 5999.0, -6001.0, 1e5], np.float32)
    q[rng.integers(0, 7, 120), odd] = vals[np.arange(120) % 6]
    got = gpu.validate_states(env, dev(q)).cpu().numpy()
    sel = np.unique(np.concatenate([odd, np.arange(300)]))
    assert np.array_equal(got[sel], oracle.validate_states(oenv, q[:, sel].copy()))


@pytest.mark.parametrize("n", [1, 3, 1023, 1024, 1025, 5000])
@pytest.mark.parametrize("kind,mu", [("mixed", -1.0), ("one point", 0.0), ("base", -1.0), ("none", -1.0)])
def test_motions_and_last_valid(gpu, oracle, n, kind, mu):
    s, b = scene(gpu, kind)
    env, oenv = gpu.Env(s, b), oracle.OracleEnv(s, b)
    a_, b_ = gpu.workload.edges(n, n, mu, 1.2, 0.001, 9.0)
    b_[0] = a_[0]
    A, B = dev(a_.T), dev(b_.T)
    rv, rc = oracle.check_motions(oenv, a_, b_, LVS, threads=8)
    for _ in range(3):  # both counter sets
        v, c = gpu.check_motions(env, A, B, LVS, exact_count=True)
        assert np.array_equal(v.cpu().numpy(), rv) and np.array_equal(c.cpu().numpy(), rc)
        assert np.array_equal(gpu.check_motions(env, A, B, LVS).cpu().numpy(), rv)
        lv, lt = gpu.check_motions_last_valid(env, A, B, LVS)
        lv, lt = lv.cpu().numpy(), lt.cpu().numpy()
        for i in np.unique(np.linspace(0, n - 1, min(n, 400)).astype(int)):
            ov, ot, _ = oracle.check_motion_last_valid(oenv, a_[i], b_[i], LVS)
            assert lv[i] == ov and (np.isnan(lt[i]) if ov else lt[i] == ot)


@pytest.mark.parametrize("n", [4, 1200, 3000])
def test_long_walks(gpu, oracle, n):
    """Edges of more segments than one block walks by itself, among short ones
    and ones with too many segments, valid and not."""
    s = np.array([[0.9, 0.3, 0.8, 0.01]], np.float32)
    env, oenv = gpu.Env(s, None), oracle.OracleEnv(s, np.zeros((0, 6), np.float32))
    rng = np.random.default_rng(n)
    a_ = rng.uniform(-1, 1, (n, 7))
    b_ = a_ + rng.normal(0, 0.002, (n, 7))
    a_[:4], b_[:4] = 0.0, 0.0
    b_[0, 0] = 3.0                      # valid: 20,000 segments and more
    a_[1] = np.array([0.2, 0.3, 0, 0.4, 0, 0.1, 0])
    b_[1] = a_[1] + 1.5
    b_[2, 5] = 2.6
    lvs = 1e-4
    rv, rc = oracle.check_motions(oenv, a_, b_, lvs, threads=8)
    b_[3, 1] = 1e5                      # too many segments (the oracle would walk them all)
    rv[3] = rc[3] = 0
    A, B = dev(a_.T), dev(b_.T)
    for _ in range(2):
        v, c = gpu.check_motions(env, A, B, lvs, exact_count=True)
        assert np.array_equal(v.cpu().numpy(), rv) and np.array_equal(c.cpu().numpy(), rc)
    lv, lt = gpu.check_motions_last_valid(env, A, B, lvs)
    lv, lt = lv.cpu().numpy(), lt.cpu().numpy()
    for i in list(range(3)) + list(range(4, n, max(1, n // 50))):
        ov, ot, _ = oracle.check_motion_last_valid(oenv, a_[i], b_[i], lvs)
        assert lv[i] == ov and (np.isnan(lt[i]) if ov else lt[i] == ot)
    assert lv[3] == 0


@pytest.mark.parametrize("n_lists", [7, 1500])
def test_state_lists(gpu, oracle, n_lists):
    s, b = scene(gpu, "one point")
    env, oenv = gpu.Env(s, b), oracle.OracleEnv(s, b)
    rng = np.random.default_rng(n_lists)
    pool = rng.uniform(-PI, PI, (20_000, 7))
    ok = oracle.validate_states(oenv, pool.astype(np.float32).T.copy()) == 1
    good, bad = pool[ok], pool[~ok]
    sizes = np.array([0, 1, 63, 64, 65, 256, 257] + [40_000] + rng.integers(0, 90, 4000).tolist())[:n_lists]
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    st = good[rng.integers(0, len(good), off[-1])].copy()
    want = np.full(n_lists, -1)
    for i in range(n_lists):
        if sizes[i] and rng.random() < 0.6:
            want[i] = rng.integers(0, sizes[i])
            st[off[i] + want[i]] = bad[i % len(bad)]
    if n_lists > 7:
        want[7] = 39_000
        st[off[7]:off[8]] = good[:1]
        st[off[7] + 39_000] = bad[0]
    for _ in range(2):
        v, f = gpu.check_state_lists(env, dev(st.T), dev(off))
        assert np.array_equal(f.cpu().numpy(), want) and np.array_equal(v.cpu().numpy() == 1, want < 0)
