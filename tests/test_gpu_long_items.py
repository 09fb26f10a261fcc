"""Long edges and lists (more positions than one block walks) in batches of one
launch and of two, valid and invalid early, late and nowhere, batch after
batch on one stream: each batch leaves its words as the next expects them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
LVS = 1e-4


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


# one edge, a few, the most of the one-launch form, the fewest of the other, more survivors than blocks
@pytest.mark.parametrize("n", [1, 5, 1024, 1025, 2600])
def test_batches_of_long_edges(gpu, oracle, n):
    s = np.array([[0.9, 0.3, 0.8, 0.05]], np.float32)
    env, oenv = gpu.Env(s, None), oracle.OracleEnv(s, np.zeros((0, 6), np.float32))
    ok = [q for q in np.random.default_rng(1).uniform(-3, 3, (400, 7))
          if oracle.state_valid(oenv, q.astype(np.float32))]
    batches = []
    for k in range(3):
        rng = np.random.default_rng(10 * n + k)
        a = np.array(ok)[rng.integers(0, len(ok), n)]
        b = a + rng.normal(0, 0.003, (n, 7))
        for e in rng.choice(n, min(n, 4), replace=False):  # 17,000 to 60,000 positions
            a[e], b[e] = ok[rng.integers(len(ok))], ok[rng.integers(len(ok))]
            b[e] = a[e] + (b[e] - a[e]) * rng.uniform(1.7, 6.0) / np.linalg.norm(b[e] - a[e])
        batches.append((a, b, oracle.check_motions(oenv, a, b, LVS, threads=8)))
    for a, b, (rv, rc) in batches * 2:
        A, B = dev(a.T), dev(b.T)
        v, c = gpu.check_motions(env, A, B, LVS, exact_count=True)
        assert np.array_equal(v.cpu().numpy(), rv) and np.array_equal(c.cpu().numpy(), rc)
        assert np.array_equal(gpu.check_motions(env, A, B, LVS).cpu().numpy(), rv)
        lv, lt = gpu.check_motions_last_valid(env, A, B, LVS)
        lv, lt = lv.cpu().numpy(), lt.cpu().numpy()
        assert np.array_equal(lv, rv)
        for i in np.flatnonzero(rv == 0)[:20]:
            assert lt[i] == oracle.check_motion_last_valid(oenv, a[i], b[i], LVS)[1]


@pytest.mark.parametrize("n_lists", [1, 9, 1024])
def test_one_launch_of_long_lists(gpu, oracle, n_lists):
    s = np.array([[0.6, 0.1, 0.5, 0.1]], np.float32)
    env, oenv = gpu.Env(s, None), oracle.OracleEnv(s, np.zeros((0, 6), np.float32))
    pool = np.random.default_rng(2).uniform(-3, 3, (4000, 7))
    good_of = oracle.validate_states(oenv, pool.astype(np.float32).T.copy()) == 1
    for k, long_bad in enumerate([None, 0, 16_384, 29_999, None]):
        rng = np.random.default_rng(100 * n_lists + k)
        sizes = rng.integers(0, 40, n_lists)
        sizes[k % n_lists] = 30_000
        off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
        st = pool[good_of][rng.integers(0, good_of.sum(), off[-1])]
        want = np.full(n_lists, -1)
        if long_bad is not None:
            st[off[k % n_lists] + long_bad] = pool[~good_of][0]
            want[k % n_lists] = long_bad
        v, f = gpu.check_state_lists(env, dev(st.T), dev(off))
        assert np.array_equal(f.cpu().numpy(), want) and np.array_equal(v.cpu().numpy() == 1, want < 0)
