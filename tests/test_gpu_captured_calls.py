"""Batched checks that a caller captures into a graph of its own and replays,
with eager calls on the same stream between the replays: each replay must start
from empty lists, whatever ran before it.  Sizes of the one-launch form and
above, edges and lists long enough for the long-item path."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def dev(x):
    import torch

    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


def captured(call, side):
    import torch

    call()  # sizes the stream's workspace
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = call()
    return graph, out


def replay(graph, side):
    import torch

    with torch.cuda.stream(side):
        graph.replay()
    torch.cuda.synchronize()


@pytest.mark.parametrize("n", [700, 3000, 140_000])
@pytest.mark.parametrize("counts", [False, True])
def test_motions(gpu, oracle, n, counts):
    import torch

    s, b = gpu.workload.obstacles(1001, 20, 16)
    env, oenv = gpu.Env(s, b), oracle.OracleEnv(s, b)
    a_, b_ = gpu.workload.edges(n, n, -1.0, 1.2, 0.001, 9.0)
    sel = np.unique(np.linspace(0, n - 1, min(n, 3000)).astype(int))
    rv, rc = oracle.check_motions(oenv, a_[sel], b_[sel], 0.05, threads=8)
    assert 0 < rv.sum() < len(sel)
    A, B = dev(a_.T), dev(b_.T)
    side = torch.cuda.Stream()

    def call():
        return gpu.check_motions(env, A, B, 0.05, exact_count=counts, stream=side.cuda_stream)

    def same(out):
        v, c = out if counts else (out, None)
        assert np.array_equal(v.cpu().numpy()[sel], rv)
        assert c is None or np.array_equal(c.cpu().numpy()[sel], rc)

    graph, out = captured(call, side)
    for i in range(4):
        for t in out if counts else (out,):
            t.fill_(77)
        torch.cuda.synchronize()
        replay(graph, side)
        same(out)
        for _ in range(i):  # either set of the eager batches may be next
            eager = call()
            torch.cuda.synchronize()
            same(eager)


@pytest.mark.parametrize("n", [4, 1200])
def test_long_edges(gpu, oracle, n):
    import torch

    s = np.array([[0.9, 0.3, 0.8, 0.01]], np.float32)
    env, oenv = gpu.Env(s, None), oracle.OracleEnv(s, np.zeros((0, 6), np.float32))
    rng = np.random.default_rng(n)
    a_ = rng.uniform(-1, 1, (n, 7))
    b_ = a_ + rng.normal(0, 0.002, (n, 7))
    a_[:3], b_[:3] = 0.0, 0.0
    b_[0, 0] = 3.0
    a_[1] = np.array([0.2, 0.3, 0, 0.4, 0, 0.1, 0])
    b_[1] = a_[1] + 1.5
    b_[2, 5] = 2.6
    lvs = 1e-4
    rv, rc = oracle.check_motions(oenv, a_, b_, lvs, threads=8)
    sel = np.concatenate([np.arange(4), np.arange(4, n, max(1, n // 50))]) if n > 4 else np.arange(4)
    last = [oracle.check_motion_last_valid(oenv, a_[i], b_[i], lvs) for i in sel]
    A, B = dev(a_.T), dev(b_.T)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        graph, (v, c) = captured(lambda: gpu.check_motions(env, A, B, lvs, exact_count=True), side)
        lgraph, (lv, lt) = captured(lambda: gpu.check_motions_last_valid(env, A, B, lvs), side)
    for _ in range(3):
        replay(graph, side)
        assert np.array_equal(v.cpu().numpy(), rv) and np.array_equal(c.cpu().numpy(), rc)
        replay(lgraph, side)
        for i, (ov, ot, _) in zip(sel, last):
            assert lv[i].item() == ov and (np.isnan(lt[i].item()) if ov else lt[i].item() == ot)


@pytest.mark.parametrize("n_lists", [5, 1500])
def test_state_lists(gpu, oracle, n_lists):
    import torch

    s = np.array([[0.6, 0.1, 0.5, 0.0]], np.float32)
    env, oenv = gpu.Env(s, None), oracle.OracleEnv(s, np.zeros((0, 6), np.float32))
    rng = np.random.default_rng(n_lists)
    pool = rng.uniform(-np.pi, np.pi, (20_000, 7))
    ok = oracle.validate_states(oenv, pool.astype(np.float32).T.copy()) == 1
    good, bad = pool[ok], pool[~ok]
    sizes = np.concatenate([[40_000, 0, 65], rng.integers(0, 90, n_lists)])[:n_lists]
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    st = good[rng.integers(0, len(good), off[-1])].copy()
    want = np.full(n_lists, -1)
    want[0] = 39_000
    st[off[0] + 39_000] = bad[0]
    for i in range(3, n_lists, 2):
        if sizes[i]:
            want[i] = sizes[i] // 2
            st[off[i] + want[i]] = bad[i % len(bad)]
    Q, O = dev(st.T), dev(off)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        graph, (v, f) = captured(lambda: gpu.check_state_lists(env, Q, O), side)
    for _ in range(3):
        replay(graph, side)
        assert np.array_equal(f.cpu().numpy(), want) and np.array_equal(v.cpu().numpy() == 1, want < 0)


def test_larger_eager_batches(gpu, oracle):
    """Eager calls outgrow the stream's workspace, which a captured batch goes on using."""
    import torch

    s, b = gpu.workload.obstacles(1001, 20, 16)
    env, oenv = gpu.Env(s, b), oracle.OracleEnv(s, b)
    side = torch.cuda.Stream()
    runs = []
    for n in (2000, 30_000, 200_000):
        a_, b_ = gpu.workload.edges(n, n, -1.0, 1.2, 0.001, 9.0)
        sel = np.unique(np.linspace(0, n - 1, 2000).astype(int))
        want = oracle.check_motions(oenv, a_[sel], b_[sel], 0.05, threads=8)
        A, B = dev(a_.T), dev(b_.T)
        with torch.cuda.stream(side):
            graph, out = captured(lambda: gpu.check_motions(env, A, B, 0.05, exact_count=True), side)
        runs.append((graph, out, sel, want, (A, B)))
        for _ in range(2):
            for graph, (v, c), sel_, (rv, rc), _keep in runs:
                v.fill_(77)
                torch.cuda.synchronize()
                replay(graph, side)
                assert np.array_equal(v.cpu().numpy()[sel_], rv) and np.array_equal(c.cpu().numpy()[sel_], rc)
