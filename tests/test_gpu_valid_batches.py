"""GPU parity of the valid-state sampler's batches with the CPU oracle: calls
that end within, at and past a batch of draws, attempts from one on, scenes
with nothing and everything valid, more calls than one launch takes, and the
generators' place afterwards."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def scene(gpu, oracle, kind):
    if kind == "nothing valid":
        s, b = np.array([[0.05, 0.0, 0.2, 0.02]], np.float32), np.zeros((0, 6), np.float32)
    elif kind == "everything valid":
        s, b = np.zeros((0, 4), np.float32), np.zeros((0, 6), np.float32)
    else:
        s, b = gpu.workload.obstacles(1002, 48, 48)
    return gpu.Env(s, b), oracle.OracleEnv(s, b)


def same(got, want):
    return all(np.array_equal(g, w) for g, w in zip(got, want))


@pytest.mark.parametrize("kind", ["nothing valid", "everything valid", "mixed"])
@pytest.mark.parametrize("calls,attempts", [(1, 1), (2, 511), (3, 512), (2, 513), (63, 100), (513, 1), (700, 3)])
def test_batches(gpu, oracle, kind, calls, attempts):
    from ompl_amd.sampler import sample_valid

    env, oenv = scene(gpu, oracle, kind)
    seeds = np.array([1, 2 ** 32 - 1, 77], np.uint32)
    got = [t.cpu().numpy() for t in sample_valid(env, seeds, calls, attempts=attempts)]
    for i, sd in enumerate(seeds.tolist()):
        assert same([g[i] for g in got], oracle.Mt19937(sd).sample_valid(oenv, calls, attempts)), i


@pytest.mark.parametrize("kind,calls,attempts", [("nothing valid", 2700, 100), ("mixed", 5400, 50)])
def test_more_than_one_launch(gpu, oracle, kind, calls, attempts):
    from ompl_amd.sampler import Rng, sample_valid

    env, oenv = scene(gpu, oracle, kind)
    seeds = np.array([5, 6], np.uint32)
    lo, hi = np.full(7, -np.pi), np.full(7, np.pi)
    got = [t.cpu().numpy() for t in sample_valid(env, seeds, calls, attempts=attempts)]
    rng = Rng(seeds)
    kept = [t.cpu().numpy() for t in rng.valid(env, calls, attempts=attempts)]
    after = rng.uniform(50, lo, hi).cpu().numpy()
    rng.close()
    for i, sd in enumerate(seeds.tolist()):
        g = oracle.Mt19937(sd)
        want = g.sample_valid(oenv, calls, attempts)
        assert same([x[i] for x in got], want) and same([x[i] for x in kept], want), i
        assert np.array_equal(after[i], g.sample_uniform(lo, hi, 50)), i


@pytest.mark.parametrize("dim,n", [(1, 311), (1, 312), (1, 313), (16, 40), (7, 45)])
def test_uniform_across_twists(gpu, oracle, dim, n):
    from ompl_amd.sampler import Rng, sample_uniform

    seeds = np.array([9, 10], np.uint32)
    lo, hi = np.linspace(-3, -1, dim), np.linspace(1, 5, dim)
    out, f32 = sample_uniform(seeds, n, lo, hi, f32_soa=True)
    out, f32 = out.cpu().numpy(), f32.cpu().numpy()
    rng = Rng(seeds)
    parts = [rng.uniform(k, lo, hi).cpu().numpy() for k in (1, n, 700)]
    rng.close()
    for i, sd in enumerate(seeds.tolist()):
        assert np.array_equal(out[i], oracle.Mt19937(sd).sample_uniform(lo, hi, n))
        assert np.array_equal(f32[:, i * n:(i + 1) * n].T, out[i].astype(np.float32))
        g = oracle.Mt19937(sd)
        assert all(np.array_equal(p[i], g.sample_uniform(lo, hi, p.shape[1])) for p in parts)
