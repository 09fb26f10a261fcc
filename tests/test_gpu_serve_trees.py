"""Served plans over the sizes at which the slice kernel changes path: trees
beyond the nodes it keeps in LDS (one wave a step in place of a quarter),
generator blocks used up in the middle of a round of steps, an iteration limit
inside a round, solutions longer than the rows it returns in place."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LVS = 0.01


# range, iteration limit, threads: small trees and limits within the first round (1, 2, 31, 33), trees of
# several hundred nodes, short steps (paths of over 128 states)
@pytest.mark.parametrize("rng,iters,threads", [(0.0, 1, 512), (0.0, 2, 512), (0.0, 31, 512), (0.0, 33, 1024),
                                               (0.0, 600, 512), (0.3, 1500, 512), (0.3, 1500, 1024),
                                               (0.02, 60, 512)])
def test_served_equals_oracle_across_sizes(gpu, oracle, rng, iters, threads):
    from ompl_amd.serve import Server, make_request

    s, b = gpu.workload.obstacles(1041, 20, 20)
    env, oenv = gpu.Env(s, b), oracle.OracleEnv(s, b)
    ok = [q for q in gpu.workload.configs(1042, 3000) if oracle.state_valid(oenv, q.astype(np.float32))]
    pairs = [(ok[2 * i], ok[2 * i + 1]) for i in range(6)]
    maxd = rng or 0.2 * 2 * math.pi * math.sqrt(7)
    srv = Server(hbm_budget_bytes=1 << 30, max_active=4, max_nodes=8192, block_threads=threads)
    ids = [srv.submit(make_request(env, a, g, seed=500 + i, lvs=LVS, max_iters=iters, rng=rng))
           for i, (a, g) in enumerate(pairs)]
    names = {1: 2, 2: 8, 3: 9, 0: 3}  # oracle status -> server status
    for i, (a, g) in enumerate(pairs):
        res = srv.wait(ids[i], 60000)
        ost, oit, opath, onodes = oracle.rrt_connect_ex(oenv, [a], [g], 500 + i, maxd, LVS, max_iters=iters)
        print(f"request {i}: status {res.status} iterations {res.iterations} nodes {res.tree_nodes} "
              f"path {res.path_len}; oracle {(ost, oit, onodes, len(opath))}", flush=True)
        assert (res.status, res.iterations, res.tree_nodes) == (names[ost], oit, onodes)
        assert np.array_equal(srv.path(ids[i]), opath)
    srv.close()
