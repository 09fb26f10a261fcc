"""Served plans whose solution goes through what several waves of the slice
kernel wrote: chains of more than 64 intermediate states, trees beyond the nodes
kept in LDS (256 each) and solutions beyond the rows returned in place (128).
The oracle's sizes are asserted, so a case that stops reaching them fails."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NAMES = {1: 2, 2: 8, 3: 9, 0: 3}  # oracle status -> server status


@pytest.mark.parametrize("rng,iters,lvs,inter,nodes,length",
                         [(0.0, 300, 0.02, True, 512, 1000), (0.0, 300, 0.01, True, 512, 2000),
                          (0.3, 1500, 0.01, False, 512, 30), (0.02, 400, 0.01, False, 512, 400)])
@pytest.mark.parametrize("threads", [512, 1024])
def test_served_equals_oracle(gpu, oracle, rng, iters, lvs, inter, nodes, length, threads):
    from ompl_amd.serve import Server, make_request

    s, b = gpu.workload.obstacles(1041, 20, 20)
    env, oenv = gpu.Env(s, b), oracle.OracleEnv(s, b)
    ok = [q for q in gpu.workload.configs(1042, 3000) if oracle.state_valid(oenv, q.astype(np.float32))]
    pairs = [(ok[2 * i], ok[2 * i + 1]) for i in range(6)]
    maxd = rng or 0.2 * 2 * math.pi * math.sqrt(7)
    want = [oracle.rrt_connect_ex(oenv, [a], [g], 500 + i, maxd, lvs, max_iters=iters, intermediate=inter)
            for i, (a, g) in enumerate(pairs)]
    assert max(w[3] for w in want) > nodes and max(len(w[2]) for w in want) > length
    srv = Server(hbm_budget_bytes=1 << 30, max_active=6, max_nodes=8192, block_threads=threads)
    ids = [srv.submit(make_request(env, a, g, seed=500 + i, lvs=lvs, max_iters=iters, rng=rng,
                                   intermediate_states=inter)) for i, (a, g) in enumerate(pairs)]
    for rid, (st, it, path, n) in zip(ids, want):
        res = srv.wait(rid, 60000)
        assert (res.status, res.iterations, res.tree_nodes) == (NAMES[st], it, n)
        assert np.array_equal(srv.path(rid), path)
    srv.close()
