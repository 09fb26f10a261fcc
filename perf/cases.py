"""The work that a program has this library do, as measurable cases.

Each case names one public entry point and its sizes; `prepare` makes what the
calling program holds before the call (scene, index, server, device arrays),
`run` is one call.  Scenes, states and edges are the synthetic workloads of
`ompl_amd.workload` (the reference's RNG); nothing depends on anything but the
seed.

Kinds:
  validity    validate_states: is each configuration collision free
  motions     check_motions: discrete motion validation of a batch of edges
  last_valid  check_motions_last_valid: the sequential lastValid overload
  knn         NearestNeighborsGPU.knn_dev: k nearest of a batch of queries
  radius      ompl_amd_nn_radius_dev: all within the RRT* radius, into the
              caller's arrays
  prm         ompl_amd_prm_build and its getters: a whole batch roadmap,
              fetched into the caller's arrays
  sample      sample_valid: valid states for a batch of samplers
  serve       a burst of RRT-Connect requests through the planning server
"""
import ctypes as C
import math

import numpy as np
import torch

import ompl_amd as oa
from ompl_amd import serve
from ompl_amd._lib import PrmStats
from ompl_amd.nn import METRIC_L2, METRIC_SE3, NearestNeighborsGPU
from ompl_amd.sampler import sample_valid

DOF = 7
LVS = 0.01  # longest valid segment, radians
STREAMS = 256  # generators a roadmap's samples come from
PI = math.pi


def listed():
    return [
        # one planner's or a few planners' candidate edges at once: latency and launches count
        {"name": "motions_61_dense", "kind": "motions", "n": 61, "spheres": 128, "boxes": 128, "mu": -1.0,
         "counts": False, "tuned": False},
        # nearest neighbours of 64 planners' samples in a tree of a few thousand states
        {"name": "knn_5k_64q_k10", "kind": "knn", "metric": "l2", "dim": 7, "n": 5000, "nq": 64, "k": 10},
        # a batch of states as a sampler or roadmap hands them over, FP32
        {"name": "validity_65k_64obs", "kind": "validity", "n": 65536, "spheres": 64, "boxes": 0, "f64": False},
        # uneven motions in a crowded scene, most of them colliding at s2; the program tuned its scene once
        {"name": "motions_16k_dense", "kind": "motions", "n": 16384, "spheres": 128, "boxes": 128, "mu": -1.0,
         "counts": False, "tuned": True},
        # long, mostly valid motions in an open scene, with the exact checked counts (benchmark logs)
        {"name": "motions_16k_sparse", "kind": "motions", "n": 16384, "spheres": 16, "boxes": 16, "mu": -0.5,
         "counts": True, "tuned": False},
        # lastValid fractions of tree extensions, an odd batch
        {"name": "last_valid_4099", "kind": "last_valid", "n": 4099, "spheres": 32, "boxes": 16, "mu": -1.0},
        # roadmap neighbours: 4,096 new states in 100,000
        {"name": "knn_100k_4096q_k10", "kind": "knn", "metric": "l2", "dim": 7, "n": 100_000, "nq": 4096, "k": 10},
        # rigid-body planning at scale
        {"name": "knn_se3_1m_65k_k16", "kind": "knn", "metric": "se3", "dim": 7, "n": 1_000_000, "nq": 65536,
         "k": 16},
        # RRT* rewiring neighbourhoods at scale
        {"name": "radius_se3_1m_65k", "kind": "radius", "n": 1_000_000, "nq": 65536},
        # a whole PRM roadmap
        {"name": "prm_200k", "kind": "prm", "samples": 200_000, "spheres": 64, "boxes": 0, "k": 10, "kstar": False},
        # valid states for 256 samplers where only one draw in eighty is valid
        {"name": "sample_valid_256x64", "kind": "sample", "streams": 256, "calls": 64, "spheres": 128, "boxes": 128},
        # a burst of planning requests over several scenes
        {"name": "serve_64_requests", "kind": "serve", "requests": 64, "envs": 8, "obstacles": 128},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["validity", "motions", "motions", "last_valid", "knn", "knn", "radius", "prm", "sample",
                       "serve"])
    scene = {"spheres": _log(rng, 8, 128), "boxes": _log(rng, 8, 128)}
    if kind == "validity":
        return {"kind": kind, "n": _log(rng, 64, 65536), **scene, "f64": rng.random() < 0.5}
    if kind == "motions":
        return {"kind": kind, "n": _log(rng, 16, 16384), **scene, "mu": rng.choice([-1.0, -0.5]),
                "counts": rng.random() < 0.5, "tuned": False}
    if kind == "last_valid":
        return {"kind": kind, "n": _log(rng, 16, 16384), **scene, "mu": rng.choice([-1.0, -0.5])}
    if kind == "knn":
        if rng.random() < 0.5:
            return {"kind": kind, "metric": "l2", "dim": rng.choice([2, 3, 6, 7]), "n": _log(rng, 500, 150_000),
                    "nq": _log(rng, 1, 16384), "k": rng.choice([1, 5, 10, 16, 24])}
        return {"kind": kind, "metric": "se3", "dim": 7, "n": _log(rng, 2000, 1_000_000), "nq": _log(rng, 1, 65536),
                "k": rng.choice([1, 10, 16])}
    if kind == "radius":
        return {"kind": kind, "n": _log(rng, 2000, 1_000_000), "nq": _log(rng, 16, 65536)}
    if kind == "prm":
        return {"kind": kind, "samples": _log(rng, 2000, 100_000), "spheres": rng.randint(16, 64),
                "boxes": rng.randint(0, 8), "k": rng.choice([5, 10, 15]), "kstar": rng.random() < 0.25}
    if kind == "sample":
        return {"kind": kind, "streams": _log(rng, 16, 256), "calls": _log(rng, 4, 64), **scene}
    return {"kind": kind, "requests": _log(rng, 4, 64), "envs": rng.randint(1, 8), "obstacles": _log(rng, 16, 128)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _u32(seed, salt=0):
    return (int(seed) * 2654435761 + 977 * salt + 12345) & 0x7FFFFFFF


def _scene(case, seed):
    return oa.workload.obstacles(_u32(seed, 1), case["spheres"], case["boxes"])


def _edges(case, seed):
    a, b = oa.workload.edges(_u32(seed, 2), case["n"], case["mu"])
    return torch.from_numpy(a.T.copy()).cuda(), torch.from_numpy(b.T.copy()).cuda()


def _points(case, seed):
    """(database, queries) as FP32 rows on the GPU, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(_u32(seed, 3))
    rows = case["n"] + case["nq"]
    if case["kind"] == "radius" or case["metric"] == "se3":
        x = torch.rand(rows, 3, generator=g, device="cuda") * 20.0 - 10.0
        q = torch.randn(rows, 4, generator=g, device="cuda", dtype=torch.float64)
        q = (q / q.norm(dim=1, keepdim=True)).float()
        p = torch.cat([x, q], 1)
    else:
        p = (torch.rand(rows, case["dim"], generator=g, device="cuda") * 2.0 - 1.0) * PI
    return p[:case["n"]].contiguous(), p[case["n"]:].contiguous()


def _rrtstar_radius(n):
    """RRT*'s radius at n states of SE(3) in a 20 x 20 x 20 box."""
    return float(np.float32(oa.rrtstar_radius(6, 8000.0 * PI ** 2, n)))


def _requests(case, seed):
    """Scenes of 16 .. `obstacles` spheres and boxes with valid starts and goals."""
    rng = np.random.default_rng(_u32(seed, 4))
    envs, valid = [], []
    for e in range(case["envs"]):
        n = int(round(math.exp(rng.uniform(math.log(16), math.log(max(case["obstacles"], 17))))))
        while True:
            s, b = oa.workload.obstacles(_u32(seed, 100 + e), n - n // 2, n // 2)
            env = oa.Env(s, b)
            q = oa.workload.configs(_u32(seed, 200 + e), 1024)
            ok = q[oa.validate_states(env, torch.from_numpy(q.T.copy()).cuda()).cpu().numpy() == 1]
            if len(ok) >= 2:
                break
            n = n // 2
        envs.append(env)
        valid.append(ok)
    reqs = []
    for i in range(case["requests"]):
        k = i % case["envs"]
        a, b = valid[k][rng.integers(len(valid[k]))], valid[k][rng.integers(len(valid[k]))]
        reqs.append(serve.make_request(envs[k], a, b, seed=_u32(seed, 300 + i), lvs=LVS, max_iters=2000))
    return envs, reqs


def prepare(case, seed):
    oa.init(0)
    kind = case["kind"]
    st = {"case": case}
    if kind == "validity":
        st["env"] = oa.Env(*_scene(case, seed))
        q = torch.from_numpy(oa.workload.configs(_u32(seed, 5), case["n"]).T.copy()).cuda()
        st["q"] = q if case["f64"] else q.float()
    elif kind in ("motions", "last_valid"):
        st["env"] = oa.Env(*_scene(case, seed))
        st["a"], st["b"] = _edges(case, seed)
        if case.get("tuned"):
            st["env"].autotune(st["a"], st["b"], LVS, reps=4)
    elif kind in ("knn", "radius"):
        db, st["q"] = _points(case, seed)
        se3 = kind == "radius" or case["metric"] == "se3"
        st["nn"] = NearestNeighborsGPU(METRIC_SE3 if se3 else METRIC_L2, 7 if se3 else case["dim"])
        st["nn"].add(db)
        if kind == "radius":
            nq, cap = case["nq"], 48 * case["nq"] + 256
            st["r"] = _rrtstar_radius(case["n"])
            st["off"] = torch.zeros(nq + 1, dtype=torch.int64, device="cuda")
            st["idx"] = torch.zeros(cap, dtype=torch.int32, device="cuda")
            st["dist"] = torch.zeros(cap, dtype=torch.float32, device="cuda")
    elif kind == "prm":
        st["env"] = oa.Env(*_scene(case, seed))
        st["seed"] = _u32(seed, 6)
        n = -(-case["samples"] // STREAMS) * STREAMS  # samples are dealt evenly to the generators
        ne = n * (case["k"] if not case["kstar"] else 40)
        st["out"] = {"nodes": np.zeros((n, DOF)), "sample": np.zeros(n, np.int32), "u": np.zeros(ne, np.int32),
                     "v": np.zeros(ne, np.int32), "valid": np.zeros(ne, np.uint8), "label": np.zeros(n, np.int32),
                     "off": np.zeros(n + 1, np.int64), "adj": np.zeros(2 * ne, np.int32)}
    elif kind == "sample":
        st["env"] = oa.Env(*_scene(case, seed))
        st["seeds"] = np.arange(case["streams"], dtype=np.uint32) + np.uint32(_u32(seed, 7))
    else:
        st["envs"], st["reqs"] = _requests(case, seed)
        st["server"] = serve.Server(hbm_budget_bytes=1 << 30, max_active=256, max_nodes=4096)
        st["paths"] = np.zeros((case["requests"], 512, DOF))
    return st


def _at(a):
    return C.c_void_p(a.data_ptr()) if torch.is_tensor(a) else a.ctypes.data_as(C.c_void_p)


def _roadmap(st, case):
    """A roadmap into the caller's arrays (room for every sample a milestone)."""
    h, s, o = C.c_void_p(), PrmStats(), st["out"]
    oa.call("ompl_amd_prm_build", st["env"].handle, st["seed"], STREAMS, case["samples"], case["k"], LVS, 1,
            2 if case["kstar"] else 0, C.byref(h), C.byref(s))
    try:
        oa.call("ompl_amd_prm_milestones", h, _at(o["nodes"]), _at(o["sample"]), len(o["nodes"]))
        oa.call("ompl_amd_prm_edges", h, _at(o["u"]), _at(o["v"]), _at(o["valid"]), len(o["u"]))
        oa.call("ompl_amd_prm_components", h, _at(o["label"]), len(o["label"]))
        oa.call("ompl_amd_prm_graph", h, _at(o["off"]), _at(o["adj"]), len(o["adj"]))
    finally:
        oa.call("ompl_amd_prm_destroy", h)
    counts = np.array([s.samples, s.milestones, s.candidate_edges, s.valid_edges, s.components, s.k], np.int64)
    return [counts, o["nodes"], o["sample"], o["u"], o["v"], o["valid"], o["label"], o["off"], o["adj"]]


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "validity":
        return oa.validate_states(st["env"], st["q"])
    if kind == "motions":
        return oa.check_motions(st["env"], st["a"], st["b"], LVS, exact_count=case["counts"])
    if kind == "last_valid":
        return oa.check_motions_last_valid(st["env"], st["a"], st["b"], LVS)
    if kind == "knn":
        return st["nn"].knn_dev(st["q"], case["k"])
    if kind == "radius":
        total = C.c_int64()
        oa.call("ompl_amd_nn_radius_dev", st["nn"].handle, _at(st["q"]), case["nq"], st["r"], _at(st["off"]),
                _at(st["idx"]), _at(st["dist"]), st["idx"].numel(), C.byref(total),
                C.c_void_p(torch.cuda.current_stream().cuda_stream))
        return [total.value, st["off"], st["idx"], st["dist"]]
    if kind == "prm":
        return _roadmap(st, case)
    if kind == "sample":
        return sample_valid(st["env"], st["seeds"], case["calls"])
    srv = st["server"]
    ids = [srv.submit(r) for r in st["reqs"]]
    res = [srv.wait(i) for i in ids]
    for k, i in enumerate(ids):
        p = srv.path(i)
        st["paths"][k, :len(p)] = p
        srv.release(i)
    status = np.array([[r.status, r.iterations, r.path_len, r.tree_nodes, r.motion_checks] for r in res], np.int64)
    return [status, st["paths"]]


# ---------------------------------------------------------------------------
# work that the path cannot do without
# ---------------------------------------------------------------------------
FK = oa.FK_FLOPS  # forward kinematics of one state


def work(case):
    """Inputs read once, outputs written once; operations: the forward
    kinematics of every state that has to be looked at (for motions one state
    per edge; long valid motions need more), and for neighbours the distances
    of the results."""
    kind = case["kind"]
    if kind == "validity":
        n = case["n"]
        return {"bytes": n * (DOF * (8 if case["f64"] else 4) + 1), "flops": n * FK}
    if kind in ("motions", "last_valid"):
        n = case["n"]
        out = 9 if kind == "last_valid" else (5 if case["counts"] else 1)
        return {"bytes": n * (2 * DOF * 8 + out), "flops": n * FK}
    if kind == "knn":
        return {"bytes": (case["n"] + case["nq"]) * case["dim"] * 4 + case["nq"] * case["k"] * 8,
                "flops": case["nq"] * case["k"] * 20}
    if kind == "radius":
        return {"bytes": (case["n"] + case["nq"]) * 28 + case["nq"] * 8 * 10 + 8 * case["nq"],
                "flops": case["nq"] * 10 * 20}
    if kind == "prm":
        n = case["samples"]
        return {"bytes": n * DOF * 8 * 2 + n * case["k"] * 16, "flops": n * FK * (1 + case["k"])}
    if kind == "sample":
        n = case["streams"] * case["calls"]
        return {"bytes": n * (DOF * 8 + 5), "flops": n * FK}
    return {"bytes": case["requests"] * 40 * DOF * 8, "flops": case["requests"] * 1000 * FK}


# ---------------------------------------------------------------------------
# 64-bit values
# ---------------------------------------------------------------------------
def _dist64(q, p, se3):
    """All distances of rows q to rows p."""
    if not se3:
        d2 = torch.zeros(q.shape[0], p.shape[0], dtype=torch.float64, device=q.device)
        for j in range(q.shape[1]):
            d2 += (q[:, j:j + 1] - p[None, :, j]) ** 2
        return d2.sqrt_()
    dt = torch.zeros(q.shape[0], p.shape[0], dtype=torch.float64, device=q.device)
    for j in range(3):
        dt += (q[:, j:j + 1] - p[None, :, j]) ** 2
    dot = (q[:, 3:] @ p[:, 3:].T.contiguous()).abs_()
    return dt.sqrt_() + torch.where(dot > 1.0, 0.0, dot.clamp_(max=1.0).acos_())


def _nearest64(db, qs, k, se3):
    """The k smallest distances per query: queries in order of their first
    coordinate, each block against the points within a window around it; a
    block whose k-th distance reaches past its window is done again with a wider one."""
    db, qs = db.double(), qs.double()
    db = db[db[:, 0].argsort()]
    order = qs[:, 0].argsort()
    first = db[:, 0].contiguous()
    out = torch.full((qs.shape[0], k), float("inf"), dtype=torch.float64, device=qs.device)
    block = max(1, min(512, (1 << 27) // max(1, db.shape[0])))
    width = 2.5 if se3 else 2.2
    for at in range(0, qs.shape[0], block):
        rows = order[at:at + block]
        q = qs[rows]
        w = width
        while True:
            lo = int(torch.searchsorted(first, q[0, 0] - w))
            hi = int(torch.searchsorted(first, q[-1, 0] + w, right=True))
            m = min(k, hi - lo)
            whole = lo == 0 and hi == db.shape[0]
            if m == k or whole:
                d = _dist64(q, db[lo:hi], se3).topk(m, dim=1, largest=False, sorted=True).values
                if whole or float(d[:, -1].max()) < w:
                    out[rows, :m] = d
                    break
            w *= 2.0
    return out


def exact(case, seed):
    if case["kind"] == "knn":
        db, q = _points(case, seed)
        return [None, _nearest64(db, q, case["k"], case["metric"] == "se3")]
    # radius: which points lie on the very edge is decided in 32 bits, so the
    # 64-bit list can have other members; the rest are truth values, counts,
    # fractions of whole numbers and copies of inputs
    return None
