"""What this framework is timed on: the calls its users make, over their range.

Every case is one kind of call with its sizes; listed() holds the usual
ones and draw() others of the same kinds between their smallest and largest
sizes.  Meshes, contexts and servers are made once per process, as a program
keeps them resident; poses, boxes, deformed vertices and trajectories come
from the seed.
"""
import math

import numpy as np
import torch

import fcl_amd as F
from fcl_amd import workloads

DEV = "cuda:0"

# OBB test 315 operations on two node records, triangle test 923; RSS bound
# 380, triangle distance 900; one GJK pass 330, one EPA pass 460.
OBB, TRI, RSS, TDIST, GJK, EPA = 315, 923, 380, 900, 330, 460


ROOM = 2600  # contact pairs per query that an exhaustive batch has room for


# ------------------------------------------------------------------- cases
def listed():
    return [
        # a program moved over from FCL unchanged: collide() per pose, one call
        # after the other, with the default request (first contact)
        {"name": "collide_calls", "kind": "collide_calls", "calls": 16, "tris": 2420, "cap": 1,
         "contact": False},
        # the same program's distance() calls, with nearest points
        {"name": "distance_calls", "kind": "distance_calls", "calls": 4, "tris": 2420},
        # a planner's batch of poses: does the part hit, and which triangles
        {"name": "first_contact", "kind": "collide", "queries": 10000, "tris": 2420, "cap": 1,
         "contact": False, "stats": False},
        # a simulator's batch: contact points, normals and depths per pose
        {"name": "contacts", "kind": "collide", "queries": 4096, "tris": 2420, "cap": 8,
         "contact": True, "stats": False},
        # every contact pair of many poses over mesh pairs of uneven sizes
        # (500 to 200,000 triangles), grouped by query: the headline workload
        {"name": "exhaustive", "kind": "exhaustive", "queries": 60000, "pairs": 16,
         "cap": 100000, "stats": False},
        # trajectories of a 20-link robot against a 500k-triangle scene,
        # booleans only, poses already in device memory
        {"name": "scene_bool", "kind": "scene_bool", "waypoints": 2048, "trajectories": 4,
         "grid": 400, "boxes": 15133},
        # the same robot and scene behind the request loop: a backlog of
        # requests of 64 to 4096 waypoints from host memory
        {"name": "serving", "kind": "serving", "requests": 48, "grid": 400, "boxes": 15133},
        # clearance of a batch of poses: distance, nearest points, triangles
        {"name": "distance", "kind": "distance", "queries": 10000, "tris": 20480},
        # primitive pairs with contact geometry (GJK / EPA and closed forms)
        {"name": "primitives", "kind": "primitives", "queries": 1000000, "cap": 1,
         "contact": True},
        # primitive links against a mesh, first contact, no geometry
        {"name": "mesh_shape", "kind": "mesh_shape", "queries": 100000, "tris": 20480, "cap": 1,
         "contact": False},
        # one frame of a deforming mesh: refit its hierarchy, then collide
        {"name": "refit_frame", "kind": "refit", "queries": 1000, "tris": 20480,
         "bottomup": True},
        # candidate pairs of a scene's objects
        {"name": "broadphase", "kind": "broadphase", "objects": 10000, "groups": False},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["collide_calls", "distance_calls", "collide", "collide", "collide",
                       "exhaustive", "exhaustive", "scene_bool", "serving", "distance",
                       "primitives", "mesh_shape", "mesh_shape", "refit", "broadphase"])
    c = {"kind": kind}
    if kind == "collide_calls":
        c.update(calls=rng.randint(4, 32), tris=_log(rng, 500, 50000),
                 cap=rng.choice([1, 1, 8, 1000]), contact=rng.random() < 0.4)
    elif kind == "distance_calls":
        c.update(calls=rng.randint(2, 6), tris=_log(rng, 500, 20480))
    elif kind == "collide":
        c.update(queries=_log(rng, 64, 20000), tris=_log(rng, 500, 50000),
                 cap=rng.choice([1, 1, 4, 16]), contact=rng.random() < 0.5,
                 stats=rng.random() < 0.3)
    elif kind == "exhaustive":
        c.update(queries=_log(rng, 1000, 60000), pairs=rng.randint(4, 16),
                 cap=rng.choice([100000, 100000, 500]), stats=rng.random() < 0.3)
    elif kind == "scene_bool":
        c.update(waypoints=_log(rng, 64, 4096), trajectories=rng.randint(1, 4),
                 grid=rng.choice([100, 200, 400]), boxes=rng.choice([500, 4000, 15133]))
    elif kind == "serving":
        c.update(requests=rng.randint(8, 48), grid=rng.choice([200, 400]),
                 boxes=rng.choice([4000, 15133]))
    elif kind == "distance":
        c.update(queries=_log(rng, 64, 10000), tris=_log(rng, 500, 20480))
    elif kind == "primitives":
        c.update(queries=_log(rng, 1000, 1000000), cap=rng.choice([1, 4]),
                 contact=rng.random() < 0.7)
    elif kind == "mesh_shape":
        c.update(queries=_log(rng, 500, 100000), tris=_log(rng, 500, 50000),
                 cap=rng.choice([1, 1, 4]), contact=rng.random() < 0.4)
    elif kind == "refit":
        c.update(queries=_log(rng, 100, 4000), tris=_log(rng, 500, 50000),
                 bottomup=rng.random() < 0.6)
    else:
        c.update(objects=_log(rng, 50, 50000), groups=rng.random() < 0.3)
    return c


# -------------------------------------------------- resident meshes and handles
_kept = {}


def _keep(key, make):
    if key not in _kept:
        _kept[key] = make()
    return _kept[key]


def _ctx(kind):
    return _keep(("ctx", kind), lambda: F.Context(0))


def _host_mesh(shape, tris, seed):
    return _keep(("host", shape, tris, seed), lambda: workloads.synth_mesh(shape, tris, seed))


def _mesh(kind, shape, tris, seed, bv=F.OBBRSS):
    def make():
        V, T = _host_mesh(shape, tris, seed)
        return _ctx(kind).mesh(V, T, bv)
    return _keep(("mesh", kind, shape, tris, seed, bv), make)


def _robot_scene(case):
    """The scene, its context and the robot's 20 link meshes, resident."""
    def make():
        ctx = F.Context(0)
        scene = ctx.mesh(*workloads.serving_scene(case["grid"], case["boxes"]))
        links = [ctx.mesh(V, T) for V, T in _keep("robot", workloads.serving_robot)]
        return {"ctx": ctx, "scene": scene, "links": np.array(links, np.int32)}
    return _keep(("scene", case["grid"], case["boxes"]), make)


def _server(case):
    r = _robot_scene(case)
    if "server" not in r:
        r["server"] = F.Server(r["ctx"], r["scene"])
    return r


# ------------------------------------------------------------------- inputs
def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _normal(g, *size):
    return torch.randn(size, generator=g, device=DEV, dtype=torch.float64)


def _uniform(g, lo, hi, *size):
    return lo + (hi - lo) * torch.rand(size, generator=g, device=DEV, dtype=torch.float64)


def _rotations(q):
    """Rotation matrices (n, 3, 3) of quaternions (n, 4), scaled to unit length."""
    w, x, y, z = (q / q.norm(dim=1, keepdim=True)).unbind(1)
    return torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                        2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                        2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)],
                       1).reshape(-1, 3, 3)


def _rotate(R, v):
    return (R * v[:, None, :]).sum(2)


def _compose(R1, t1, R2, t2):
    """(R1, t1) after (R2, t2), as (n, 12) poses."""
    R = (R1[:, :, :, None] * R2[:, None, :, :]).sum(2)
    return torch.cat([R.reshape(-1, 9), _rotate(R1, t2) + t1], 1)


def _pose_pairs(g, n, half=None, shell=None):
    """n pairs of poses somewhere in a room: the second body relative to the
    first at a uniform random rotation, its translation uniform in
    [-half, half]^3 or of a length uniform in shell = (lo, hi)."""
    R1, t1 = _rotations(_normal(g, n, 4)), _uniform(g, -3, 3, n, 3)
    R2 = _rotations(_normal(g, n, 4))
    if shell is None:
        t2 = _uniform(g, -half, half, n, 3)
    else:
        d = _normal(g, n, 3)
        t2 = d / d.norm(dim=1, keepdim=True) * _uniform(g, shell[0], shell[1], n, 1)
    tf1 = torch.cat([R1.reshape(-1, 9), t1], 1).contiguous()
    return tf1, _compose(R1, t1, R2, t2).contiguous()


def _trajectory(g, waypoints, links=20, extent=4.0):
    """Poses (waypoints, links, 12): each link starts near a common base over
    the scene and moves by a random walk, turning about an axis of its own."""
    base = torch.cat([_uniform(g, -0.85 * extent, 0.85 * extent, 2), _uniform(g, 0.05, 0.45, 1)])
    t = base + _uniform(g, -0.4, 0.4, links, 3)
    t[:, 2].clamp_(min=-0.05)
    step = 0.01 * _normal(g, waypoints, links, 3)
    step[0] = 0
    t = t + step.cumsum(0)
    R0 = _rotations(_normal(g, links, 4)).repeat(waypoints, 1, 1)
    axis = _normal(g, links, 3)
    axis = (axis / axis.norm(dim=1, keepdim=True)).repeat(waypoints, 1)
    half = 0.5 * (0.02 * _normal(g, waypoints, links)).cumsum(0).reshape(-1, 1)
    turn = _rotations(torch.cat([half.cos(), half.sin() * axis], 1))
    zero = torch.zeros((waypoints * links, 3), device=DEV, dtype=torch.float64)
    out = _compose(turn, zero, R0, zero)
    out[:, 9:] = t.reshape(-1, 3)
    return out.reshape(waypoints, links, 12).contiguous()


def _shapes(g, n):
    """n primitive records in turn over box, sphere, capsule, cylinder and a
    convex of 32 points (dimensions log-uniform in [0.05, 1]), as device
    bytes, and the pool of convex points."""
    kind = torch.randint(0, 5, (n,), generator=g, device=DEV)
    dims = torch.exp(_uniform(g, math.log(0.05), 0.0, n, 3))
    scale = dims[:, 0].clone()
    dims[kind == F.SPHERE, 1:] = 0
    dims[(kind == F.CAPSULE) | (kind == F.CYLINDER), 2] = 0
    dims[kind == F.CONVEX] = 0
    convex = torch.nonzero(kind == F.CONVEX)[:, 0]
    rec = torch.zeros((n, 5), dtype=torch.int64, device=DEV)
    rec[:, 0] = kind
    rec[convex, 0] += 32 << 32
    rec[:, 1:4] = dims.view(torch.int64)
    rec[convex, 4] = 32 * torch.arange(len(convex), device=DEV)
    pool = _normal(g, max(1, len(convex)), 32, 3)
    pool[:len(convex)] *= scale[convex][:, None, None]
    return rec.view(torch.uint8).reshape(-1), pool.reshape(-1, 3)


def _ints(*size):
    return torch.zeros(size, dtype=torch.int32, device=DEV)


def _doubles(*size):
    return torch.zeros(size, dtype=torch.float64, device=DEV)


def _longs(*size):
    return torch.zeros(size, dtype=torch.int64, device=DEV)


def prepare(case, seed):
    kind, g = case["kind"], _generator(seed)
    s = dict(case)
    if kind in ("collide_calls", "distance_calls"):
        bv = F.OBBRSS if kind == "collide_calls" else F.RSS
        s["ctx"] = _ctx(kind)
        s["meshes"] = [_mesh(kind, 0, case["tris"], i + 1, bv) for i in range(2)]
        # radii up to 1.15: poses that overlap about half the time, or (for
        # distance) are apart
        tf = _pose_pairs(g, case["calls"], half=1.6) if kind == "collide_calls" else \
            _pose_pairs(g, case["calls"], shell=(2.05, 4.0))
        s["tf1"], s["tf2"] = (t.cpu().numpy() for t in tf)
    elif kind == "collide":
        n, cap = case["queries"], case["cap"]
        s["ctx"] = _ctx(kind)
        s["qm"] = torch.tensor([_mesh(kind, 0, case["tris"], 1), _mesh(kind, 0, case["tris"], 2)],
                               dtype=torch.int32, device=DEV).repeat(n, 1)
        s["tf1"], s["tf2"] = _pose_pairs(g, n, half=1.6)
        s["counts"], s["pairs"], s["num"] = _ints(n), _ints(n * cap, 3), _longs(1)
        s["geometry"] = ((_doubles(n * cap, 3), _doubles(n * cap, 3), _doubles(n * cap))
                         if case["contact"] else None)
        s["tests"] = (_longs(n), _longs(n)) if case["stats"] else (None, None)
    elif kind == "exhaustive":
        s.update(_prepare_exhaustive(case, g))
    elif kind == "scene_bool":
        r = _robot_scene(case)
        tf2 = torch.cat([_trajectory(g, case["waypoints"]).reshape(-1, 12)
                         for _ in range(case["trajectories"])]).contiguous()
        n = len(tf2)
        link = torch.from_numpy(r["links"]).to(DEV).repeat(n // len(r["links"]))
        s["ctx"] = r["ctx"]
        s["qm"] = torch.stack([torch.full_like(link, r["scene"]), link], 1).contiguous()
        s["tf1"] = torch.eye(4, 3, device=DEV, dtype=torch.float64).reshape(1, 12).repeat(n, 1)
        s["tf2"], s["counts"], s["num"] = tf2, _ints(n), _longs(1)
    elif kind == "serving":
        r = _server(case)
        requests = []
        for i in torch.randperm(case["requests"], generator=g, device=DEV).tolist():
            waypoints = int(64 * 64 ** ((i + 0.5) / case["requests"]))  # log-uniform, 64 to 4096
            poses = torch.empty((waypoints, len(r["links"]), 12), dtype=torch.float64,
                                pin_memory=True)
            poses.copy_(_trajectory(g, waypoints))
            requests.append((r["links"], poses.numpy()))
        s["server"], s["requests"] = r["server"], requests
        s["arrivals"] = np.zeros(len(requests))
    elif kind == "distance":
        n = case["queries"]
        s["ctx"] = _ctx(kind)
        s["qm"] = torch.tensor([_mesh(kind, 0, case["tris"], i + 1, F.RSS) for i in range(2)],
                               dtype=torch.int32, device=DEV).repeat(n, 1)
        s["tf1"], s["tf2"] = _pose_pairs(g, n, shell=(1.9, 4.0))
        s["distance"], s["points"], s["ids"] = _doubles(n), _doubles(n, 6), _ints(n, 2)
    elif kind == "primitives":
        n, cap = case["queries"], case["cap"]
        s["ctx"] = _ctx(kind)
        s["shapes"], s["pool"] = _shapes(g, 2 * n)
        s["pair_shapes"] = torch.arange(2 * n, dtype=torch.int32, device=DEV).reshape(n, 2)
        s["tf1"], s["tf2"] = _pose_pairs(g, n, half=1.0)
        s["counts"] = _ints(n)
        s["geometry"] = ((_doubles(n * cap, 3), _doubles(n * cap, 3), _doubles(n * cap))
                         if case["contact"] else None)
    elif kind == "mesh_shape":
        n, cap = case["queries"], case["cap"]
        s["ctx"] = _ctx(kind)
        mesh = _mesh(kind, 0, case["tris"], 1)
        s["qm"] = torch.full((n,), mesh, dtype=torch.int32, device=DEV)
        s["shapes"], s["pool"] = _shapes(g, 64)  # a robot's link shapes
        s["qs"] = torch.randint(0, 64, (n,), generator=g, device=DEV).to(torch.int32)
        s["tf1"], s["tf2"] = _pose_pairs(g, n, shell=(0.8, 1.6))
        s["counts"], s["primitives"] = _ints(n), _ints(n * cap)
        s["geometry"] = ((_doubles(n * cap, 3), _doubles(n * cap, 3), _doubles(n * cap))
                         if case["contact"] else None)
    elif kind == "refit":
        n = case["queries"]
        s["ctx"] = _ctx(kind)
        s["mesh"] = _mesh(kind, 0, case["tris"], 1)
        V = torch.from_numpy(_host_mesh(0, case["tris"], 1)[0]).to(DEV)
        wave = _normal(g, 3, 3)
        s["vertices"] = (V + 0.08 * torch.sin(_compose_waves(V, wave))).contiguous()
        s["qm"] = torch.tensor([s["mesh"], _mesh(kind, 0, 2420, 2)], dtype=torch.int32,
                               device=DEV).repeat(n, 1)
        s["tf1"], s["tf2"] = _pose_pairs(g, n, half=1.6)
        s["counts"], s["pairs"], s["num"] = _ints(n), _ints(n, 3), _longs(1)
        s["cap"], s["geometry"], s["tests"] = 1, None, (_longs(n), _longs(n))
    else:
        n = case["objects"]
        # boxes of sides up to a tenth of their spacing region: about two
        # overlaps per object
        centre = _uniform(g, -0.5, 0.5, n, 3) * n ** (1 / 3)
        size = torch.exp(_uniform(g, math.log(0.1), math.log(1.0), n, 3))
        s["ctx"] = _ctx(kind)
        s["aabbs"] = torch.cat([centre - size, centre + size], 1).contiguous()
        s["pairs"], s["num"] = _ints(16 * n, 2), _longs(1)
        s["group"] = torch.randint(0, 2, (n,), generator=g, device=DEV).to(torch.int32) \
            if case["groups"] else None
    return s


def _compose_waves(V, wave):
    return (V[:, None, :] * wave[None]).sum(2) * 3.0


def _prepare_exhaustive(case, g):
    """Mesh pairs of 500 to 200,000 triangles (log-uniform, icospheres and
    terrains), the queries split over them unevenly (Dirichlet(1))."""
    rng = np.random.default_rng(0x5EED)
    ids = []
    for i in range(2 * case["pairs"]):
        shape, tris = int(rng.integers(0, 2)), int(math.exp(rng.uniform(math.log(500),
                                                                        math.log(200000))))
        ids.append(_mesh("exhaustive", shape, tris, i + 1))
    n = case["queries"]
    counts = workloads.dirichlet_split(n, case["pairs"], rng)
    qm = np.repeat(np.array(ids, np.int32).reshape(-1, 2), counts, axis=0)
    tf1, tf2 = _pose_pairs(g, n, half=2.2)
    return {"ctx": _ctx("exhaustive"), "qm": torch.from_numpy(qm).to(DEV), "tf1": tf1,
            "tf2": tf2, "counts": _ints(n), "pairs": _ints(ROOM * n + 500000, 3),
            "num": _longs(1), "sorted": _longs(ROOM * n + 500000) - 1,
            "tests": (_longs(n), _longs(n)) if case["stats"] else (None, None)}


# --------------------------------------------------------------------- calls
def run(s):
    return _RUN[s["kind"]](s)


def _run_collide_calls(s):
    """Per call: the contact pairs and the traversal's test counts."""
    call = s["ctx"].collide_contact if s["contact"] else s["ctx"].collide
    rows = [np.full((s["calls"], s["cap"], 2), -1, np.int32)]
    if s["contact"]:
        rows += [np.zeros((s["calls"], s["cap"]) + size) for size in ((3,), (3,), ())]
    tests = np.zeros((s["calls"], 2), np.int64)
    for q in range(s["calls"]):
        *found, tests[q] = call(s["meshes"][0], s["tf1"][q], s["meshes"][1], s["tf2"][q],
                                cap=s["cap"])
        for r, f in zip(rows, found):
            r[q, :len(f)] = f
    return [rows, tests]


def _run_distance_calls(s):
    out = [s["ctx"].distance(s["meshes"][0], s["tf1"][q], s["meshes"][1], s["tf2"][q])
           for q in range(s["calls"])]
    return {"distance": np.array([o[0] for o in out]), "points": np.stack([o[1] for o in out]),
            "ids": np.stack([o[2] for o in out]), "tests": np.stack([o[3] for o in out])}


def _run_collide(s):
    """Contacts in query order; the rows of a query keep the order of its
    contacts, unused rows carry the query number n."""
    n = s["queries"]
    s["pairs"].fill_(n)
    s["ctx"].collide_batch_async(s["qm"], s["tf1"], s["tf2"], s["cap"], s["counts"], s["pairs"],
                                 s["num"], engine=F.ENGINE_FAST, bv_tests=s["tests"][0],
                                 leaf_tests=s["tests"][1], contact=s["geometry"],
                                 stream=torch.cuda.current_stream().cuda_stream)
    rows = [s["pairs"]] + list(s["geometry"] or ())
    if s["cap"] == 1:  # at most one row per query: straight to its place
        at = s["pairs"][:, 0].long()
        rows = [r.new_zeros((n + 1,) + r.shape[1:]).index_copy_(0, at, r) for r in rows]
    else:
        order = torch.argsort(s["pairs"][:, 0], stable=True)
        rows = [r[order] for r in rows]
    return [s["counts"], s["num"], rows, list(s["tests"])]


def _run_exhaustive(s):
    """Contact pairs sorted by query, then triangles (the engine gives them
    in no particular order), in a list that has room for more."""
    stream = torch.cuda.current_stream().cuda_stream
    s["ctx"].collide_batch_async(s["qm"], s["tf1"], s["tf2"], s["cap"], s["counts"], s["pairs"],
                                 s["num"], engine=F.ENGINE_FAST, bv_tests=s["tests"][0],
                                 leaf_tests=s["tests"][1], stream=stream)
    s["ctx"].sync(stream)
    k = int(s["num"].item())
    rec = s["pairs"][:k]
    keys = (rec[:, 0].long() << 42) | (rec[:, 1].long() << 21) | rec[:, 2].long()
    s["sorted"][:k] = torch.sort(keys)[0]
    return [s["counts"], s["num"], s["sorted"], list(s["tests"])]


def _run_scene_bool(s):
    s["ctx"].collide_batch_async(s["qm"], s["tf1"], s["tf2"], 1, s["counts"], None, s["num"],
                                 engine=F.ENGINE_BOOL,
                                 stream=torch.cuda.current_stream().cuda_stream)
    return s["counts"]


def _run_serving(s):
    results, _, _ = s["server"].replay(s["requests"], s["arrivals"])
    return np.concatenate([r.reshape(-1) for r in results])


def _run_distance(s):
    s["ctx"].distance_batch_async(s["qm"], s["tf1"], s["tf2"], s["distance"], s["points"],
                                  s["ids"], engine=F.ENGINE_FAST,
                                  stream=torch.cuda.current_stream().cuda_stream)
    return {"distance": s["distance"], "points": s["points"], "ids": s["ids"]}


def _run_primitives(s):
    s["ctx"].shape_collide_batch_async(s["shapes"], s["pool"], s["pair_shapes"], s["tf1"],
                                       s["tf2"], s["cap"], s["counts"], contact=s["geometry"],
                                       stream=torch.cuda.current_stream().cuda_stream)
    return [s["counts"], list(s["geometry"] or ())]


def _run_mesh_shape(s):
    s["ctx"].mesh_shape_collide_batch_async(s["qm"], s["shapes"], s["pool"], s["qs"], s["tf1"],
                                            s["tf2"], s["cap"], s["counts"],
                                            primitives=s["primitives"], contact=s["geometry"],
                                            stream=torch.cuda.current_stream().cuda_stream)
    return [s["counts"], s["primitives"], list(s["geometry"] or ())]


def _run_refit(s):
    s["ctx"].mesh_refit(s["mesh"], s["vertices"], bottomup=s["bottomup"],
                        stream=torch.cuda.current_stream().cuda_stream)
    return _run_collide(s)


def _run_broadphase(s):
    s["ctx"].broadphase_pairs_async(s["aabbs"], s["pairs"], s["num"], groups=s["group"],
                                    stream=torch.cuda.current_stream().cuda_stream)
    return [s["pairs"], s["num"]]


_RUN = {"collide_calls": _run_collide_calls, "distance_calls": _run_distance_calls,
        "collide": _run_collide, "exhaustive": _run_exhaustive, "scene_bool": _run_scene_bool,
        "serving": _run_serving, "distance": _run_distance, "primitives": _run_primitives,
        "mesh_shape": _run_mesh_shape, "refit": _run_refit, "broadphase": _run_broadphase}


# ---------------------------------------------------------------- work and limits
def work(case):
    """Inputs and outputs once, and the tests of the reference's recursion
    (their number per query as measured on these inputs)."""
    kind = case["kind"]
    tris = case.get("tris", 0)
    mesh = 128 * 2 * tris + 72 * tris  # a hierarchy's FP64 nodes and its triangles
    if kind == "collide_calls":
        n = case["calls"]
        return {"bytes": n * (192 + 16) + 2 * min(mesh, 20000 * n),
                "flops": n * (290 * OBB + 4.4 * TRI)}
    if kind == "distance_calls":
        n = case["calls"]
        return {"bytes": n * (192 + 80) + 2 * mesh, "flops": n * (2550 * RSS + 175 * TDIST)}
    if kind in ("collide", "refit"):
        n, cap = case["queries"], case.get("cap", 1)
        row = 12 + (56 if case.get("contact") else 0)
        w = {"bytes": n * (8 + 192 + 4 + 0.5 * cap * row) + 2 * mesh,
             "flops": n * ((290 + 30 * (cap - 1)) * OBB + (4.4 + 1.9 * (cap - 1)) * TRI)}
        if kind == "refit":
            w["bytes"] += tris * (12 + 12 + 2 * (128 + 128 + 64 + 64 + 8) + 128)
            w["flops"] += n * 6200 * OBB + 2 * tris * 2000
        return w
    if kind == "exhaustive":
        n = case["queries"]
        contacts = min(1820, case["cap"])
        return {"bytes": n * (8 + 192 + 4 + contacts * (12 + 8)) + 1e8,
                "flops": n * (62000 * OBB + 4100 * TRI)}
    if kind in ("scene_bool", "serving"):
        n = 20 * (case["waypoints"] * case["trajectories"] if kind == "scene_bool"
                  else case["requests"] * 970)
        scene = (2 * case["grid"] ** 2 + 12 * case["boxes"]) * (2 * 64 + 72)
        return {"bytes": n * (8 + 192 + 4) + scene, "flops": n * (374 * OBB + 50 * TRI)}
    if kind == "distance":
        n = case["queries"]
        return {"bytes": n * (8 + 192 + 64) + 2 * mesh, "flops": n * (16300 * RSS + 259 * TDIST)}
    if kind == "primitives":
        n = case["queries"]
        rows = n * 0.26 * 56 if case["contact"] else 0
        return {"bytes": n * (8 + 80 + 192 + 0.4 * 768 + 4) + rows,
                "flops": n * (4.3 * GJK + (2.6 * EPA if case["contact"] else 0))}
    if kind == "mesh_shape":
        n = case["queries"]
        return {"bytes": n * (4 + 4 + 192 + 4 + 4 + (56 if case["contact"] else 0)) + mesh,
                "flops": n * (258 * OBB + 79 * GJK)}
    n = case["objects"]
    return {"bytes": n * 48 + 16 * n * 8, "flops": n * 2 * math.log2(max(n, 2))}


def tolerance(case):
    kind = case["kind"]
    if kind in ("distance_calls", "distance"):
        # 64-bit distances of coordinates near 1: a few hundred roundings;
        # points of nearly parallel features lose some digits more
        return {"rel": 1e-10, "max": 1e-7}
    if kind in ("primitives", "mesh_shape") and case["contact"]:
        # GJK and EPA end at a tolerance of 1e-6 on 64-bit numbers
        return {"rel": 1e-6, "max": 1e-4}
    if kind in ("collide", "collide_calls") and case["contact"]:
        return {"rel": 1e-10, "max": 1e-7}
    return "exact"


# ------------------------------------------------------------------ exact values
def exact(case, seed):
    """distance(): the minimum over all triangle pairs.  (Contact points come
    from the order of the traversal and from iterations that end at their own
    tolerance, and batches of distances take minutes this way: no value.)"""
    if case["kind"] != "distance_calls":
        return None
    g = _generator(seed)
    tf1, tf2 = _pose_pairs(g, case["calls"], shell=(2.05, 4.0))
    tri = []
    for i in range(2):
        V, T = _host_mesh(0, case["tris"], i + 1)
        tri.append(torch.from_numpy(V).to(DEV)[torch.from_numpy(T).to(DEV).long()])
    dist, points = [], []
    for q in range(case["calls"]):
        posed = [(t[:, :, None, :] * p[:9].reshape(3, 3)).sum(3) + p[9:]
                 for t, p in zip(tri, (tf1[q], tf2[q]))]
        d, P, Q = _mesh_distance(*posed)
        dist.append(d)
        points.append(torch.stack([P, Q]))
    touching = min(dist) == 0  # any common point is a nearest one
    return {"distance": torch.tensor(dist, dtype=torch.float64),
            "points": None if touching else torch.stack(points), "ids": None, "tests": None}


def _mesh_distance(A, B):
    """Distance and nearest points of triangle sets (n,3,3) and (m,3,3): pairs
    whose bounding spheres are too far apart are left out."""
    ca, cb = A.mean(1), B.mean(1)
    ra, rb = ((x - c[:, None]).norm(dim=2).amax(1) for x, c in ((A, ca), (B, cb)))
    low = torch.cdist(ca, cb, compute_mode="donot_use_mm_for_euclid_dist")
    near = low.min()
    keep = torch.nonzero(low - ra[:, None] - rb[None] <= near)
    best = None
    for part in keep.split(1 << 18):
        a, b = A[part[:, 0]], B[part[:, 1]]
        d, P, Q = _triangle_distance(a, b)
        i = int(d.argmin())
        if best is None or float(d[i]) < best[0]:
            best = (float(d[i]), P[i], Q[i])
    return best


def _triangle_distance(a, b):
    found = []
    for i in range(3):
        for j in range(3):
            found.append(_segments(a[:, i], a[:, (i + 1) % 3], b[:, j], b[:, (j + 1) % 3]))
    for k in range(3):
        found.append(_onto(a[:, k], b))
        Q, P, ok = _onto(b[:, k], a)
        found.append((P, Q, ok))
        for x, y in ((a, b), (b, a)):
            X, ok = _pierce(x[:, k], x[:, (k + 1) % 3], y)
            found.append((X, X, ok))
    d = torch.stack([torch.where(ok, (P - Q).norm(dim=1), torch.inf) for P, Q, ok in found])
    i = d.argmin(0)
    at = torch.arange(len(i), device=d.device)
    return (d[i, at], torch.stack([f[0] for f in found])[i, at],
            torch.stack([f[1] for f in found])[i, at])


def _dot(u, v):
    return (u * v).sum(1, keepdim=True)


def _segments(p, p1, q, q1):
    """Nearest points of segments pp1 and qq1: the clamped solution of the two
    lines, then each parameter once more for the other's."""
    u, v, w = p1 - p, q1 - q, p - q
    a, b, c, d, e = _dot(u, u), _dot(u, v), _dot(v, v), _dot(u, w), _dot(v, w)
    det = a * c - b * b
    s = torch.where(det > 1e-14 * a * c, (b * e - c * d) / det.clamp(min=1e-300), 0.0).clamp(0, 1)
    t = ((b * s + e) / c).clamp(0, 1)
    s = ((b * t - d) / a).clamp(0, 1)
    return p + s * u, q + t * v, torch.ones(len(p), dtype=torch.bool, device=p.device)


def _inside(X, t):
    n = torch.linalg.cross(t[:, 1] - t[:, 0], t[:, 2] - t[:, 0])
    ok = torch.ones(len(X), dtype=torch.bool, device=X.device)
    for k in range(3):
        edge = t[:, (k + 1) % 3] - t[:, k]
        ok &= _dot(torch.linalg.cross(edge, X - t[:, k]), n)[:, 0] >= 0
    return ok


def _onto(X, t):
    """The foot of X on the triangle's plane, where it lies in the triangle."""
    n = torch.linalg.cross(t[:, 1] - t[:, 0], t[:, 2] - t[:, 0])
    n = n / n.norm(dim=1, keepdim=True)
    Y = X - _dot(X - t[:, 0], n) * n
    return X, Y, _inside(Y, t)


def _pierce(p, q, t):
    """Where segment pq goes through the triangle."""
    n = torch.linalg.cross(t[:, 1] - t[:, 0], t[:, 2] - t[:, 0])
    x, y = _dot(p - t[:, 0], n), _dot(q - t[:, 0], n)
    X = p + (x / (x - y)) * (q - p)
    return X, (x * y < 0)[:, 0] & _inside(X, t)
