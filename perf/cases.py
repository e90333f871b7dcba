"""Cases for timing the contact-detection path, as a program uses it: the
plug-in point and the filter called on their own, the discrete and the
continuous phase, whole steps (resident inputs replayed from a graph, or body
states in and contacts out), the solver, the broad phase, and the learned
gate's training.

A case names its form (``op``) and its sizes; ``prepare`` builds the context a
program would hold (trees, bodies, pair list, weights) and its result buffers
from a seed, ``run`` is one pass through the public calls.  Results are read
through the C interface into the program's own buffers, as a C++ caller does;
the buffers have room to spare, and rows beyond a pass's count stay zero.
Bodies share a pool of trees, as instanced meshes do, so that large scenes are
made quickly.
"""
import ctypes
import math

import numpy as np

import delta2_amd as d2
from delta2_amd import learned, scenes

DT = scenes.DT
GRAVITY = (0.0, 0.0, -9.8)


def listed():
    return [
        # the plug-in point as a caller's traversal first meets it: one early level of one body pair
        {"name": "bucket_few", "op": "bucket", "mesh": "sphere2", "n": 13},
        # the same call on a deep level of two large meshes
        {"name": "bucket_level", "op": "bucket", "mesh": "sphere3", "n": 6007},
        # the contact filter alone, on one touching pair's contacts
        {"name": "filter_pair", "op": "filter", "n": 701, "patch": 0.45},
        # a small interactive scene: 100 bodies, the whole step replayed from a graph, contacts read back
        {"name": "step_100", "op": "step", "bodies": 100, "mesh": "sphere2", "pool": 100, "density": 0.1,
         "fp32": True, "graph": True, "gate": False},
        # the reference path itself in double precision: discrete contacts of tumbling hulls and spheres
        {"name": "narrow_fp64", "op": "narrow", "bodies": 311, "mesh": "mix2", "pool": 48, "density": 0.12,
         "fp32": False, "graph": False, "gate": False},
        # continuous detection with the step rule over a mid-size scene, the learned gate proposing pairs
        {"name": "ccd_gate", "op": "ccd", "bodies": 1501, "mesh": "sphere2", "pool": 96, "density": 0.1,
         "fp32": True, "graph": False, "gate": True},
        # the 4096-body workload's shape: spheres and hulls, mostly apart, one step replayed from a graph
        {"name": "step_4096", "op": "step", "bodies": 4096, "mesh": "mix3", "pool": 128, "density": 0.04,
         "fp32": True, "graph": True, "gate": False},
        # many small independent scenes advanced together: states in, pairs, clusters, step, contacts out
        {"name": "batch_scenes", "op": "loop", "bodies": 6000, "scenes": 48, "mesh": "sphere2", "pool": 128,
         "density": 0.1, "fp32": True, "funnel": False},
        # the falling pile in its funnel: one huge cluster; states in, pairs, clusters, step, contacts out
        {"name": "pile", "op": "loop", "bodies": 11003, "scenes": 1, "mesh": "sphere3", "pool": 256,
         "density": 0.1, "fp32": True, "funnel": True},
        # simulation with contact response: stacked layers settling on floors, solver included
        {"name": "sim_layers", "op": "sim", "scenes": 24, "side": 4, "layers": 2},
        # broad phase and cluster separation of a large field of bodies
        {"name": "broad_field", "op": "broad", "bodies": 65536, "statics": 3, "density": 0.1},
        # the learned gate's training step: loss and gradient of one minibatch
        {"name": "gate_grad", "op": "grad", "n": 4099},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["bucket", "filter", "narrow", "ccd", "step", "step", "loop", "loop", "sim", "broad", "grad", "infer"])
    if op == "bucket":
        return {"op": op, "mesh": rng.choice(["sphere2", "sphere3"]), "n": _log_int(rng, 5, 9000)}
    if op == "filter":
        return {"op": op, "n": _log_int(rng, 9, 4000), "patch": rng.uniform(0.1, 0.8)}
    if op in ("narrow", "ccd", "step"):
        n = _log_int(rng, 40, 1200 if op == "narrow" else 4000)
        return {"op": op, "bodies": n, "mesh": rng.choice(["sphere2", "mix2", "mix3"]), "pool": min(n, rng.randint(24, 96)),
                "density": rng.uniform(0.03, 0.12), "fp32": rng.random() < 0.7, "graph": op == "step" and rng.random() < 0.6,
                "gate": op == "ccd" and rng.random() < 0.4}
    if op == "loop":
        funnel = rng.random() < 0.4
        return {"op": op, "bodies": _log_int(rng, 500, 8000), "scenes": 1 if funnel else rng.randint(2, 80),
                "mesh": rng.choice(["sphere2", "sphere3"]), "pool": rng.randint(32, 128), "density": rng.uniform(0.05, 0.1),
                "fp32": True, "funnel": funnel}
    if op == "sim":
        return {"op": op, "scenes": rng.randint(1, 24), "side": rng.randint(2, 4), "layers": rng.randint(1, 2)}
    if op == "broad":
        return {"op": op, "bodies": _log_int(rng, 1000, 65000), "statics": rng.randint(0, 5),
                "density": rng.uniform(0.03, 0.12)}
    if op == "grad":
        return {"op": op, "n": _log_int(rng, 300, 20000)}
    return {"op": "infer", "n": _log_int(rng, 500, 200000)}


# --- the program's result buffers ----------------------------------------------
_TYPES = {"i4": (np.int32, ctypes.c_int32), "f8": (np.float64, ctypes.c_double)}


def _buffers(**spec):
    return {k: np.zeros(shape, dtype=_TYPES[t][0]) for k, (shape, t) in spec.items()}


def _contact_buffers(bodies, per_body, per_pair):
    pairs, rows = 4 * bodies + 64, per_body * bodies + 4096
    out = _buffers(offsets=(pairs + 1, "i4"), ints=((rows, 8), "i4"), reals=((rows, 11), "f8"))
    if per_pair:
        out.update(_buffers(per_pair=((pairs, 2), "f8"), steps=(bodies + 1, "f8")))
    return out


def _ptr(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_int32 if a.dtype == np.int32 else ctypes.c_double))


def _ok(ctx, rc):
    if rc != d2.D2_OK:
        raise d2.D2Error(rc, d2.lib().d2_last_error(ctx.h).decode())


# --- inputs ------------------------------------------------------------------
def _meshes(kind, count, rng):
    """`count` meshes: icospheres scaled U(0.5, 1.5) and, for a mix, every
    second one the hull of points on an ellipsoid."""
    V, F = scenes.icosphere(int(kind[-1]), 1.0)
    out = []
    for k in range(count):
        if kind.startswith("mix") and k % 2:
            out.append(scenes.ellipsoid_hull(rng))
        else:
            out.append((V * rng.uniform(0.5, 1.5), F))
    return out


def _pool(kind, count, rng, stream=50000):
    """Trees, bounding radii and inverse inertias of `count` meshes."""
    meshes = _meshes(kind, count, rng)
    trees = scenes.build_trees_parallel(meshes, stream + int(rng.integers(1 << 20)))
    radii = np.array([np.max(np.linalg.norm(V, axis=1)) for V, _ in meshes])
    inv = np.stack([np.linalg.inv(scenes.mass_properties(V, F)[2]) for V, F in meshes])
    return trees, radii, inv


def _records(rng, pos, vel, inv, spin=0.3):
    """Body records at rest poses `pos` with random rotations and spins."""
    n = pos.shape[0]
    q = rng.normal(size=(n, 4))
    r = np.zeros((n, 40))
    r[:, 0:4] = q / np.linalg.norm(q, axis=1, keepdims=True)
    r[:, 4:7] = pos
    r[:, 7:10] = vel
    r[:, 10:13] = rng.normal(0.0, spin, size=(n, 3))
    r[:, 14:28] = r[:, 0:14]
    r[:, 28:37] = inv.reshape(n, 9)
    r[:, 37] = scenes.GEO_EPS
    r[:, 39] = DT
    return r


def _field(case, rng):
    """A cube of bodies at the case's number density: jittered lattice sites,
    so that neighbours touch without piling into each other."""
    n = case["bodies"]
    pitch = case["density"] ** (-1.0 / 3.0)
    m = math.ceil(n ** (1.0 / 3.0))
    site = rng.permutation(m ** 3)[:n]
    pos = np.stack([site % m, (site // m) % m, site // (m * m)], axis=1) * pitch
    return pos + rng.uniform(-0.35, 0.35, size=(n, 3)) * pitch


def _context(case):
    ctx = d2.Context(0, d2.D2_FP32 if case.get("fp32") else d2.D2_FP64)
    if case.get("graph"):
        ctx.set_graph(True)
    if case.get("gate"):
        ctx.mlp_set_params(learned.load_weights())
        ctx.set_learned(True)
    return ctx


def _prepare_bucket(case, rng):
    trees, radii, inv = _pool(case["mesh"], 2, rng)
    gap = 0.97 * (radii[0] + radii[1])  # the surfaces just overlap
    pos = np.array([[0.0, 0.0, 0.0], gap * _unit(rng)])
    rec = _records(rng, pos, np.zeros((2, 3)), inv)
    centre = []
    for (nodes, buckets), r in zip(trees, rec):  # every node's centre in the world
        c = np.stack([buckets[:, k * 8:k * 8 + 8].sum(axis=1) / np.maximum(nodes[:, 7], 1) for k in range(9)], axis=1)
        c = (c[:, 0:3] + c[:, 3:6] + c[:, 6:9]) / 3.0
        centre.append(c @ _rotation(r[0:4]).T + r[4:7])
    leaf = [np.nonzero(t[0][:, 2] == 0)[0] for t in trees]
    d = np.linalg.norm(centre[0][leaf[0]][:, None] - centre[1][leaf[1]][None], axis=2).ravel()
    n = min(case["n"], d.size)
    near = np.sort(np.argpartition(d, n - 1)[:n])
    pairs = np.stack([leaf[0][near // leaf[1].size], leaf[1][near % leaf[1].size]], axis=1).astype(np.int32)
    ctx = d2.Context(0, d2.D2_FP64)
    ctx.upload_trees(trees)
    ctx.upload_bodies([0, 1], rec)
    return {"op": "bucket", "ctx": ctx, "pairs": pairs, "out": _buffers(used=(n, "i4"), ints=((64 + 4 * n, 8), "i4"),
                                                                        reals=((64 + 4 * n, 11), "f8"))}


def _unit(rng):
    v = rng.normal(size=3)
    return v / np.linalg.norm(v)


def _rotation(q):
    w, x, y, z = q
    return np.array([[1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y)],
                     [2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x)],
                     [2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)]])


def _prepare_filter(case, rng):
    """Contacts of one pair spread over a patch: nearly half interpenetrate
    (distance 0), the bounds come from a handful of leaf triangles."""
    n = case["n"]
    ang, rad = rng.uniform(0, 2 * np.pi, n), case["patch"] * np.sqrt(rng.uniform(0, 1, n))
    mid = np.stack([rad * np.cos(ang), rad * np.sin(ang), 0.3 * rad * rad], axis=1)
    half = 0.5 * rng.uniform(0.0, 0.02, size=n) * (rng.uniform(size=n) > 0.45)
    leaf = rng.uniform(0.0, 0.01, size=17)
    reals = np.zeros((n, 11))
    off = np.array([0.0, 0.0, 1.0]) * half[:, None]
    reals[:, 0:3], reals[:, 3:6] = mid + off, mid - off
    reals[:, 6] = 0.01 + leaf[rng.integers(17, size=n)]
    reals[:, 7] = 0.01 + leaf[rng.integers(17, size=n)]
    return {"op": "filter", "ctx": d2.Context(0, d2.D2_FP64), "reals": reals,
            "out": _buffers(order=(n, "i4"), kept=(n, "i4"))}


def _prepare_path(case, rng):
    """narrow / ccd / step: trees, bodies and the broad phase's pairs resident."""
    trees, radii, inv = _pool(case["mesh"], case["pool"], rng)
    n = case["bodies"]
    tob = rng.integers(case["pool"], size=n).astype(np.int32)
    rec = _records(rng, _field(case, rng), rng.normal(0.0, 1.0, size=(n, 3)), inv[tob])
    pairs = scenes.broad_phase(rec, radii[tob])
    ctx = _context(case)
    ctx.upload_trees(trees)
    ctx.upload_bodies(tob, rec)
    op = case["op"]
    if op == "narrow":
        ctx.project_future(rec[:, 39])
        ctx.upload_pairs(pairs)
    else:
        ctx.upload_pairs(pairs, np.minimum(rec[pairs[:, 0], 39], rec[pairs[:, 1], 39]))
    if op == "step":
        ctx.upload_clusters(*scenes.clusters(pairs, n, rec))
    return {"op": op, "ctx": ctx, "out": _contact_buffers(n, 120, op != "narrow")}


def _prepare_loop(case, rng):
    """Body states on the host, trees resident; scenes share space but not pairs."""
    n, k = case["bodies"], case["scenes"]
    trees, radii, inv = _pool(case["mesh"], case["pool"], rng)
    tob = rng.integers(case["pool"], size=n).astype(np.int32)
    group = None
    if case["funnel"]:  # inside the funnel and in the column above it, falling
        pos = _funnel_positions(rng, n, case["density"])
        vel = rng.normal(0.0, 1.0, size=(n, 3)) + np.array([0.0, 0.0, -3.0])
    else:  # scenes of uneven sizes, bodies placed at random in each one's box
        share = np.exp(rng.uniform(np.log(16), np.log(512), size=k))
        group = np.sort(rng.choice(k, size=n, p=share / share.sum())).astype(np.int32)
        side = (np.bincount(group, minlength=k) / case["density"]) ** (1.0 / 3.0)
        pos = rng.uniform(0.0, 1.0, size=(n, 3)) * side[group][:, None]
        vel = rng.normal(0.0, 1.0, size=(n, 3))
    rec = _records(rng, pos, vel, inv[tob])
    if case["funnel"]:
        V, F = scenes.funnel_mesh(n_theta=64, n_z=24)
        trees = [scenes.tree_build(V, F, d2.pcg_seed(42, 40000))] + trees
        wall = scenes.body_record(np.array([1.0, 0.0, 0.0, 0.0]), np.zeros(3), np.zeros(3), np.zeros((3, 3)), static=True)
        rec = np.concatenate([wall[None], rec])
        tob = np.concatenate([[0], tob + 1]).astype(np.int32)
    ctx = _context(case)
    ctx.upload_trees(trees)
    ctx.upload_bodies(tob, rec)
    if group is not None:
        ctx.upload_groups(group)
    out = _contact_buffers(n, 220 if case["mesh"] == "sphere3" else 120, True)
    out.update(_buffers(pairs=((out["offsets"].size - 1, 2), "i4")))
    return {"op": "loop", "ctx": ctx, "tob": tob, "rec": rec, "out": out}


def _funnel_positions(rng, n, density):
    funnel = np.pi * 40.0 / 3.0 * (20.0 ** 2 + 20.0 * 4.0 + 4.0 ** 2)
    top = 40.0 + max(0.0, (n / density - funnel) / (np.pi * 20.0 ** 2))
    out = np.zeros((0, 3))
    while out.shape[0] < n:
        c = rng.uniform(-1.0, 1.0, size=(3 * n, 3)) * np.array([20.0, 20.0, 0.5 * top]) + np.array([0.0, 0.0, 0.5 * top])
        wall = np.where(c[:, 2] < 40.0, 4.0 + 16.0 * c[:, 2] / 40.0, 20.0)
        out = np.concatenate([out, c[np.hypot(c[:, 0], c[:, 1]) < wall - 0.3]])
    return out[:n]


def _prepare_sim(case, rng):
    """Scenes of `layers` stacked layers of side x side spheres, a few
    millimetres apart and above a static floor, settling slowly."""
    k, side, layers = case["scenes"], case["side"], case["layers"]
    FV = np.array([[-10, -10, 0], [10, -10, 0], [10, 10, 0], [-10, 10, 0]], dtype=float)
    FF = np.array([[0, 1, 2], [0, 2, 3]], dtype=np.int32)
    V, F = scenes.icosphere(1, 0.5)
    vol, _, inertia = scenes.mass_properties(V, F)
    stream = d2.pcg_seed(42, 54)
    trees = [scenes.tree_build(FV, FF, stream), scenes.tree_build(V, F, stream)]
    ext, gap = V.max(axis=0) - V.min(axis=0), 0.003
    rec, tob = [], []
    for _ in range(k):
        rec.append(scenes.body_record(np.array([1.0, 0, 0, 0]), np.zeros(3), np.zeros(3), np.zeros((3, 3)), static=True))
        tob.append(0)
        for z in range(layers):
            for i in range(side):
                for j in range(side):
                    p = np.array([i - 0.5 * side, j - 0.5 * side, z]) * (ext + gap)
                    p[2] += gap - V[:, 2].min()
                    v = rng.normal(0.0, 0.05, size=3) * np.array([1.0, 1.0, 0.1]) - np.array([0.0, 0.0, 0.05])
                    rec.append(scenes.body_record(np.array([1.0, 0, 0, 0]), p, v, np.linalg.inv(inertia)))
                    tob.append(1)
    rec, tob = np.stack(rec), np.array(tob, dtype=np.int32)
    ctx = d2.Context(0, d2.D2_FP32)
    ctx.upload_trees(trees)
    ctx.upload_bodies(tob, rec)
    ctx.upload_groups(np.repeat(np.arange(k), 1 + layers * side * side).astype(np.int32))
    ctx.solver_bodies(np.where(tob == 0, 1.0, vol), np.full(tob.size, 0.4))
    return {"op": "sim", "ctx": ctx, "tob": tob, "rec": rec,
            "out": _buffers(status=(tob.size, "i4"), steps=(tob.size, "f8"))}


def _prepare_broad(case, rng):
    n, s = case["bodies"], case["statics"]
    trees, _, inv = _pool("sphere1", 24, rng)
    tob = rng.integers(24, size=n).astype(np.int32)
    side = (n / case["density"]) ** (1.0 / 3.0)
    rec = _records(rng, rng.uniform(0.0, side, size=(n, 3)), rng.normal(0.0, 1.0, size=(n, 3)), inv[tob])
    rec[rng.permutation(n)[:s], 38] = 1.0
    ctx = d2.Context(0, d2.D2_FP32)
    ctx.upload_trees(trees)
    ctx.upload_bodies(tob, rec)
    ctx.project_future(rec[:, 39])
    return {"op": "broad", "ctx": ctx,
            "out": _buffers(pairs=((4 * n + 64, 2), "i4"), max_time=(4 * n + 64, "f8"), of_pair=(4 * n + 64, "i4"),
                            of_body=(n, "i4"), first=(n, "i4"), min_time=(n, "f8"), step=(n, "f8"))}


def _gate_inputs(case, seed):
    """Network parameters, feature rows and labels as training meets them."""
    rng = np.random.default_rng(seed)
    n = case["n"]
    params = learned.init_params(int(rng.integers(1 << 30)))
    X = rng.normal(0.0, 0.5, size=(n, 24)).astype(np.float32)
    T = np.stack([rng.uniform(0.0, 1.0, size=n), rng.choice([0.3, 0.7, 1.25], size=n)], axis=1).astype(np.float32)
    return params, X, T


def _prepare_gate(case, seed):
    params, X, T = _gate_inputs(case, seed)
    ctx = d2.Context(0, d2.D2_FP32)
    ctx.mlp_set_params(params)
    return {"op": case["op"], "ctx": ctx, "X": X, "T": T}


def prepare(case, seed):
    if case["op"] in ("grad", "infer"):
        return _prepare_gate(case, seed)
    make = {"bucket": _prepare_bucket, "filter": _prepare_filter, "narrow": _prepare_path, "ccd": _prepare_path,
            "step": _prepare_path, "loop": _prepare_loop, "sim": _prepare_sim, "broad": _prepare_broad}[case["op"]]
    return make(case, np.random.default_rng(seed))


# --- one pass ------------------------------------------------------------------
def _read_contacts(ctx, out):
    """The last run's contacts (and its continuous phase's per-pair values)."""
    if ctx.n_out > out["ints"].shape[0] or ctx.n_pairs >= out["offsets"].size:
        raise RuntimeError("more results than the buffers hold")
    L = d2.lib()
    _ok(ctx, L.d2_result_contacts(ctx.h, _ptr(out["offsets"]), _ptr(out["ints"]), _ptr(out["reals"])))
    if "per_pair" in out:
        _ok(ctx, L.d2_result_pairs(ctx.h, _ptr(out["per_pair"])))


def _step(ctx, out):
    n = ctypes.c_int64(0)
    _ok(ctx, d2.lib().d2_step_run(ctx.h, DT, 1, _ptr(out["steps"]), ctypes.byref(n)))
    ctx.n_out = n.value


def run(state):
    op, ctx, out = state["op"], state["ctx"], state.get("out")
    L = d2.lib()
    if op == "bucket":
        hits = ctypes.c_int64(0)
        _ok(ctx, L.d2_find_contacts_bucket(ctx.h, 0, 1, out["used"].size, _ptr(state["pairs"]), _ptr(out["used"]),
                                           out["ints"].shape[0], _ptr(out["ints"]), _ptr(out["reals"]),
                                           ctypes.byref(hits)))
        return out
    if op == "filter":
        k = ctypes.c_int(0)
        _ok(ctx, L.d2_filter_contacts(ctx.h, out["order"].size, _ptr(state["reals"]), 0.0, _ptr(out["order"]),
                                      _ptr(out["kept"]), ctypes.byref(k)))
        out["kept"][k.value:] = -1  # only the first k entries are results
        return out
    if op == "grad":
        loss, grad = ctx.mlp_loss_grad(state["X"], state["T"], learned.LW, learned.DELTA)
        return {"loss": loss, "grad": grad}
    if op == "infer":
        return {"y": ctx.mlp_infer(state["X"])}
    if op in ("narrow", "ccd"):
        ctx.narrow_run(True) if op == "narrow" else ctx.ccd_run()
        _read_contacts(ctx, out)
        return out
    if op == "step":
        _step(ctx, out)
        _read_contacts(ctx, out)
        return out
    if op == "broad":
        if ctx.broad_phase(mode=1) > out["max_time"].size:
            raise RuntimeError("more results than the buffers hold")
        ctx.build_clusters()
        _ok(ctx, L.d2_pairs_download(ctx.h, _ptr(out["pairs"]), _ptr(out["max_time"])))
        _ok(ctx, L.d2_clusters_download(ctx.h, _ptr(out["of_pair"]), _ptr(out["of_body"]), _ptr(out["first"]),
                                        _ptr(out["min_time"]), _ptr(out["step"])))
        return out
    rec = state["rec"]  # loop, sim: the host owns the body states
    ctx.upload_bodies(state["tob"], rec)
    ctx.project_future(np.minimum(2.0 * rec[:, 39], DT))
    ctx.broad_phase(mode=1)
    ctx.build_clusters()
    _step(ctx, out)
    if op == "loop":
        _read_contacts(ctx, out)
        _ok(ctx, L.d2_pairs_download(ctx.h, _ptr(out["pairs"]), None))
        return out
    status, _ = ctx.solve(GRAVITY)
    ctx.commit_step()
    out["status"][:status.size] = status
    out["bodies"] = ctx.download_bodies()
    return out


# --- what a pass cannot do without -----------------------------------------------
NODES = {"1": 45, "2": 161, "3": 665}  # tree nodes of an icosphere by subdivision
TREE_NODE = 16 + 24 * 9 * 2  # bytes: a node record's ids and its bucket's triangles, about two of eight used


def work(case):
    """Bytes: trees, body records and pairs in, contacts out, once each.
    Operations: the tests that report a contact (about 600 in each triangle
    distance, 6000 in each continuous test) at the scenes' usual counts."""
    op = case["op"]
    if op == "bucket":
        return {"bytes": case["n"] * (8 + 4 + 2 * TREE_NODE + 3 * 120), "flops": case["n"] * 5 * 600}
    if op == "filter":
        return {"bytes": case["n"] * (88 + 4 + 2), "flops": case["n"] * 40}
    if op in ("grad", "infer"):
        per = 24 * 64 + 64 * 64 + 64 * 2
        return {"bytes": case["n"] * (96 + 8) + 4 * 5890, "flops": case["n"] * per * (6 if op == "grad" else 2)}
    if op == "broad":
        return {"bytes": case["bodies"] * (320 + 112 + 4 + 2.2 * (8 + 8 + 4)), "flops": case["bodies"] * 8 * 60}
    if op == "sim":
        n = case["scenes"] * case["layers"] * case["side"] ** 2
        return {"bytes": n * (640 + 8 * 88), "flops": n * 8 * 40 * 1000}
    n = case["bodies"]
    pairs = n * 22.0 * case["density"]
    trees = case["pool"] * NODES[case["mesh"][-1]] * TREE_NODE
    hits = 35 if op == "ccd" else 25
    flops = pairs * hits * ((600 if op != "ccd" else 0) + (6000 if op != "narrow" else 0))
    return {"bytes": trees + n * 320 + pairs * (16 + 16) + pairs * hits * 120, "flops": flops}


def exact(case, seed):
    """The gate's outputs in 64 bits (with the weights rounded to bf16, which
    the network is defined with).  The other outputs are orders, index sets
    and the double-precision traversal's own values."""
    if case["op"] not in ("grad", "infer"):
        return None
    params, X, T = _gate_inputs(case, seed)
    u = params.view(np.uint32)
    p = ((u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000).astype(np.uint32).view(np.float32).astype(np.float64)
    W1, b1, W2, b2, W3, b3 = np.split(p, np.cumsum([24 * 64, 64, 64 * 64, 64, 64 * 2]))
    W1, W2, W3 = W1.reshape(24, 64), W2.reshape(64, 64), W3.reshape(64, 2)
    x, t = X.astype(np.float64), T.astype(np.float64)
    h1 = np.maximum(x @ W1 + b1, 0.0)
    h2 = np.maximum(h1 @ W2 + b2, 0.0)
    y = h2 @ W3 + b3
    if case["op"] == "infer":
        return {"y": y}
    r, delta, lw = y - t, float(np.float32(learned.DELTA)), np.array(learned.LW)
    a = np.abs(r)
    loss = (np.where(a <= delta, 0.5 * r * r, delta * (a - 0.5 * delta)) * lw).sum(axis=1).mean()
    d3 = np.where(a <= delta, r, np.sign(r) * delta) * lw / case["n"]
    d2v = (d3 @ W3.T) * (h2 > 0)
    d1 = (d2v @ W2.T) * (h1 > 0)
    grad = np.concatenate([(x.T @ d1).ravel(), d1.sum(axis=0), (h1.T @ d2v).ravel(), d2v.sum(axis=0),
                           (h2.T @ d3).ravel(), d3.sum(axis=0)])
    return {"loss": float(loss), "grad": grad}
