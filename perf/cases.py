"""The workloads the framework's speed is followed on, each one pass through
its public entry points.

  update  one ParticleSystem.update(dt): the loop an unchanged caller of the
          reference's class runs, once per frame or per coupling sub-step
  run     ParticleSystem.run(dt, steps): a stretch of a simulation between two
          looks at its state; box walls and equal spheres, or log-normal radii
          around a torus-knot boundary given by a distance map
  stages  the per-stage C entry points (integrate, calcHash, sort, reorder,
          collide) on caller-owned arrays: the drop-in boundary of the
          reference's particleSystem.cu
  batch   Batch.run of independent scenes of uneven sizes, and their state
          back on the host: a parameter study
  build   DistanceMap.from_mesh of a closed mesh, and the map's values at its
          lattice vertices: a rigid body enters the scene
  labels  mesh_signed_distance of host points: a surrogate's training labels
  query   queryMap of device points: collision queries against a body's map
  grad    one gradient of every body's distance network over its samples: the
          body of each training step
  eval    distances of device points from the networks, in BF16 (inference) or
          FP32 (the training arithmetic)

Particle states are settled beds (the lattice of reset() after it has fallen),
the state a simulation spends nearly all of its steps in.  They go on moving
from pass to pass, as a simulation does.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from fullc0ntact_amd import Context, ParticleSystem, make_params
from fullc0ntact_amd import meshes, statistics
from fullc0ntact_amd._lib import DeviceArray, check, lib
from fullc0ntact_amd.batch import Batch, ensemble_scene_counts, jittered_params
from fullc0ntact_amd.distance_map import DistanceMap, mesh_signed_distance
from fullc0ntact_amd.sdf import BF16, FP32, SdfSurrogate

DT = 0.5


def listed() -> list[dict]:
    return [
        # the class defaults (r = 1/16), one sphere per rigid body, stepped frame by
        # frame: launches and latency count
        dict(name="update-1331", kind="update", n=1331, inv_r=16, grid=16, settle=600),
        # the 4096-sphere case (r = 1/64 in a 64^3 grid)
        dict(name="run-4096", kind="run", n=4096, inv_r=64, grid=64, settle=600, steps=100,
             knot=False),
        # an ordinary scene: odd count, radii that differ, a rigid boundary
        dict(name="run-knot-120011", kind="run", n=120011, inv_r=128, grid=128, settle=800,
             steps=20, knot=True),
        # the 1M-sphere bed (r = 1/128 in a 256^3 grid), step by step and as a run
        dict(name="update-1M", kind="update", n=1 << 20, inv_r=128, grid=256, settle=1500),
        dict(name="run-1M", kind="run", n=1 << 20, inv_r=128, grid=256, settle=1500, steps=20,
             knot=False),
        # an unchanged host program of the reference, at a ragged size
        dict(name="stages-500009", kind="stages", n=500009, inv_r=128, grid=128, settle=1000),
        # a parameter study over uneven scenes
        dict(name="batch-32", kind="batch", scenes=32, lo=2000, hi=60000, inv_r=64, grid=64,
             settle=300, steps=50),
        # a body's map at the resolution of a contact query, a 6144-triangle knot
        dict(name="build-64", kind="build", cells=64, nu=256, nv=12),
        # the labels of one network at build_scene's default sample count
        dict(name="labels-65536", kind="labels", n=65536, nu=256, nv=12),
        # a million queries against one map
        dict(name="query-1000003", kind="query", n=1000003, cells=64),
        # a training step of eight bodies' networks at build_scene's minibatch
        # scale, and the inference of their networks
        dict(name="grad-8x16384", kind="grad", bodies=8, samples=16384),
        dict(name="eval-bf16-500003", kind="eval", n=500003, bodies=8, bf16=True),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _inv_r(n: int) -> int:
    """The smallest power of two 1/r whose reset() lattice fits the box."""
    s = 1
    while s ** 3 < n:
        s += 1
    k = 16
    while k < s:
        k *= 2
    return k


def _settle(n: int) -> int:
    return 600 if n <= 20000 else 1000


def draw(rng) -> dict:
    kind = rng.choice(["update", "run", "run", "stages", "batch", "build", "labels", "query",
                       "grad", "eval"])
    if kind in ("update", "stages"):
        n = _log_int(rng, 600, 1000000)
        return dict(kind=kind, n=n, inv_r=_inv_r(n), grid=max(64, _inv_r(n)), settle=_settle(n))
    if kind == "run":
        knot = rng.random() < 0.4
        n = _log_int(rng, 3000, 200000) if knot else _log_int(rng, 600, 900000)
        inv_r = 128 if knot else _inv_r(n)
        steps = rng.randint(3, max(4, min(100, 16000000 // n)))
        return dict(kind=kind, n=n, inv_r=inv_r, grid=max(64, inv_r), settle=_settle(n),
                    steps=steps, knot=knot)
    if kind == "batch":
        return dict(kind=kind, scenes=rng.randint(3, 40), lo=_log_int(rng, 500, 5000),
                    hi=_log_int(rng, 6000, 50000), inv_r=64, grid=64, settle=200,
                    steps=rng.randint(20, 50))
    mesh = rng.choice([(64, 8), (128, 12), (256, 12)])
    if kind == "build":
        return dict(kind=kind, cells=rng.randint(12, 64), nu=mesh[0], nv=mesh[1])
    if kind == "labels":
        return dict(kind=kind, n=_log_int(rng, 500, 65536), nu=mesh[0], nv=mesh[1])
    if kind == "query":
        return dict(kind=kind, n=_log_int(rng, 300, 1000000), cells=rng.randint(24, 64))
    if kind == "grad":
        return dict(kind=kind, bodies=rng.randint(1, 8), samples=_log_int(rng, 300, 16384))
    return dict(kind=kind, n=_log_int(rng, 300, 500000), bodies=rng.randint(1, 8),
                bf16=rng.random() < 0.6)


# ---------------------------------------------------------------------------
# What a user's program has in hand before the call.
# ---------------------------------------------------------------------------
_ctx = None


def _context() -> Context:
    """The program's one context: its passes follow each other on one stream."""
    global _ctx
    if _ctx is None:
        _ctx = Context()
    return _ctx


class _Raw:
    """A device array by its address, for torch.as_tensor."""

    def __init__(self, ptr: int, shape, typestr: str):
        self.__cuda_array_interface__ = dict(data=(ptr, False), shape=tuple(shape),
                                             typestr=typestr, version=3, strides=None)


def _view(ps: ParticleSystem, name: str) -> torch.Tensor:
    """A system's device array as a tensor that keeps the system alive (the
    memory is the system's, and goes with it)."""
    t = torch.as_tensor(_Raw(ps.device_arrays()[name], (ps.getNumParticles(), 4), "<f4"),
                        device="cuda")
    t.owner = ps
    return t


def _knot_mesh(nu: int, nv: int, seed: int):
    """The benchmark hopper's (2, 3) torus-knot tube, its size drawn."""
    rng = np.random.default_rng(seed)
    return meshes.torus_knot(2, 3, nu, nv, radius=float(rng.uniform(0.10, 0.13)),
                             scale=float(rng.uniform(0.23, 0.27)), center=(0.0, 0.0, -0.55))


def _knot_map(ctx, cells: int, seed: int) -> DistanceMap:
    v, f = _knot_mesh(256, 12, seed)
    return DistanceMap.from_mesh(ctx, v, f, (cells,) * 3, 2.0 / cells, (-1.0, -1.0, -1.0))


def _bed(case: dict, seed: int) -> dict:
    """A particle system whose lattice has fallen for `settle` steps."""
    n, r = case["n"], 1.0 / case["inv_r"]
    ps = ParticleSystem(n, (case["grid"],) * 3, context=_context())
    s = dict(ps=ps)
    if case.get("knot"):
        rmax = float(np.float32(r * math.sqrt(3.0)))
        ps.m_params = make_params(n, case["grid"], rmax)
        rng = np.random.default_rng(seed)
        side = int(math.floor(1.3 / (2.0 * rmax)))  # a block inside the unit cylinder
        i = np.arange(n)
        at = np.stack([i % side, (i // side) % side, i // (side * side)], 1)
        pos = np.empty((n, 4), np.float32)
        pos[:, :3] = (at - [0.5 * (side - 1), 0.5 * (side - 1), 0.0]) * 2.0 * rmax \
            + [0.0, 0.0, rmax - 1.0] + rng.uniform(-0.1, 0.1, (n, 3)) * rmax
        pos[:, 3] = statistics.polydisperse_radii(n, r, 0.25, 3.0, seed=seed)
        vel = np.zeros((n, 4), np.float32)
        vel[:, :3] = rng.uniform(-0.01, 0.01, (n, 3))
        ps.setArray(ps.POSITION, pos, 0, n)
        ps.setArray(ps.VELOCITY, vel, 0, n)
        ps.setPolydisperse(True)
        s["map"] = _knot_map(ps.ctx, 64, seed)
        ps.setBoundary(s["map"])
    else:
        ps.m_params = make_params(n, case["grid"], r)
        ps.reset(ps.CONFIG_GRID, seed, 0.1, 0.01)
    ps.run(DT, case["settle"])
    ps.sync()
    s["pos"], s["vel"] = _view(ps, "pos"), _view(ps, "vel")
    return s


def _points(n: int, seed: int) -> np.ndarray:
    """Points in the cube [-1, 1]^3, as float64."""
    return np.random.default_rng(seed).uniform(-1.0, 1.0, (n, 3))


def _networks(ctx, bodies: int, seed: int) -> SdfSurrogate:
    rng = np.random.default_rng(seed)
    return SdfSurrogate(ctx, rng.uniform(-0.1, 0.1, (bodies, 3)), rng.uniform(0.8, 1.2, bodies),
                        seed=seed)


def _samples(case: dict, seed: int):
    """Points of every body's box and the distances of a rippled sphere."""
    p = _points(case["bodies"] * case["samples"], seed + 1).astype(np.float32)
    r = np.linalg.norm(p, axis=1)
    return p, (r - 0.5 - 0.05 * np.sin(7.0 * p[:, 0])).astype(np.float32)


def _lattice(m: DistanceMap) -> torch.Tensor:
    """The float32 coordinates of a map's lattice vertices, x fastest."""
    ax = [torch.from_numpy((m.bmin[a] + np.arange(m.cells[a] + 1) * np.float64(
        np.float32(m.cell_size))).astype(np.float32)) for a in range(3)]
    z, y, x = torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    return torch.stack([x, y, z], -1).reshape(-1, 3).contiguous().cuda()


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    s = dict(case=case)
    if kind in ("update", "run"):
        s.update(_bed(case, seed))
    elif kind == "stages":
        bed = _bed(case, seed)
        ps = bed["ps"]
        n, cells = case["n"], ps.m_params.numCells
        ctx = s["ctx"] = _context()
        ctx.set_parameters(ps.m_params)
        s["params"] = ps.m_params
        s["pos"], s["vel"] = bed["pos"].clone(), bed["vel"].clone()
        for k in ("sortedPos", "sortedVel"):
            s[k] = torch.empty_like(s["pos"])
        for k in ("hash", "index"):
            s[k] = torch.empty(n, dtype=torch.int32, device="cuda")
        for k in ("cellStart", "cellEnd"):
            s[k] = torch.empty(cells, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        del bed["pos"], bed["vel"]
        ps.close()
    elif kind == "batch":
        counts = ensemble_scene_counts(case["scenes"], case["lo"], case["hi"])
        b = s["batch"] = Batch(counts, (case["grid"],) * 3, context=_context())
        b.set_params(jittered_params(make_params(0, case["grid"], 1.0 / case["inv_r"]),
                                     case["scenes"], seed=seed))
        b.reset(seed=seed, jitter_frac=0.1, vel_amp=0.01)
        b.run(DT, case["settle"])
        b.sync()
    elif kind == "build":
        s["ctx"] = _context()
        s["mesh"] = _knot_mesh(case["nu"], case["nv"], seed)
        c = case["cells"]
        probe = DistanceMap.from_mesh(s["ctx"], *s["mesh"], (c,) * 3, 2.0 / c, (-1.0,) * 3)
        s["pts"] = _lattice(probe)
        probe.close()
        s["out"] = _query_out(len(s["pts"]))
    elif kind == "labels":
        s["ctx"] = _context()
        s["mesh"] = _knot_mesh(case["nu"], case["nv"], seed)
        s["pts"] = _points(case["n"], seed + 1)
    elif kind == "query":
        s["ctx"] = _context()
        s["map"] = _knot_map(s["ctx"], case["cells"], seed)
        s["pts"] = torch.from_numpy(_points(case["n"], seed + 1).astype(np.float32)).cuda()
        s["out"] = _query_out(case["n"])
    elif kind == "grad":
        s["ctx"] = _context()
        s["net"] = _networks(s["ctx"], case["bodies"], seed)
        p, y = _samples(case, seed)
        s["pts"] = DeviceArray.from_host(s["ctx"], p)
        s["labels"] = DeviceArray.from_host(s["ctx"], y)
    else:
        s["ctx"] = _context()
        s["net"] = _networks(s["ctx"], case["bodies"], seed)
        n = case["n"]
        s["pts"] = torch.from_numpy(_points(n, seed + 1).astype(np.float32)).cuda()
        s["of"] = (torch.arange(n, device="cuda") * case["bodies"] // n).to(torch.int32)
        s["out"] = torch.empty(n, device="cuda")
    torch.cuda.synchronize()
    return s


def _query_out(n: int) -> dict:
    return dict(dist=torch.empty(n, device="cuda"), cp=torch.empty(n, 3, device="cuda"),
                normal=torch.empty(n, 3, device="cuda"))


def _query(s: dict, m: DistanceMap) -> dict:
    o, p = s["out"], s["pts"]
    check(lib.fc_distmap_query(s["ctx"].handle, m.handle, p.data_ptr(), len(p),
                               o["dist"].data_ptr(), o["cp"].data_ptr(), o["normal"].data_ptr()))
    return o


# ---------------------------------------------------------------------------
# One pass.
# ---------------------------------------------------------------------------
def run(s: dict):
    case = s["case"]
    kind = case["kind"]
    if kind == "update":
        s["ps"].update(DT)
        return dict(pos=s["pos"], vel=s["vel"])
    if kind == "run":
        s["ps"].run(DT, case["steps"])
        return dict(pos=s["pos"], vel=s["vel"])
    if kind == "stages":
        n, h = case["n"], s["ctx"].handle
        d = {k: v.data_ptr() for k, v in s.items() if isinstance(v, torch.Tensor)}
        check(lib.fc_integrate_system(h, d["pos"], d["vel"], C.c_float(DT), n))
        check(lib.fc_calc_hash(h, d["hash"], d["index"], d["pos"], n))
        check(lib.fc_sort_particles(h, d["hash"], d["index"], n))
        check(lib.fc_reorder_data_and_find_cell_start(
            h, d["cellStart"], d["cellEnd"], d["sortedPos"], d["sortedVel"], d["hash"],
            d["index"], d["pos"], d["vel"], n, s["params"].numCells))
        check(lib.fc_collide(h, d["vel"], d["sortedPos"], d["sortedVel"], d["index"],
                             d["cellStart"], d["cellEnd"], n, s["params"].numCells))
        return {k: s[k] for k in ("pos", "vel", "sortedPos", "sortedVel", "hash", "index",
                                  "cellStart", "cellEnd")}
    if kind == "batch":
        b = s["batch"]
        b.run(DT, case["steps"])
        return dict(pos=b.get_array(0), vel=b.get_array(1))
    if kind == "build":
        c = case["cells"]
        s["map"] = DistanceMap.from_mesh(s["ctx"], *s["mesh"], (c,) * 3, 2.0 / c, (-1.0,) * 3)
        return _query(s, s["map"])
    if kind == "labels":
        sd, cp = mesh_signed_distance(s["ctx"], *s["mesh"], s["pts"])
        return dict(sdf=sd, cp=cp)
    if kind == "query":
        return _query(s, s["map"])
    if kind == "grad":
        g, loss = s["net"].loss_grad(s["pts"], s["labels"], case["samples"])
        return dict(grad=g[:, :s["net"].nparams], loss=loss)
    check(lib.fc_sdf_eval(s["net"].handle, s["of"].data_ptr(), s["pts"].data_ptr(), case["n"],
                          s["out"].data_ptr(), BF16 if case["bf16"] else FP32))
    return s["out"]


# ---------------------------------------------------------------------------
# What one pass cannot do without.
# ---------------------------------------------------------------------------
_NET_MACS = 32 * 64 + 2 * 64 * 64 + 64  # products of one network evaluation


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("update", "run", "stages"):
        # per step the state is read once and written once; about 12 contacts
        # of a sphere at 45 operations; a stage caller also gets the sorted
        # state, the (hash, index) pairs and the dense cell tables
        n, steps = case["n"], case.get("steps", 1)
        extra = n * 40 + 8 * case["grid"] ** 3 if kind == "stages" else 0
        return dict(bytes=steps * n * 64 + extra, flops=steps * n * 12 * 45)
    if kind == "batch":
        n = int(ensemble_scene_counts(case["scenes"], case["lo"], case["hi"]).sum())
        return dict(bytes=case["steps"] * n * 64, flops=case["steps"] * n * 12 * 45)
    if kind == "build":
        # the map (32 B a vertex) is written, and read back by the query
        v = (case["cells"] + 1) ** 3
        tri = 2 * case["nu"] * case["nv"]
        return dict(bytes=v * (32 + 12 + 28) + tri * 24, flops=v * 200)
    if kind == "labels":
        return dict(bytes=case["n"] * (24 + 32) + 2 * case["nu"] * case["nv"] * 24,
                    flops=case["n"] * 200)
    if kind == "query":
        # every vertex of the map once, each point in and its answer out
        return dict(bytes=case["n"] * 40 + 32 * (case["cells"] + 1) ** 3, flops=case["n"] * 100)
    if kind == "grad":
        m = case["bodies"] * case["samples"]
        return dict(bytes=m * 16 + case["bodies"] * 84000, flops=6 * m * _NET_MACS)
    return dict(bytes=case["n"] * 20 + case["bodies"] * 42000, flops=2 * case["n"] * _NET_MACS)


# ---------------------------------------------------------------------------
# The same outputs in binary64, by plain torch.
# ---------------------------------------------------------------------------
def _dot(a, b):
    return (a * b).sum(-1)


def _map64(m: DistanceMap) -> dict:
    """A map's contents as its lattice holds them, in binary64."""
    lay = m.download()
    shape = tuple(c + 1 for c in reversed(m.cells))
    f64 = {k: torch.from_numpy(np.asarray(v, np.float64)).cuda() for k, v in lay.items()}
    g = dict(dist=f64["distance"].reshape(shape), cp=f64["contact_points"].reshape(*shape, 3),
             normal=f64["normals"].reshape(*shape, 3))
    at = f64["vertex_coords"].reshape(*shape, 3)
    g["axes"] = [at[0, 0, :, 0], at[0, :, 0, 1], at[:, 0, 0, 2]]
    g["cells"], g["cell"] = m.cells, float(np.float32(m.cell_size))
    g["lo"] = torch.tensor(m.bmin, dtype=torch.float64, device="cuda")
    g["hi"] = torch.tensor(m.bmax, dtype=torch.float64, device="cuda")
    return g


def _query64(g: dict, q: torch.Tensor):
    """(inside, distance, closest point, normal) of float64 points."""
    inside = ((q >= g["lo"]) & (q <= g["hi"])).all(1)
    c, w = [], []
    for a in range(3):
        i = ((q[:, a] - g["lo"][a]).abs() / g["cell"]).long().clamp(0, g["cells"][a] - 1)
        ax = g["axes"][a]
        c.append(i)
        w.append((q[:, a] - ax[i]) / (ax[i + 1] - ax[i]))
    d = torch.zeros(len(q), dtype=torch.float64, device=q.device)
    p = torch.zeros_like(q)
    for k in range(8):
        o = (k & 1, (k >> 1) & 1, k >> 2)
        t = torch.ones_like(d)
        for a in range(3):
            t = t * (w[a] if o[a] else 1.0 - w[a])
        at = (c[2] + o[2], c[1] + o[1], c[0] + o[0])
        d += t * g["dist"][at]
        p += t[:, None] * g["cp"][at]
    nrm = g["normal"][c[2], c[1], c[0]].clone()
    d[~inside] = 5.0
    p[~inside] = 0.0
    nrm[~inside] = 0.0
    return inside, d, p, nrm


def _integrate64(pos, vel, rad, P, dt, g):
    vel = (vel + torch.tensor([P.gravity.x, P.gravity.y, P.gravity.z], dtype=torch.float64,
                              device=pos.device) * dt) * P.globalDamping
    pos = pos + vel * dt
    bd = P.boundaryDamping
    if g is None:
        for a in range(3):
            hi, lo = pos[:, a] > 1.0 - rad, pos[:, a] < -1.0 + rad
            pos[:, a] = torch.where(hi, 1.0 - rad, torch.where(lo, -1.0 + rad, pos[:, a]))
            vel[:, a] = torch.where(hi | lo, vel[:, a] * bd, vel[:, a])
        return pos, vel
    pc = pos * torch.tensor([1.0, 1.0, 0.0], dtype=torch.float64, device=pos.device)
    length = pc.norm(dim=1)
    _, d, cp, _ = _query64(g, pos)
    hit = d < rad
    nn = pos - cp
    nn = nn / nn.norm(dim=1, keepdim=True)
    pos = torch.where(hit[:, None], pos + nn * (rad - d + 0.1 * rad)[:, None], pos)
    kick = torch.tensor([0.5 * bd, 0.5 * bd, 0.7 * bd], dtype=torch.float64, device=pos.device)
    vel = torch.where(hit[:, None], vel * kick, vel)
    out = length > 1.0
    push = pc / length.clamp_min(1e-300)[:, None] * (length - 1.0 + rad)[:, None]
    pos = torch.where(out[:, None], pos - push, pos)
    vel = torch.where(out[:, None], vel * torch.tensor([bd, bd, 1.0], dtype=torch.float64,
                                                       device=pos.device), vel)
    for limit, side in ((10.0 - rad, 1.0), (rad - 1.0, -1.0)):
        over = (pos[:, 2] - limit) * side > 0
        pos[:, 2] = torch.where(over, limit, pos[:, 2])
        vel[:, 2] = torch.where(over, vel[:, 2] * bd, vel[:, 2])
    return pos, vel


def _collide64(pos, vel, rad, P, scene, spring, damping):
    """New velocities: every pair in contact, found through the grid."""
    n, G = len(pos), (P.gridSize.x, P.gridSize.y, P.gridSize.z)
    org = (P.worldOrigin.x, P.worldOrigin.y, P.worldOrigin.z)
    cs = (P.cellSize.x, P.cellSize.y, P.cellSize.z)
    cell = [torch.floor((pos[:, a] - org[a]) / cs[a]).nan_to_num(0.0).long() & (G[a] - 1)
            for a in range(3)]
    cells = G[0] * G[1] * G[2]

    def key(x, y, z):
        return scene * cells + (z * G[1] + y) * G[0] + x

    h = key(*cell)
    order = torch.argsort(h, stable=True)
    ends = torch.bincount(h, minlength=cells * (int(scene.max()) + 1)).cumsum(0)
    force = torch.zeros_like(pos)

    def add(i, j, at, from_a):
        d = at[j] - from_a
        dist = d.norm(dim=1)
        reach = rad[i] + (rad[j] if at is pos else P.colliderRadius)
        m = dist < reach
        i, j, d, dist, reach = i[m], j[m], d[m], dist[m], reach[m]
        nrm = d / dist[:, None]
        rv = (vel[j] if at is pos else 0.0) - vel[i]
        tv = rv - _dot(rv, nrm)[:, None] * nrm
        f = nrm * (-spring[i] * (reach - dist))[:, None] + rv * damping[i][:, None] \
            + tv * P.shear + d * P.attraction
        force.index_add_(0, i, f)

    every = torch.arange(n, device=pos.device)
    for k in range(27):
        o = (k % 3 - 1, k // 3 % 3 - 1, k // 9 - 1)
        c = key(*[(cell[a] + o[a]) & (G[a] - 1) for a in range(3)])
        start = torch.where(c > 0, ends[(c - 1).clamp_min(0)], 0)
        left = ends[c] - start
        i = every
        t = 0
        while True:
            i = i[left[i] > t]
            if len(i) == 0:
                break
            j = order[start[i] + t]
            keep = i != j
            add(i[keep], j[keep], pos, pos[i[keep]])
            t += 1
    ball = torch.tensor([[P.colliderPos.x, P.colliderPos.y, P.colliderPos.z]],
                        dtype=torch.float64, device=pos.device)
    add(every, torch.zeros_like(every), ball, pos)
    return vel + force


def _steps64(pos4, vel4, P, steps, g=None, poly=False, scene=None, spring=None, damping=None):
    pos, vel = pos4[:, :3].double(), vel4[:, :3].double()
    n = len(pos)

    def full(v):
        return torch.full((n,), float(v), dtype=torch.float64, device=pos.device)

    rad = pos4[:, 3].double() if poly else full(P.particleRadius)
    scene = torch.zeros(n, dtype=torch.long, device=pos.device) if scene is None else scene
    spring = full(P.spring) if spring is None else spring
    damping = full(P.damping) if damping is None else damping
    for _ in range(steps):
        pos, vel = _integrate64(pos, vel, rad, P, DT, g)
        vel = _collide64(pos, vel, rad, P, scene, spring, damping)
    return (torch.cat([pos, pos4[:, 3:].double()], 1),
            torch.cat([vel, torch.zeros_like(vel[:, :1])], 1))


def _mesh64(v, f, q: torch.Tensor):
    """(signed distance, closest point) of float64 points: every triangle."""
    tri = torch.from_numpy(np.asarray(v, np.float64)[np.asarray(f, np.int64)]).cuda()
    A, B, Cc = tri[:, 0], tri[:, 1], tri[:, 2]
    sd, cps = [], []
    for p in q.split(max(1, 6000000 // len(tri))):
        best = torch.full((len(p),), math.inf, dtype=torch.float64, device=p.device)
        at = torch.zeros_like(p)
        X = p[:, None]
        # the three edges
        for s, e in ((A, B), (B, Cc), (Cc, A)):
            d = e - s
            t = (_dot(X - s, d) / _dot(d, d)).clamp(0.0, 1.0)
            c = s + t[..., None] * d
            r, k = _dot(X - c, X - c).min(1)
            hit = r < best
            best = torch.where(hit, r, best)
            at = torch.where(hit[:, None], c[torch.arange(len(p), device=p.device), k], at)
        # the inside, where the foot of the perpendicular lies in it
        nrm = torch.linalg.cross(B - A, Cc - A)
        h = _dot(X - A, nrm) / _dot(nrm, nrm)
        foot = X - h[..., None] * nrm
        ok = torch.ones_like(h, dtype=torch.bool)
        for s, e in ((A, B), (B, Cc), (Cc, A)):
            ok &= _dot(torch.linalg.cross((e - s).expand_as(foot), foot - s), nrm) >= 0
        r, k = torch.where(ok, h * h * _dot(nrm, nrm), math.inf).min(1)
        hit = r < best
        best = torch.where(hit, r, best)
        at = torch.where(hit[:, None], foot[torch.arange(len(p), device=p.device), k], at)
        # the winding number, as the sum of solid angles
        a, b, c = A - X, B - X, Cc - X
        la, lb, lc = a.norm(dim=-1), b.norm(dim=-1), c.norm(dim=-1)
        w = torch.atan2(_dot(a, torch.linalg.cross(b, c)),
                        la * lb * lc + _dot(a, b) * lc + _dot(b, c) * la + _dot(c, a) * lb)
        inside = w.sum(1) / (2.0 * math.pi) > 0.5
        sd.append(torch.where(inside, -best.sqrt(), best.sqrt()))
        cps.append(at)
    return torch.cat(sd), torch.cat(cps)


def _net64(net: SdfSurrogate, body: int, p: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """One network's output (without its halfExtent) for float64 points and
    the flat float64 parameters w."""
    _, freq, frame = net.params()
    fr = torch.from_numpy(frame[body].astype(np.float64)).cuda()
    t = ((p - fr[:3]) / fr[3]) @ torch.from_numpy(freq[body].astype(np.float64)).cuda().T
    h = torch.cat([torch.sin(2 * math.pi * t), torch.cos(2 * math.pi * t)], 1)
    at = 0
    for i, o in ((32, 64), (64, 64), (64, 64)):
        W, b = w[at:at + i * o].reshape(i, o), w[at + i * o:at + i * o + o]
        h = torch.nn.functional.silu(h @ W + b)
        at += i * o + o
    return h @ w[at:at + 64] + w[at + 64]


def exact(case: dict, seed: int):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind in ("update", "run", "stages"):
        P = s["params"] if kind == "stages" else s["ps"].m_params
        pos, vel = _steps64(s["pos"].clone(), s["vel"].clone(), P, case.get("steps", 1),
                            _map64(s["map"]) if "map" in s else None, bool(case.get("knot")))
        # long runs amplify every rounding: their velocities have no value
        # that another arithmetic would give
        out = dict(pos=pos, vel=vel if case.get("steps", 1) <= 5 else None)
        if kind == "stages":
            out.update({k: None for k in ("sortedPos", "sortedVel", "hash", "index",
                                          "cellStart", "cellEnd")})
        return out
    if kind == "batch":
        b = s["batch"]
        pos, vel = (torch.from_numpy(b.get_array(k)).cuda() for k in (0, 1))
        ps = b.get_params()
        scene = torch.repeat_interleave(torch.arange(b.num_scenes),
                                        torch.from_numpy(np.diff(b.offsets.astype(np.int64))))
        scene = scene.cuda()

        def per_scene(name):
            return torch.tensor([getattr(p, name) for p in ps], dtype=torch.float64,
                                device="cuda")[scene]

        pos, _ = _steps64(pos, vel, ps[0], case["steps"], scene=scene,
                          spring=per_scene("spring"), damping=per_scene("damping"))
        return dict(pos=pos, vel=None)
    if kind == "build":
        sd, cp = _mesh64(*s["mesh"], s["pts"].double())
        # the normal of a lattice vertex is that of its cell's first corner;
        # on the upper faces that is another vertex
        m = case["cells"] + 1
        nrm = (s["pts"].double() - cp).reshape(m, m, m, 3)
        i = torch.arange(m, device="cuda").clamp(max=m - 2)
        return dict(dist=sd, cp=cp, normal=nrm[i][:, i][:, :, i].reshape(-1, 3))
    if kind == "labels":
        sd, cp = _mesh64(*s["mesh"], torch.from_numpy(s["pts"]).cuda())
        return dict(sdf=sd, cp=cp)
    if kind == "query":
        _, d, p, nrm = _query64(_map64(s["map"]), s["pts"].double())
        return dict(dist=d, cp=p, normal=nrm)
    net = s["net"]
    params = torch.from_numpy(net.params()[0].astype(np.float64))[:, :net.nparams].cuda()
    half = net.params()[2][:, 3].astype(np.float64)
    if kind == "grad":
        p, y = (torch.from_numpy(a.astype(np.float64)).cuda() for a in _samples(case, seed))
        grads, losses = [], []
        for b in range(case["bodies"]):
            at = slice(b * case["samples"], (b + 1) * case["samples"])
            w = params[b].clone().requires_grad_(True)
            loss = ((_net64(net, b, p[at], w) - y[at] / half[b]) ** 2).mean()
            loss.backward()
            grads.append(w.grad)
            losses.append(loss.detach())
        return dict(grad=torch.stack(grads), loss=torch.stack(losses))
    out = torch.empty(case["n"], dtype=torch.float64, device="cuda")
    for b in range(case["bodies"]):
        m = s["of"] == b
        out[m] = _net64(net, b, s["pts"][m].double(), params[b]) * half[b]
    return out
