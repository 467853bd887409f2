"""The calls a program makes into this framework, over the range of their sizes.

Each case is one call (or the few calls that belong together) through the public
entry points: World.step on single and batched scenes, the grid and
sweep-and-prune pair searches over device AABBs, the sort / bound-search / scan
primitives, and the warm-start network's forward, gradients and training.

A step starts from a given body state (a simulation reset to a state and stepped,
as planners and reinforcement-learning loops do), so every pass steps the same
state: the state is written into the world's device arrays, then one step runs
from the captured graph.  The states are resting contact: cubes in columns,
hulls in loose packings a few layers deep, cubes on a terrain, with small
velocities, since a settled pile is what a simulation spends its time on.
"""
import ctypes
import math

import numpy as np
import torch

from experiments_amd import _lib as L
from experiments_amd import scenes
from experiments_amd.warmstart import Mlp, load_weights
from experiments_amd.world import World, reference_config


def listed():
    return [
        # a handful of bodies in one world, stepped every frame: launch latency
        dict(name="step_lattice_48", kind="lattice", nx=4, ny=3, nz=4, iters=4),
        # 4,096 unit cubes in columns on a ground box
        dict(name="step_lattice_4096", kind="lattice", nx=16, ny=16, nz=16, iters=8),
        # one large world: 65,536 hulls of 8 to 32 vertices on a ground box
        dict(name="step_hulls_65536", kind="hulls", n=65536, iters=10),
        # thousands of small piles stepped together (learning environments)
        dict(name="step_piles_4096", kind="piles", scenes=4096, lo=8, hi=512, iters=10, tol=0.0, warm=0),
        # fewer piles, each solved to a residual from the previous impulses
        # (how the warm start's training data are made)
        dict(name="step_piles_256_tol", kind="piles", scenes=256, lo=8, hi=128, iters=256, tol=1e-3, warm=1),
        # cubes on a concave triangle mesh (the demo's ground)
        dict(name="step_terrain_4096", kind="terrain", n=4096, quads=100, iters=8),
        # a million boxes of mixed sizes through the grid search
        dict(name="grid_1048576", kind="grid", n=1048576, levels=4),
        # the AABBs of a large scene through sweep and prune, a ground among them
        dict(name="sap_65537", kind="sap", n=65537, axis=0),
        # cell lists: sort (cell, item), count each cell's items, scan the counts
        dict(name="cells_1000003", kind="cells", n=1000003, bits=18),
        # warm-start network over all contacts of a large batched step
        dict(name="mlp_forward_582217", kind="mlp_forward", n=582217),
        # its gradients over a small batch, and training steps on large ones
        dict(name="mlp_gradients_5000", kind="mlp_gradients", n=5000),
        dict(name="mlp_train_65536", kind="mlp_train", samples=1 << 20, batch=65536, steps=8),
    ]


def _size(rng, lo, hi):
    """Log-uniform in [lo, hi], odd sizes as likely as any."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["lattice", "hulls", "piles", "piles", "terrain", "grid", "sap", "cells",
                       "mlp_forward", "mlp_gradients", "mlp_train"])
    if kind == "lattice":
        return dict(kind=kind, nx=rng.randint(2, 18), ny=rng.randint(1, 16), nz=rng.randint(2, 16),
                    iters=rng.randint(4, 10))
    if kind == "hulls":
        return dict(kind=kind, n=_size(rng, 100, 65536), iters=rng.randint(4, 10))
    if kind == "piles":
        if rng.random() < 0.3:
            return dict(kind=kind, scenes=_size(rng, 2, 256), lo=rng.randint(4, 12),
                        hi=rng.randint(32, 128), iters=256, tol=1e-3, warm=rng.choice([0, 1]))
        return dict(kind=kind, scenes=_size(rng, 2, 2048), lo=rng.randint(4, 12),
                    hi=rng.randint(32, 512), iters=rng.randint(4, 10), tol=0.0, warm=0)
    if kind == "terrain":
        return dict(kind=kind, n=_size(rng, 16, 4096), quads=rng.randint(20, 100),
                    iters=rng.randint(4, 8))
    if kind == "grid":
        return dict(kind=kind, n=_size(rng, 1000, 1000000), levels=4)
    if kind == "sap":
        return dict(kind=kind, n=_size(rng, 500, 65000), axis=rng.choice([0, 2]))
    if kind == "cells":
        return dict(kind=kind, n=_size(rng, 500, 4000000), bits=rng.randint(8, 20))
    if kind == "mlp_forward":
        return dict(kind=kind, n=_size(rng, 1, 1000000))
    if kind == "mlp_gradients":
        return dict(kind=kind, n=_size(rng, 1, 100000))
    return dict(kind="mlp_train", samples=_size(rng, 200000, 1000000), batch=_size(rng, 64, 65536),
                steps=rng.randint(1, 8))


# ---------------------------------------------------------------- worlds

def _quats(rng, n, angle=None):
    """Uniform rotations, or rotations of about `angle` around random axes."""
    if angle is None:
        q = rng.normal(size=(n, 4))
    else:
        q = np.concatenate([0.5 * angle * rng.normal(size=(n, 3)), np.ones((n, 1))], 1)
    return (q / np.linalg.norm(q, axis=1, keepdims=True)).astype(np.float32)


def _hull_points(rng, nverts):
    """nverts points on a sphere of radius U[0.5, 1]."""
    v = rng.normal(size=(nverts, 3))
    v *= (0.5 + 0.5 * rng.random()) / np.linalg.norm(v, axis=1, keepdims=True)
    return v.astype(np.float32)


def _lattice_state(case, rng):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    j, k, i = [a.reshape(-1) for a in np.meshgrid(np.arange(ny), np.arange(nz), np.arange(nx),
                                                  indexing="ij")]
    n = nx * ny * nz
    pos = np.stack([(i - (nx - 1) / 2.0) * 1.05, 0.495 + 0.993 * j, (k - (nz - 1) / 2.0) * 1.05], 1)
    pos += rng.uniform(-1, 1, (n, 3)) * np.array([0.01, 0.002, 0.01])
    half = 0.6 * max(nx, nz) + 10.0
    shapes = [scenes.cube_points(0.5), scenes.box_points(half, 1.0, half)]
    return dict(shapes=shapes, pos=pos, quat=_quats(rng, n, 0.003), shape=np.zeros(n, np.int64),
                mass=np.ones(n), scene=np.zeros(n, np.int64), ground=[(0, 1)])


def _hulls_state(case, rng):
    n = case["n"]
    layers = min(10, max(1, int(round(n ** (1 / 3.0)))))
    m = int(math.ceil(math.sqrt(n / layers)))
    s = 1.42
    b = np.arange(n)
    layer, cell = b // (m * m), b % (m * m)
    pos = np.stack([(cell % m - (m - 1) / 2.0) * s, 0.65 + layer * 1.36,
                    (cell // m - (m - 1) / 2.0) * s], 1)
    pos += rng.uniform(-0.12, 0.12, (n, 3))
    half = 0.5 * s * m + 10.0
    pool = 256
    shapes = ([scenes.cube_points(0.5)] + [_hull_points(rng, 8) for _ in range(pool)] +
              [_hull_points(rng, 32) for _ in range(pool)] + [scenes.box_points(half, 1.0, half)])
    kind = b % 3
    shape = np.where(kind == 0, 0, np.where(kind == 1, 1 + (b // 3) % pool, 1 + pool + (b // 3) % pool))
    return dict(shapes=shapes, pos=pos, quat=_quats(rng, n), shape=shape,
                mass=rng.uniform(1, 10, n), scene=np.zeros(n, np.int64),
                ground=[(0, len(shapes) - 1)])


def _pile_counts(case):
    """Bodies per scene, log-uniform over the scenes."""
    u = (np.arange(case["scenes"]) + 0.5) / case["scenes"]
    return (case["lo"] * (case["hi"] / case["lo"]) ** u).astype(np.int64)


def _piles_state(case, rng):
    ns, pool = case["scenes"], 256
    cnt = _pile_counts(case)[rng.permutation(ns)]
    scene = np.repeat(np.arange(ns), cnt)
    n = len(scene)
    b = np.arange(n) - np.repeat(np.cumsum(cnt) - cnt, cnt)
    m = np.minimum(8, np.ceil(np.sqrt(cnt))).astype(np.int64)[scene]
    layer, cell = b // (m * m), b % (m * m)
    s = 1.33
    pos = np.stack([(cell % m - (m - 1) / 2.0) * s, 0.6 + layer * 1.24,
                    (cell // m - (m - 1) / 2.0) * s], 1)
    pos += rng.uniform(-0.1, 0.1, (n, 3))
    shapes = ([scenes.cube_points(0.5)] + [_hull_points(rng, 8) for _ in range(pool)] +
              [scenes.box_points(30.0, 1.0, 30.0)])
    shape = np.where(b % 2 == 0, 0, 1 + (np.arange(n) // 2) % pool)
    return dict(shapes=shapes, pos=pos, quat=_quats(rng, n), shape=shape, mass=np.ones(n),
                scene=scene, ground=[(sc, len(shapes) - 1) for sc in range(ns)])


def _terrain_state(case, rng):
    n, quads = case["n"], case["quads"]
    m = int(math.ceil(math.sqrt(n)))
    half = 0.75 * m + 2.0
    height = lambda x, z: 0.2 * np.sin(0.3 * x) * np.cos(0.25 * z)  # noqa: E731
    b = np.arange(n)
    x, z = (b % m - (m - 1) / 2.0) * 1.5, (b // m - (m - 1) / 2.0) * 1.5
    x, z = x + rng.uniform(-0.1, 0.1, n), z + rng.uniform(-0.1, 0.1, n)
    pos = np.stack([x, height(x, z) + 0.5 + rng.uniform(-0.02, 0.005, n), z], 1)
    g = np.linspace(-half, half, quads + 1)
    gx, gz = [a.reshape(-1) for a in np.meshgrid(g, g, indexing="ij")]
    i, j = [a.reshape(-1) for a in np.meshgrid(np.arange(quads), np.arange(quads), indexing="ij")]
    a = i * (quads + 1) + j
    bb, c, d = a + 1, a + quads + 2, a + quads + 1
    tris = np.stack([np.stack([a, bb, c], 1), np.stack([a, c, d], 1)], 1).reshape(-1, 3)
    mesh = (np.stack([gx, height(gx, gz), gz], 1).astype(np.float32), tris.astype(np.int32))
    return dict(shapes=[scenes.cube_points(0.5)], mesh=mesh, pos=pos, quat=_quats(rng, n, 0.05),
                shape=np.zeros(n, np.int64), mass=np.ones(n), scene=np.zeros(n, np.int64),
                ground=[(0, "mesh")])


_STATES = dict(lattice=_lattice_state, hulls=_hulls_state, piles=_piles_state,
               terrain=_terrain_state)


class _DeviceArray:
    """One of a world's device arrays (mi_rb_device_ptrs) for torch.  A tensor
    made from it keeps it, and it keeps the world, which frees the memory when
    it goes."""

    def __init__(self, world, ptr, shape):
        self.world = world
        self.__cuda_array_interface__ = dict(shape=shape, typestr="<f4", data=(ptr, False), version=2)


def _prepare_world(case, seed):
    torch.cuda.init()
    rng = np.random.default_rng(seed)
    st = _STATES[case["kind"]](case, rng)
    n = len(st["pos"]) + len(st["ground"])
    tris = len(st["mesh"][1]) if "mesh" in st else 0
    w = World(reference_config(
        max_bodies=max(n, 16), max_shapes=len(st["shapes"]) + tris + 2,
        max_hull_vertices=max(1 << 16, 40 * len(st["shapes"]) + 3 * tris),
        max_pairs=max(1 << 16, 16 * n), max_contacts=max(1 << 16, 6 * n), max_pairs_per_body=64,
        dt=1.0 / 60.0, solver_dt=1.0 / 60.0, solver_iterations=case["iters"],
        residual_tolerance=case.get("tol", 0.0), warm_start=case.get("warm", 0)))
    for pts in st["shapes"]:
        w.add_hull(pts)
    mesh = w.add_concave_mesh(*st["mesh"]) if tris else None
    # bodies scene by scene, each scene's ground first (at y = -1, top at 0; a
    # mesh at the origin)
    pos = np.ascontiguousarray(st["pos"], np.float32)
    quat, shape, mass, scene = st["quat"], st["shape"].tolist(), st["mass"].tolist(), st["scene"]
    starts = np.searchsorted(scene, np.arange(len(st["ground"]) + 1)).tolist()
    add, h, out = L.lib().mi_rb_register_body, w.h, ctypes.c_int()
    ref, pp, qp = ctypes.byref(out), pos.ctypes.data, quat.ctypes.data
    vel = []
    for (sc, g), lo, hi in zip(st["ground"], starts[:-1], starts[1:]):
        w.add_body(0.0, (0, 0, 0) if g == "mesh" else (0, -1, 0), (0, 0, 0, 1),
                   mesh if g == "mesh" else g, sc)
        vel.append(np.zeros((1, 8), np.float32))
        for b in range(lo, hi):
            L.check("mi_rb_register_body", add(h, mass[b], pp + 12 * b, qp + 16 * b, shape[b], sc, ref))
        v = np.zeros((hi - lo, 8), np.float32)
        v[:, 0:3] = 0.1 * rng.normal(size=(hi - lo, 3))
        v[:, 4:7] = 0.1 * rng.normal(size=(hi - lo, 3))
        vel.append(v)
    w.upload()
    vel = np.concatenate(vel)
    w.set_state(linvel=vel[:, :4], angvel=vel[:, 4:])
    w.use_graph(True)
    v = L.DeviceView()
    L.call("mi_rb_device_ptrs", w.h, ctypes.byref(v))
    now = [torch.as_tensor(_DeviceArray(w, p, (n, 4)), device="cuda")
           for p in (v.pos, v.quat, v.linvel, v.angvel)]
    return dict(world=w, now=now, start=[t.clone() for t in now],
                stream=torch.cuda.ExternalStream(v.stream))


def _run_world(s):
    with torch.cuda.stream(s["stream"]):
        for t, t0 in zip(s["now"], s["start"]):
            t.copy_(t0)
    s["world"].step(1)
    return dict(zip(("pos", "quat", "linvel", "angvel"), s["now"]))


def _bodies(case):
    if case["kind"] == "lattice":
        return case["nx"] * case["ny"] * case["nz"]
    if case["kind"] == "piles":
        return int(_pile_counts(case).sum())
    return case["n"]


def _work_world(case):
    n = _bodies(case)
    # state in and out, mass, inertia, shape and scene; about one and a half
    # manifolds a body, each point about 70 operations a normal sweep and each
    # tangent about 100 a friction sweep, 15 sweeps of a tolerance solve; about
    # 5,000 operations a manifold to find it
    sweeps = 15 if case.get("tol", 0.0) > 0 else case["iters"]
    tris = 2 * case["quads"] ** 2 * 60 if case["kind"] == "terrain" else 0
    return dict(bytes=n * (64 + 64 + 28) + tris, flops=1.5 * n * (sweeps * (4 * 70 + 2 * 100) + 5000))


# ---------------------------------------------------------------- pair searches

class _Handle:
    """A C handle and the call that frees it."""

    def __init__(self, create, destroy, *args):
        self.h = ctypes.c_void_p()
        self.destroy = destroy
        L.call(create, *args, ctypes.byref(self.h))

    def __del__(self):
        if self.h:
            getattr(L.lib(), self.destroy)(self.h)


def _vp(t):
    return ctypes.c_void_p(t.data_ptr())


def _generator(seed):
    torch.cuda.init()
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _aabbs(gen, n, box, rmin, rmax):
    """Half spheres and half boxes' bounds: radius log-uniform in [rmin, rmax],
    centres uniform in a box^3 domain."""
    u = torch.rand((n, 8), generator=gen, device="cuda")
    r = torch.exp(math.log(rmin) + u[:, 0] * math.log(rmax / rmin))
    stretch = torch.where(u[:, 1:2] < 0.5, 1.0, 1.0 + 0.7 * u[:, 5:8])
    c = (u[:, 2:5] - 0.5) * box
    mn = torch.zeros((n, 4), device="cuda")
    mx = torch.zeros((n, 4), device="cuda")
    mn[:, :3], mx[:, :3] = c - r[:, None] * stretch, c + r[:, None] * stretch
    return mn, mx


def _prepare_grid(case, seed):
    n = case["n"]
    # the density of a million bodies in a 400^3 domain, radii in [0.25, 2]
    mn, mx = _aabbs(_generator(seed), n, 400.0 * (n / 1048576.0) ** (1 / 3.0), 0.25, 2.0)
    side = 8
    while side < 256 and side * 1.414 < 400.0 * (n / 1048576.0) ** (1 / 3.0):
        side *= 2
    cap = max(1 << 14, 8 * n)
    desc = L.GridDesc(1.414, (ctypes.c_int * 3)(side, side, side), cap, 1, case["levels"])
    h = _Handle("mi_rb_grid_create", "mi_rb_grid_destroy", ctypes.byref(desc), n)
    return dict(h=h, mn=mn, mx=mx, n=n, call="mi_rb_grid_find_pairs", large=None,
                pairs=torch.zeros((cap, 2), dtype=torch.int32, device="cuda"),
                num=torch.zeros(1, dtype=torch.int32, device="cuda"))


def _prepare_sap(case, seed):
    n = case["n"]
    # a layer of bodies about ten deep on a ground box, the last AABB
    gen = _generator(seed)
    side = 1.45 * math.sqrt(n / 10.0)
    mn, mx = _aabbs(gen, n, 1.0, 0.5, 1.0)
    c = (torch.rand((n, 3), generator=gen, device="cuda") - 0.5) * torch.tensor(
        [side, 13.0, side], device="cuda")
    c = c - 0.5 * (mn + mx)[:, :3]
    mn[:, :3] += c
    mx[:, :3] += c
    mn[-1, :3] = torch.tensor([-side, -8.5, -side], device="cuda")
    mx[-1, :3] = torch.tensor([side, -6.5, side], device="cuda")
    large = torch.zeros(n, dtype=torch.int32, device="cuda")
    large[-1] = 1
    cap = max(1 << 14, 24 * n)
    desc = L.SapDesc(case["axis"], cap)
    h = _Handle("mi_rb_sap_create", "mi_rb_sap_destroy", ctypes.byref(desc), n)
    return dict(h=h, mn=mn, mx=mx, n=n, call="mi_rb_sap_find_pairs", large=large,
                pairs=torch.zeros((cap, 2), dtype=torch.int32, device="cuda"),
                num=torch.zeros(1, dtype=torch.int32, device="cuda"))


def _run_pairs(s):
    L.call(s["call"], s["h"].h, _vp(s["mn"]), _vp(s["mx"]),
           None if s["large"] is None else _vp(s["large"]), s["n"], _vp(s["pairs"]), _vp(s["num"]),
           None)
    return dict(pairs=s["pairs"], num=s["num"])


# ---------------------------------------------------------------- primitives

def _prepare_cells(case, seed):
    n, bits = case["n"], case["bits"]
    gen = _generator(seed)
    kv = torch.empty((n, 2), dtype=torch.int32, device="cuda")
    kv[:, 0] = torch.randint(0, 1 << bits, (n,), generator=gen, device="cuda", dtype=torch.int32)
    kv[:, 1] = torch.arange(n, device="cuda", dtype=torch.int32)
    cells = 1 << bits
    return dict(h=_Handle("mi_rb_radix_sort_create", "mi_rb_radix_sort_destroy", max(n, cells)),
                kv=kv, sorted=torch.empty_like(kv), n=n, bits=bits, cells=cells,
                counts=torch.zeros(cells, dtype=torch.int32, device="cuda"),
                offsets=torch.zeros(cells, dtype=torch.int32, device="cuda"),
                total=torch.zeros(1, dtype=torch.int32, device="cuda"))


def _run_cells(s):
    s["sorted"].copy_(s["kv"])  # the sort is in place
    L.call("mi_rb_radix_sort_kv", s["h"].h, _vp(s["sorted"]), s["n"], s["bits"], None)
    L.call("mi_rb_bound_search", _vp(s["sorted"]), s["n"], _vp(s["counts"]), s["cells"], 2, None)
    L.call("mi_rb_exclusive_scan_u32", s["h"].h, _vp(s["counts"]), _vp(s["offsets"]), s["cells"],
           _vp(s["total"]), None)
    return dict(sorted=s["sorted"], counts=s["counts"], offsets=s["offsets"], total=s["total"])


# ---------------------------------------------------------------- the network

def _contact_rows(gen, n):
    """Features of n contacts as the constraint setup writes them, and the
    impulses (network units) they lead to."""
    u = torch.rand((n, 12), generator=gen, device="cuda")
    g = torch.randn((n, 8), generator=gen, device="cuda")
    x = torch.zeros((n, 16), device="cuda")
    nrm = g[:, 0:3] * 0.5
    nrm[:, 1] += 1.0
    x[:, 0:3] = nrm / nrm.norm(dim=1, keepdim=True)
    x[:, 3] = 0.2 - 0.6 * u[:, 0]
    x[:, 4:7] = 0.3 * g[:, 3:6]
    x[:, 7] = 1.0 / (1.0 + 9.0 * u[:, 1])
    x[:, 8] = torch.where(u[:, 2] < 0.1, 0.0, 1.0 / (1.0 + 9.0 * u[:, 3]))
    has = (u[:, 4] < 0.8).float()
    x[:, 9] = has * 3.0 * u[:, 5] * u[:, 6]
    x[:, 10] = has * 0.5 * g[:, 6] * u[:, 5]
    x[:, 11] = has * 0.5 * g[:, 7] * u[:, 5]
    x[:, 12] = torch.ceil(4.0 * u[:, 7]).clamp(1, 4) * 0.25
    x[:, 13] = has
    x[:, 14] = 1.0 + 2.0 * u[:, 8]
    x[:, 15] = 0.6 * u[:, 9]
    t = torch.stack([x[:, 9] * (0.9 + 0.2 * u[:, 10]) + (1 - has) * u[:, 11],
                     x[:, 10] * 0.95, x[:, 11] * 0.95], 1).contiguous()
    return x, t


def _prepare_mlp(case, seed):
    gen = _generator(seed)
    net = Mlp(seed=1 + seed % 1000)
    w0 = net.get_weights() if case["kind"] == "mlp_train" else load_weights()
    net.set_weights(*w0)
    x, t = _contact_rows(gen, case.get("samples", case.get("n")))
    return dict(kind=case["kind"], net=net, w0=w0, x=x, t=t, case=dict(case), seed=seed % 1000)


def _run_mlp(s):
    net, c = s["net"], s["case"]
    if s["kind"] == "mlp_forward":
        return dict(y=net.forward(s["x"]))
    if s["kind"] == "mlp_gradients":
        g, loss = net.gradients(s["x"], s["t"])
        return dict(gradients=g, loss=loss)
    net.set_weights(*s["w0"])
    loss = net.train(s["x"], s["t"], c["batch"], c["steps"], 2e-3, s["seed"])
    w, b = net.get_weights()
    return dict(weights=torch.from_numpy(w.view(np.int16)).view(torch.bfloat16), biases=b, loss=loss)


def _exact_mlp(case, seed):
    """The network in 64 bits: inputs and hidden activations rounded to
    bfloat16 (its definition), everything else in double."""
    if case["kind"] == "mlp_train":
        return None  # the minibatches are the library's own draws
    s = _prepare_mlp(case, seed)
    w16, bias = s["w0"]
    w = torch.from_numpy(w16.astype(np.int32) << 16).view(torch.float32).double().cuda()
    b = torch.from_numpy(bias).double().cuda()
    w1, w2, w3 = w[:1024].view(64, 16), w[1024:5120].view(64, 64), w[5120:].view(3, 64)
    b1, b2, b3 = b[:64], b[64:128], b[128:]
    r16 = lambda v: v.float().bfloat16().double()  # noqa: E731
    x, t = r16(s["x"]), s["t"].double()
    a1 = (x @ w1.T + b1).relu()
    h1 = r16(a1)
    a2 = (h1 @ w2.T + b2).relu()
    h2 = r16(a2)
    y = h2 @ w3.T + b3
    if case["kind"] == "mlp_forward":
        return dict(y=y)
    e = y - t
    dy = 2.0 * e / (3.0 * len(x))
    d2 = (dy @ w3) * (a2 > 0)
    d1 = (d2 @ w2) * (a1 > 0)
    g = torch.cat([(d1.T @ x).reshape(-1), (d2.T @ h1).reshape(-1), (dy.T @ h2).reshape(-1),
                   d1.sum(0), d2.sum(0), dy.sum(0)])
    return dict(gradients=g, loss=float((e * e).sum() / (3.0 * len(x))))


# ---------------------------------------------------------------- the module's functions

def prepare(case, seed):
    kind = case["kind"]
    if kind in _STATES:
        return _prepare_world(case, seed)
    if kind == "grid":
        return _prepare_grid(case, seed)
    if kind == "sap":
        return _prepare_sap(case, seed)
    if kind == "cells":
        return _prepare_cells(case, seed)
    return _prepare_mlp(case, seed)


def run(state):
    if "world" in state:
        return _run_world(state)
    if "call" in state:
        return _run_pairs(state)
    if "cells" in state:
        return _run_cells(state)
    return _run_mlp(state)


def work(case):
    kind = case["kind"]
    if kind in _STATES:
        return _work_world(case)
    if kind in ("grid", "sap"):
        # boxes in, about two (grid) or eight (layered scene) pairs a body out
        pairs = 2 if kind == "grid" else 8
        return dict(bytes=case["n"] * (32 + 8 * pairs), flops=case["n"] * 27 * 6)
    if kind == "cells":
        # pairs in and out, counts and offsets out
        return dict(bytes=16 * case["n"] + 8 * (1 << case["bits"]), flops=0)
    ops = 2 * 5312
    if kind == "mlp_forward":
        return dict(bytes=case["n"] * 76, flops=case["n"] * ops)
    if kind == "mlp_gradients":
        return dict(bytes=case["n"] * 76 + 5443 * 4, flops=3 * case["n"] * ops)
    return dict(bytes=case["steps"] * case["batch"] * 76, flops=3 * case["steps"] * case["batch"] * ops)


def exact(case, seed):
    return _exact_mlp(case, seed) if case["kind"].startswith("mlp") else None
