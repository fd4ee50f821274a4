"""Workloads that programs built on this framework run, as timeable cases.

A case is a dict of plain values.  prepare() makes what the program holds
before the call (the simulation or batch it advances, the points it meshes,
the mesh it trains or updates on), run() is one pass through the public entry
points with its outputs, work() the bytes and floating-point operations the
pass cannot do without, exact() the outputs that plain torch gives in 64 bits.

Simulations and batches are advanced by a pass (a snapshot interval: a few
steps, then the state is fetched), so their later passes continue the run.
"""
import ctypes as C
import math

import numpy as np
import torch

from proteusgpu_amd import _native, api
from proteusgpu_amd.generators import (batch_points, box_sizes, gaussian_mixture, jittered_lattice,
                                       kelvin_helmholtz_state, sod_state, uniform_points)

_ctx = None


def _context():
    """The program's one context (one GPU, one stream)."""
    global _ctx
    if _ctx is None:
        _ctx = api.Context(0)
    return _ctx


def listed():
    return [
        # smallest runs: a shear-layer box of a few thousand cells, where launches
        # and host round trips are the step
        dict(name="sim_kh2d_2k", kind="sim", dim=2, n=2000, setup="kh", boundary="periodic", buff=0.1, k=16,
             move="regularized", flux="physical", steps=8),
        # the 2D Sod tube: 10,000 uniform generators, 20 moving steps
        dict(name="sim_sod2d_10k", kind="sim", dim=2, n=10000, setup="sod", boundary="reflective", buff=0.04, k=16,
             move="regularized", flux="physical", steps=20),
        # a small 3D run of an odd size
        dict(name="sim_sod3d_20k", kind="sim", dim=3, n=20011, setup="sod", boundary="reflective", buff=0.04, k=32,
             move="regularized", flux="physical", steps=5),
        # the plain method at full size: fixed k = 32 with certificate restarts,
        # host-driven step, mesh moving with the fluid
        dict(name="sim_sod3d_1m", kind="sim", dim=3, n=1000000, setup="sod", boundary="reflective", buff=0.04, k=32,
             move="fluid", flux="physical", steps=4),
        # the benchmark's step: learned k, the whole step one graph launch
        dict(name="batch_sod3d_1m_learned", kind="batch", dim=3, boxes=1, lo=1000000, hi=1000000, setup="sod",
             boundary="reflective", buff=0.04, k=32, move="fluid", learned=True, steps=4),
        # many uneven 2D periodic boxes in one captured step
        dict(name="batch_kh2d_64boxes", kind="batch", dim=2, boxes=64, lo=1000, hi=65536, setup="kh",
             boundary="periodic", buff=0.1, k=16, move="regularized", learned=False, steps=4),
        # the largest: a blast wave on a jittered lattice of 126^3 generators
        dict(name="batch_sedov3d_2m", kind="batch", dim=3, boxes=1, lo=2000376, hi=2000376, setup="sedov",
             boundary="reflective", buff=0.04, k=32, move="regularized", learned=False, steps=3),
        # meshing through the reference's call: points in, the whole VMesh out;
        # clustered points (64 Gaussians and a uniform background, periodic)
        dict(name="mesh_clustered3d_400k", kind="mesh", dim=3, n=400000, points="clustered", boundary="periodic",
             buff=0.04, k=32),
        # the same call on a small uniform 2D set
        dict(name="mesh_uniform2d_10k", kind="mesh", dim=2, n=10000, points="uniform", boundary="periodic", buff=0.04,
             k=16),
        # the static-mesh solver: CFL step and HLL update, ten times, on a 1M mesh
        dict(name="static_sod3d_1m", kind="static", dim=3, n=1000000, boundary="reflective", buff=0.04, k=32,
             flux="physical", steps=10),
        # neighbour lists alone, device arrays in and out
        dict(name="knn_uniform3d_1m", kind="knn", dim=3, n=1000000, points="uniform", k=32),
        # training the k classifier on the seeds of a built mesh
        dict(name="train_k_200k", kind="train", dim=3, n=200000, boundary="reflective", buff=0.04, k=32, steps=400,
             batch=4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges: sizes spread over their logarithm,
    the options the entry points take in use."""
    kind = rng.choice(["sim", "sim", "sim", "batch", "batch", "mesh", "mesh", "static", "knn", "train"])
    dim = rng.choice([2, 3])
    k = rng.choice([16, 20, 24]) if dim == 2 else rng.choice([24, 32, 40, 48, 64])
    periodic = rng.random() < 0.4
    # ghost layers are wider than the cells of the smallest boxes
    buff = 0.1 if dim == 2 else 0.12
    boundary = "periodic" if periodic else "reflective"
    if kind == "sim":
        n = _log_int(rng, 1000, 200000) if dim == 2 else _log_int(rng, 60000 if periodic else 14000, 800000)
        return dict(kind=kind, dim=dim, n=n, setup="kh" if periodic else "sod", boundary=boundary, buff=buff, k=k,
                    move="regularized", flux="physical", steps=rng.randint(2, 8) if n < 100000 else 2)
    if kind == "batch":
        if dim == 2:
            return dict(kind=kind, dim=2, boxes=rng.randint(2, 96), lo=1000, hi=_log_int(rng, 2000, 65536),
                        setup="kh" if periodic else "sod", boundary=boundary, buff=buff, k=k, move="regularized",
                        learned=rng.random() < 0.5, steps=rng.randint(2, 4))
        lo = _log_int(rng, 20000, 200000)
        return dict(kind=kind, dim=3, boxes=rng.randint(1, 3), lo=lo, hi=int(lo * rng.uniform(1.0, 2.0)),
                    setup="sod", boundary="reflective", buff=buff, k=k, move="regularized",
                    learned=rng.random() < 0.5, steps=rng.randint(2, 4))
    if kind == "mesh":
        n = _log_int(rng, 2000, 300000) if dim == 2 else _log_int(rng, 20000, 300000)
        points = "uniform" if dim == 2 else rng.choice(["uniform", "clustered", "lattice"])
        return dict(kind=kind, dim=dim, n=n, points=points, boundary=rng.choice(["periodic", "reflective", "none"]),
                    buff=0.04, k=k)
    if kind == "static":
        n = _log_int(rng, 2000, 300000) if dim == 2 else _log_int(rng, 14000, 800000)
        return dict(kind=kind, dim=dim, n=n, boundary="reflective", buff=buff, k=k,
                    flux=rng.choice(["physical", "reference"]), steps=rng.randint(1, 10))
    if kind == "knn":
        n = _log_int(rng, 1000, 2000000) if dim == 2 else _log_int(rng, 14000, 2000000)
        return dict(kind=kind, dim=dim, n=n, points="uniform", k=rng.choice([8, 16, 24, 32, 48, 64, 96]))
    n = _log_int(rng, 14000, 200000)
    return dict(kind="train", dim=3, n=n, boundary="reflective", buff=0.04, k=32, steps=rng.randint(50, 400),
                batch=rng.choice([1024, 4096, 16384]))


def _points(case, n, seed):
    if case.get("points") == "clustered":
        return gaussian_mixture(n, 64, 0.002, 0.05, 0.2, seed)
    if case.get("points") == "lattice":
        return jittered_lattice(max(2, round(n ** (1.0 / case["dim"]))), case["dim"], seed)
    return uniform_points(n, case["dim"], seed)


def _gamma(case):
    return 1.4 if case.get("setup", "sod") == "sod" else 5.0 / 3.0


def _sedov(n, seed):
    """A blast of unit energy in the 32 cells nearest the centre of a cold gas."""
    m = round(n ** (1.0 / 3.0))
    pts = jittered_lattice(m, 3, seed)
    hot = np.argpartition(np.sum((pts - 0.5) ** 2, axis=1), 32)[:32]
    E = np.full(len(pts), 1e-5 / (5.0 / 3.0 - 1.0))
    E[hot] += len(pts) / 32.0
    return pts, np.ones(len(pts)), np.zeros((len(pts), 3)), E


def _trained(ctx, dim, k, boundary, buff):
    """A classifier trained on another point set of the same workload."""
    km = api.KModel(ctx, seed=1)
    mesh = api.Mesh(ctx, uniform_points(30000, dim, 43), boundary=boundary, buff=buff, k=k)
    km.train_mesh(mesh, steps=200, batch=4096, lr=3e-3)
    mesh.free()
    return km


def prepare(case, seed):
    ctx = _context()
    kind, dim, k = case["kind"], case["dim"], case["k"]
    if kind == "sim":
        pts = uniform_points(case["n"], dim, seed)
        state = sod_state(pts, _gamma(case)) if case["setup"] == "sod" else kelvin_helmholtz_state(pts)
        sim = api.Simulation(ctx, pts, *state, boundary=case["boundary"], buff=case["buff"], k=k, gamma=_gamma(case),
                             cfl=0.3, flux=case["flux"], move_mesh=case["move"])
        return dict(kind=kind, sim=sim, steps=case["steps"])
    if kind == "batch":
        km = None
        if case["setup"] == "sedov":
            pts, *state = _sedov(case["lo"], seed)
            sizes = np.array([len(pts)])
        else:
            sizes = box_sizes(case["boxes"], case["lo"], case["hi"], 11)
            pts = batch_points(sizes, dim, seed + 1000)
            state = sod_state(pts, _gamma(case)) if case["setup"] == "sod" else kelvin_helmholtz_state(pts)
        b = api.Batch(ctx, sizes, pts, *state, boundary=case["boundary"], buff=case["buff"], k=k, gamma=_gamma(case),
                      cfl=0.3, flux="physical", move_mesh=case["move"])
        if case["learned"]:
            km = _trained(ctx, dim, k, case["boundary"], case["buff"])
            b.set_kmodel(km)
        return dict(kind=kind, batch=b, km=km, steps=case["steps"])
    if kind == "mesh":
        # the program's own VMesh arrays, with room for ghosts and faces
        ns = int(case["n"] * (1.5 if case["boundary"] == "periodic" else 1.05)) + 1000
        nf = ns * (16 if dim == 3 else 7)
        out = {"cell_ids": np.zeros(ns, np.int64), "seeds": np.zeros((ns, 3)), "volumes": np.zeros(ns),
               "face_counts": np.zeros(ns, np.int64), "face_ptr": np.zeros(ns, np.int64),
               "neighbor_cell": np.zeros(nf, np.int32), "face_normal": np.zeros((nf, 3)), "face_area": np.zeros(nf),
               "ghost_ids": np.zeros(ns, np.int64), "status": np.zeros(ns, np.int32), "kcert": np.zeros(ns, np.int32),
               "cell_centroid": np.zeros((ns, 3)), "face_centroid": np.zeros((nf, 3))}
        view = _native.VMeshView()
        for name, a in out.items():
            setattr(view, name, a.ctypes.data)
        return dict(kind=kind, pts=_points(case, case["n"], seed), boundary=case["boundary"], buff=case["buff"], k=k,
                    out=out, view=view, ns=ns, nf=nf)
    if kind == "static":
        pts = uniform_points(case["n"], dim, seed)
        mesh = api.Mesh(ctx, pts, boundary=case["boundary"], buff=case["buff"], k=k)
        st = api.HydroState(ctx, mesh, *sod_state(pts, 1.4))
        return dict(kind=kind, mesh=mesh, st=st, flux=case["flux"], steps=case["steps"])
    if kind == "knn":
        n = case["n"]
        dev = torch.device("cuda", 0)
        pts = torch.from_numpy(_points(case, n, seed)).to(dev)
        return dict(kind=kind, pts=pts, k=k, sorted=torch.empty_like(pts),
                    perm=torch.empty(n, dtype=torch.int32, device=dev),
                    rows=torch.empty((n, k), dtype=torch.int32, device=dev))
    if kind == "train":
        mesh = api.Mesh(ctx, uniform_points(case["n"], dim, seed), boundary=case["boundary"], buff=case["buff"], k=k)
        return dict(kind=kind, mesh=mesh, km=api.KModel(ctx, seed=seed + 1), steps=case["steps"], batch=case["batch"])
    raise ValueError(kind)


def run(s):
    ctx, kind = _context(), s["kind"]
    if kind == "sim":
        # a snapshot interval: moving-mesh steps (a full rebuild each), then the state
        dt = [s["sim"].step() for _ in range(s["steps"])]
        return dict(zip(("x", "rho", "vel", "E"), s["sim"].get()), dt=np.array(dt))
    if kind == "batch":
        for _ in range(s["steps"]):
            s["batch"].step()
        return dict(zip(("x", "rho", "vel", "E"), s["batch"].get()), dt=s["batch"].dt())
    if kind == "mesh":
        m = api.Mesh(ctx, s["pts"], boundary=s["boundary"], buff=s["buff"], k=s["k"])
        if m.n_seeds > s["ns"] or m.num_faces > s["nf"]:
            raise ValueError("the mesh is larger than the program's arrays")
        _native.check(_native.lib().pg_mesh_copy_out(ctx.h, m.h, C.byref(s["view"])))
        counts = dict(n_seeds=m.n_seeds, num_faces=m.num_faces, n_failed=m.n_failed)
        m.free()
        return dict(s["out"], **counts)
    if kind == "static":
        dt = []
        for _ in range(s["steps"]):
            dt.append(s["st"].dt_cfl(1.4, 0.3))
            s["st"].step(1.4, dt[-1], s["flux"])
        return dict(zip(("rho", "vel", "E"), s["st"].copy_out()), dt=np.array(dt))
    if kind == "knn":
        n, dim = s["pts"].shape
        _native.check(_native.lib().pg_knn_solve_noalloc(ctx.h, dim, s["pts"].data_ptr(), n, s["k"],
                                                         s["sorted"].data_ptr(), s["perm"].data_ptr(),
                                                         s["rows"].data_ptr(), None))
        return dict(sorted=s["sorted"], perm=s["perm"], rows=s["rows"])
    loss = s["km"].train_mesh(s["mesh"], steps=s["steps"], batch=s["batch"], lr=3e-3)
    return dict(params=s["km"].params, loss=np.float32(loss))


def _mesh_flops(dim):
    """Operations of one cell's build: in 3D about 20 planes cut the cell,
    each tested against about 25 vertices (8 operations) and making 7 new
    ones (70 each), then 15.5 faces of 5.2 corners (60 per corner) and the
    distances of about 130 candidate neighbours; in 2D 9 planes, 8 vertices,
    2 new ones (25 each), 6 faces and 40 candidates."""
    return 20 * 25 * 8 + 20 * 7 * 70 + 15.5 * 5.2 * 60 + 130 * 8 if dim == 3 else 9 * 8 * 6 + 9 * 2 * 25 + 6 * 30 + 40 * 5


def _hydro_flops(dim):
    """Operations of one cell's update: half its faces' Riemann problems."""
    return (15.5 if dim == 3 else 6) / 2 * 250 + 60


def work(case):
    kind, dim, k = case["kind"], case["dim"], case["k"]
    state = 8 * (2 * dim + 2)  # position, momentum, mass and energy of a cell
    faces = 15.5 if dim == 3 else 6
    if kind in ("sim", "batch"):
        if kind == "sim":
            n = case["n"]
        elif case["lo"] == case["hi"]:
            n = case["boxes"] * case["lo"]
        else:
            n = case["boxes"] * (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"])
        return dict(bytes=n * state * (2 * case["steps"] + 2), flops=n * case["steps"] * (_mesh_flops(dim) + _hydro_flops(dim)))
    n = case["n"]
    if kind == "mesh":
        # points in; per cell ids, seed, volume, centroid, counts, statuses; per face 60 bytes
        return dict(bytes=n * (8 * dim + 8 * 10 + 8 + faces * 60), flops=n * _mesh_flops(dim))
    if kind == "static":
        # per step the faces (normal, area, neighbour), volumes and the state, read and written
        return dict(bytes=n * case["steps"] * (faces * 36 + 8 + 16 * (dim + 2)) + 8 * n * (dim + 2),
                    flops=n * case["steps"] * (faces * 150 + 40))
    if kind == "knn":
        return dict(bytes=n * (16 * dim + 4 + 4 * k), flops=n * 4 * k * 3 * dim)
    # training: 16-64-64-6 network, forward and backward, 16 features and a label per drawn seed
    return dict(bytes=case["steps"] * (case["batch"] * 68 + 16 * 5638), flops=case["steps"] * case["batch"] * 6 * 5504)


def exact(case, seed):
    """The sorted points of the neighbour-list call (a stable sort by grid
    cell); the meshes, states and parameters have no short plain form."""
    if case["kind"] != "knn":
        return None
    n, dim = case["n"], case["dim"]
    pts = torch.from_numpy(_points(case, n, seed))
    N = max(1, int(np.float32((n / 3.1) ** (1.0 / dim)) + np.float32(0.5)))
    c = torch.clamp(torch.floor(pts * N).long(), 0, N - 1)
    cell = c[:, 0] + c[:, 1] * N + (c[:, 2] * N * N if dim == 3 else 0)
    return dict(sorted=pts[torch.argsort(cell, stable=True)], perm=None, rows=None)
