"""The framework's performance cases: the calls a user's program makes, over the range of sizes it makes them.

``listed`` names the cases, ``draw`` gives more of the same ranges, ``prepare`` makes what the program holds before the call
(inputs on the GPU and a context), ``run`` is one pass through the public entry points, ``work`` what a pass cannot do without,
and ``exact`` its outputs in 64 bits where they have a value of their own.

Shapes and sizes are those of the synthetic workloads (sphere 20k at depth 6, torus 200k at depth 7, displaced sphere 2M at depth 9,
ellipsoids and tori of 5k-150k points in batches, requests of 10k-1M points) and of the bunny scan (35,947 points, depth 7).
"""
import ctypes
import importlib
import math

import numpy as np
import torch

pkg = importlib.import_module("poisson-surface-reconstruction-gpu_amd")
binding, synth = pkg.binding, pkg.synth

PRECISION = {"fp32": binding.PRECISION_FP32, "mixed": binding.PRECISION_MIXED}


def reconstruct(shape, points, depth, precision, layout="packed", name=None):
    c = {"path": "reconstruct", "shape": shape, "points": points, "depth": depth, "precision": precision, "layout": layout}
    return {"name": name, **c} if name else c


def listed():
    return [
        # the smallest call: a preview, or the first one of a session (the smoke test's size); launches and waits are all of it
        reconstruct("sphere", 4000, 5, "fp32", name="sphere_4k_d5_fp32"),
        # a small object scan at the depth below the default
        reconstruct("sphere", 20000, 6, "mixed", name="sphere_20k_d6_mixed"),
        # the size and depth of the bunny scan, passed as 64-byte surfel records as the reference's callers hold them
        reconstruct("rotated", 35947, 7, "mixed", layout="surfel", name="scan_36k_d7_mixed_surfel"),
        # the headline workload, in both forms of the solver
        reconstruct("torus", 200000, 7, "mixed", name="torus_200k_d7_mixed"),
        reconstruct("torus", 200000, 7, "fp32", name="torus_200k_d7_fp32"),
        # a large request of the serving stream, an odd size
        reconstruct("rotated", 300007, 8, "mixed", name="request_300k_d8_mixed"),
        # the largest: a dense scan at the greatest depth
        reconstruct("displaced", 2000000, 9, "mixed", name="displaced_2m_d9_mixed"),
        # many uneven clouds in one call, as the server makes it (the plan whose meshes equal the single calls')
        {"name": "batch_32_d7_mixed", "path": "batch", "clouds": 32, "lo": 5000, "hi": 150000, "depth": 7, "precision": "mixed"},
        # the step before a reconstruction, for a scan that comes without normals
        {"name": "normals_200k_k10", "path": "point_normals", "shape": "torus", "points": 200000, "k": 10, "knn": False},
        # the steps after it: one vertex per edge crossing, normals to shade it, colours of the scanned points
        {"name": "weld_200k_d7", "path": "weld", "shape": "torus", "points": 200000, "depth": 7},
        {"name": "mesh_normals_28k", "path": "mesh_normals", "rows": 213, "columns": 131},
        {"name": "colors_28k_from_200k", "path": "colors", "shape": "torus", "points": 200000, "vertices": 27903},
    ]


def _log_size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["reconstruct"] * 6 + ["batch", "point_normals", "point_normals", "weld", "mesh_normals", "colors"])
    shape = rng.choice(["sphere", "torus", "rotated", "displaced"])
    if path == "reconstruct":
        n = _log_size(rng, 4000, 1000000)
        depth = 5 if n < 10000 else synth.depth_for_size(n)
        if rng.random() < 0.25:
            depth = max(4, depth - 1)
        return reconstruct(shape, n, depth, rng.choice(["mixed", "mixed", "fp32"]), rng.choice(["packed", "packed", "surfel"]))
    if path == "batch":
        lo = _log_size(rng, 4000, 20000)
        return {"path": path, "clouds": rng.randint(2, 32), "lo": lo, "hi": _log_size(rng, lo, 150000), "depth": rng.choice([6, 7, 7]),
                "precision": rng.choice(["mixed", "mixed", "fp32"])}
    if path == "point_normals":
        return {"path": path, "shape": shape, "points": _log_size(rng, 4000, 1000000), "k": rng.choice([6, 8, 10, 10, 10, 12, 16]),
                "knn": rng.random() < 0.25}
    if path == "weld":
        n = _log_size(rng, 10000, 400000)
        return {"path": path, "shape": shape, "points": n, "depth": synth.depth_for_size(n)}
    if path == "mesh_normals":
        return {"path": path, "rows": _log_size(rng, 30, 900), "columns": _log_size(rng, 30, 600)}
    n = _log_size(rng, 4000, 1000000)
    return {"path": path, "shape": shape, "points": n, "vertices": _log_size(rng, 2000, max(2001, n // 3))}


def _cloud(shape, n, seed):
    """An oriented cloud (xyz, normals), float32 numpy."""
    seed = 7919 * int(seed) + 104729
    if shape == "sphere":
        return synth.sphere(n=n, seed=seed)
    if shape == "torus":
        return synth.torus(n=n, seed=seed)
    if shape == "displaced":
        return synth.displaced_sphere(n=n, seed=seed)
    return synth.batch64(count=1, seed=seed, lo=n, hi=n)[0]  # an ellipsoid or a torus, turned at random


def _gpu(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _points_on_device(case, seed):
    """(xyz, normals) as the call takes them: packed, or one tensor of 64-byte surfel records and None."""
    xyz, nrm = _cloud(case["shape"], case["points"], seed)
    if case.get("layout") == "surfel":
        rec = np.zeros((len(xyz), 16), np.float32)  # xyz at +16 bytes, the normal at +32
        rec[:, 4:7], rec[:, 8:11] = xyz, nrm
        return _gpu(rec), None
    return _gpu(xyz), _gpu(nrm)


def _batch_sizes(case):
    n, lo, hi = case["clouds"], case["lo"], case["hi"]
    return [int(round(lo * (hi / lo) ** (i * 7 % n / max(1, n - 1)))) for i in range(n)]  # log-spaced, in no sorted order


def _torus_grid(case, seed):
    """A closed triangle mesh with uneven vertices: a torus of rows x columns quads."""
    nu, nv = case["rows"], case["columns"]
    r = np.random.RandomState(seed + 17)
    u = (np.arange(nu)[:, None] + 0.4 * r.rand(nu, nv)) * (2 * np.pi / nu)
    v = (np.arange(nv)[None, :] + 0.4 * r.rand(nu, nv)) * (2 * np.pi / nv)
    rho = 0.3 + 0.1 * np.cos(v)
    vert = 0.5 + np.stack([rho * np.cos(u), rho * np.sin(u), 0.1 * np.sin(v)], axis=-1)
    i, j = np.meshgrid(np.arange(nu), np.arange(nv), indexing="ij")
    at = lambda a, b: (a % nu) * nv + b % nv  # noqa: E731
    q = np.stack([at(i, j), at(i + 1, j), at(i + 1, j + 1), at(i, j), at(i + 1, j + 1), at(i, j + 1)], axis=-1)
    return vert.reshape(-1, 3).astype(np.float32), q.reshape(-1, 3).astype(np.int32)


def _coloured(case, seed):
    """A coloured cloud and the mesh vertices to colour: points near its surface."""
    xyz, nrm = _cloud(case["shape"], case["points"], seed)
    r = np.random.RandomState(seed + 29)
    at = np.sort(r.randint(0, len(xyz), case["vertices"]))
    vert = xyz[at] + 0.002 * r.standard_normal((len(at), 3))
    return xyz, r.rand(len(xyz), 3).astype(np.float32), vert.astype(np.float32)


def prepare(case, seed):
    path = case["path"]
    if path == "batch":
        clouds = [synth.batch64(count=1, seed=7919 * int(seed) + 131 * i + 7, lo=n, hi=n)[0] for i, n in enumerate(_batch_sizes(case))]
        rec = pkg.PoissonReconstruction(depth=case["depth"], precision=PRECISION[case["precision"]], batch_cg_plan=0)
        return {"path": path, "rec": rec, "clouds": [(_gpu(x), _gpu(n)) for x, n in clouds],
                "buffers": [_mesh_buffers(case["depth"]) for _ in clouds]}
    if path == "mesh_normals":
        vert, tri = (_gpu(a) for a in _torus_grid(case, seed))
        mesh = binding.Mesh(ctypes.c_void_p(vert.data_ptr()), ctypes.c_void_p(tri.data_ptr()), vert.shape[0], tri.shape[0])
        return {"path": path, "rec": pkg.PoissonReconstruction(), "mesh": mesh, "buffers": (vert, tri)}
    if path == "colors":
        xyz, color, vert = (_gpu(a) for a in _coloured(case, seed))
        return {"path": path, "rec": pkg.PoissonReconstruction(), "xyz": xyz, "color": color, "vert": vert}
    xyz, nrm = _points_on_device(case, seed)
    if path == "point_normals":
        return {"path": path, "rec": pkg.PoissonReconstruction(), "xyz": xyz, "k": case["k"], "knn": case["knn"]}
    rec = pkg.PoissonReconstruction(depth=case["depth"], precision=PRECISION[case.get("precision", "mixed")])
    if path == "weld":
        rec.SolvePoissionReconstructionMesh(xyz, nrm)
    return {"path": path, "rec": rec, "xyz": xyz, "nrm": nrm, "buffers": _mesh_buffers(case["depth"])}


def _mesh_buffers(depth):
    """Vertex and index buffers of a fixed size (the reference's callers map buffers of fixed capacity too): a closed surface has
    about 3.4 triangles for each of the 4^depth cells of a face of the finest grid."""
    rows = 16 * 4 ** depth
    return torch.zeros((rows, 3), device="cuda"), torch.zeros((rows, 3), dtype=torch.int32, device="cuda")


def _keep(rec, mesh, buffers):
    """Copies the mesh out of the context's buffers, which last until its next call, into the program's own; rows past its length stay zero."""
    for own, part in zip(buffers, rec.mesh_tensors(mesh)):
        own[:len(part)].copy_(part)
    return buffers


def run(state):
    path, rec = state["path"], state["rec"]
    if path == "reconstruct":
        return _keep(rec, rec.SolvePoissionReconstructionMesh(state["xyz"], state["nrm"]), state["buffers"])
    if path == "batch":
        return [_keep(rec, m, own) for m, own in zip(rec.ReconstructBatch(state["clouds"]), state["buffers"])]
    if path == "point_normals":
        return rec.EstimateNormals(state["xyz"], k=state["k"], with_knn=state["knn"])
    if path == "weld":
        return _keep(rec, rec.WeldMesh(), state["buffers"])
    if path == "mesh_normals":
        return rec.MeshNormals(state["mesh"])
    return rec.VertexColors(state["vert"], state["xyz"], state["color"])


def _mesh_size(depth, n):
    """About how many (vertices, triangles) a closed surface gives: 3.4 triangles per cell of the finest grid's faces."""
    t = int(min(3.4 * 4 ** depth, 4 * n))
    return int(0.54 * t), t


def _reconstruct_work(n, depth):
    """Points in and mesh out; the operations are those of the stages that grow with the input: the splat of each point on 27
    nodes, the divergence and operator of each node (27 neighbours), 20 solver sweeps, the field at the mesh's corners (27 terms a level)."""
    v, t = _mesh_size(depth, n)
    nodes = 1.3 * t
    return {"bytes": 24 * n + 12 * v + 12 * t, "flops": n * 27 * 12 + nodes * 27 * (20 + 2 * 20) + 2 * v * 27 * 6 * depth}


def work(case):
    path = case["path"]
    if path == "reconstruct":
        return _reconstruct_work(case["points"], case["depth"])
    if path == "batch":
        parts = [_reconstruct_work(n, case["depth"]) for n in _batch_sizes(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    if path == "point_normals":
        n, k = case["points"], case["k"]
        return {"bytes": n * (12 + 12 + 4 + (4 * k if case["knn"] else 0)), "flops": n * (8 * 9 * k + 20 * k + 300)}
    if path == "weld":
        v, t = _mesh_size(case["depth"], case["points"])
        return {"bytes": 16 * v + 12 * t + 12 * v + 12 * t, "flops": v}
    if path == "mesh_normals":
        v = case["rows"] * case["columns"]
        return {"bytes": 12 * v + 24 * v + 12 * v, "flops": 2 * v * 40}
    return {"bytes": 24 * case["points"] + 24 * case["vertices"], "flops": case["vertices"] * (8 * 40 + 50)}


def _nearest(query, points, k):
    """Indices of each query's k nearest points, float64, nearest first: queries in blocks of one neighbourhood each, against the points
    in the block's box, widened until the k-th distance lies inside it."""
    lo, ext = points.min(0).values, (points.max(0).values - points.min(0).values).max()
    cell = ((query - lo) / ext * 63).long().clamp(0, 63)
    code = torch.zeros(len(query), dtype=torch.long, device=query.device)
    for b in range(6):
        for a in range(3):
            code |= ((cell[:, a] >> b) & 1) << (3 * b + a)
    order = torch.argsort(code, stable=True)
    out = torch.empty((len(query), k), dtype=torch.long, device=query.device)
    for rows in order.split(1024):
        q, margin = query[rows], 0.01 * ext
        while True:
            near = ((points >= q.min(0).values - margin) & (points <= q.max(0).values + margin)).all(1).nonzero()[:, 0]
            if len(near) >= k:
                d = (q[:, None, 0] - points[None, near, 0]) ** 2
                for a in (1, 2):
                    d += (q[:, None, a] - points[None, near, a]) ** 2
                d, at = d.topk(k, dim=1, largest=False)
                if len(near) == len(points) or bool(d[:, -1].max().sqrt() <= margin):
                    break
            margin = margin * 2
        out[rows] = near[at]
    return out


def exact(case, seed):
    """Float64 values of the passes that are formulas on their inputs.  A reconstruction's (and its welded form's) have none: which
    crossings a mesh has, and so its length and order, follow from its own 32-bit field and rules."""
    path = case["path"]
    if path == "mesh_normals":
        vert, tri = _torus_grid(case, seed)
        p = torch.from_numpy(vert).double()[torch.from_numpy(tri).long()]
        f = torch.nn.functional.normalize(torch.linalg.cross(p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]), dim=1, eps=0.0)
        total = torch.zeros((len(vert), 3), dtype=torch.float64)
        for c in range(3):
            total.index_add_(0, torch.from_numpy(tri[:, c]).long(), f)
        return torch.nn.functional.normalize(total, dim=1, eps=0.0)
    if path == "colors":
        xyz, color, vert = (_gpu(a).double() for a in _coloured(case, seed))
        at = _nearest(vert, xyz, 4)
        d = ((xyz[at] - vert[:, None]) ** 2).sum(-1)
        return ((d / d.sum(1, keepdim=True))[..., None] * color[at]).sum(1)
    if path == "point_normals":
        xyz = _gpu(_cloud(case["shape"], case["points"], seed)[0]).double()
        at = _nearest(xyz, xyz, case["k"])
        p = xyz[at]
        d = p - p.mean(1, keepdim=True)
        value, vector = np.linalg.eigh((d.transpose(1, 2).contiguous() @ d).cpu().numpy())  # ascending
        n = _gpu(vector[:, :, 0])
        n = torch.where((-xyz * n).sum(1, keepdim=True) < 0, -n, n)  # towards the viewpoint, the origin
        return n, _gpu(value[:, 0] / value.sum(1)), None
    return None
