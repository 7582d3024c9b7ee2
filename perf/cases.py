"""Performance cases of the octree library: what its users have it do, through its public entry points
(the Octree / Batch classes of octree_amd and the C ABI behind them).

Each case is a plain dict. "task" names the path:

  frame    a new host cloud taken through the whole pipeline: points, sort, build, kNN of every point
  probe    a handful of host query centres against a cloud that is already built (counts and kNN)
  csr      host query indices, result lists copied back into the caller's host buffers
  lists    result lists of consecutive points, in the caller's device buffers
  count    neighbour counts of every point, on the device
  knn      k nearest neighbours of consecutive points, in the caller's device buffers
  reorder  a device cloud and its per-point attribute records put into curve order
  batch    many clouds of uneven size, rebuilt and searched with mixed radii and k in one device pass

Clouds (built on the GPU from the seed alone): "box" is the uniform 100 x 100 x 20 m box at 5 points/m^3,
"tile" an airborne-LiDAR tile at 50 points/m^2 (terrain, buildings, vegetation), "sweep" a mobile-laser-scan
sweep (ground returns with density ~ 1/d^2 around a trajectory, facades, poles). All lie on a 1 mm grid, in no
particular order. Every case keeps these densities at every size.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "octrees-benchmark_amd"))
import octree_amd as A  # noqa: E402

KERNELS = {"sphere": A.K_SPHERE, "circle": A.K_CIRCLE, "cube": A.K_CUBE, "square": A.K_SQUARE}
ALGOS = {"neighbors": A.A_NEIGHBORS, "prune": A.A_PRUNE, "struct": A.A_STRUCT}
PRECS = {"fp64": A.PREC_FP64, "fp32": A.PREC_FP32}
ENCODERS = {"morton": A.ENC_MORTON, "hilbert": A.ENC_HILBERT}
DEV = "cuda"


def listed():
    return [
        # one scan of a rotating sensor, new every 100 ms: normals from 16 neighbours
        {"name": "frame_120k_knn16", "task": "frame", "cloud": "tile", "n": 120_000, "enc": "morton", "leaf": 32, "k": 16},
        # interactive picking: 64 places asked about in a cloud that stays
        {"name": "probe_64_of_1m", "task": "probe", "cloud": "box", "n": 1_000_000, "enc": "hilbert", "leaf": 32,
         "prec": "fp32", "radius": 2.5, "nq": 64, "k": 10},
        # the plain workload of the benchmark: 10 000 random centres in the 1 M-point box, lists to the host
        {"name": "csr_10k_of_1m", "task": "csr", "cloud": "box", "n": 1_000_000, "enc": "morton", "leaf": 32,
         "prec": "fp64", "algo": "prune", "kernel": "sphere", "radius": 2.5, "nq": 10_000},
        # per-point features of a piece of a tile: index lists that the next kernel of the program reads
        {"name": "lists_prune_1m_of_5m", "task": "lists", "cloud": "tile", "n": 5_000_000, "enc": "hilbert", "leaf": 128,
         "prec": "fp32", "algo": "prune", "kernel": "sphere", "radius": 1.0, "nq": 1_000_000},
        # the same as ranges (neighborsStruct), the form that large neighbourhoods are asked for in
        {"name": "lists_struct_2m_of_20m", "task": "lists", "cloud": "tile", "n": 20_000_000, "enc": "hilbert", "leaf": 128,
         "prec": "fp32", "algo": "struct", "kernel": "sphere", "radius": 2.5, "nq": 2_000_000},
        # the headline workload: every point of the 50 M-point tile counts its neighbours
        {"name": "count_tile_50m", "task": "count", "cloud": "tile", "n": 50_000_000, "enc": "hilbert", "leaf": 128,
         "prec": "fp32", "algo": "struct", "kernel": "sphere", "radius": 2.5},
        # voxel-shaped neighbourhoods, the box kernels, in plain FP64
        {"name": "count_cube_4m", "task": "count", "cloud": "box", "n": 4_000_000, "enc": "morton", "leaf": 64,
         "prec": "fp64", "algo": "prune", "kernel": "cube", "radius": 1.5},
        # kNN graph of a tile
        {"name": "knn10_tile_10m", "task": "knn", "cloud": "tile", "n": 10_000_000, "enc": "hilbert", "leaf": 128,
         "prec": "fp32", "k": 10, "nq": 10_000_000},
        # large neighbourhoods in plain FP64 (feature scales, outlier removal)
        {"name": "knn100_1m_of_4m", "task": "knn", "cloud": "box", "n": 4_000_000, "enc": "hilbert", "leaf": 64,
         "prec": "fp64", "k": 100, "nq": 1_000_000},
        # encode + sort of the 50 M-point tile with its 32-byte attribute records
        {"name": "reorder_tile_50m", "task": "reorder", "cloud": "tile", "n": 50_000_000, "enc": "hilbert"},
        # the same for a mobile-laser-scan sweep, whose keys cluster along the trajectory
        {"name": "reorder_sweep_20m", "task": "reorder", "cloud": "sweep", "n": 20_000_000, "enc": "morton"},
        # many clouds of uneven size with mixed radii and k, rebuilt and searched, results to the host
        {"name": "batch_48_clouds_12m", "task": "batch", "clouds": 48, "n": 12_000_000, "leaf": 64, "prec": "fp32",
         "per": 3_000, "kmax": 64},
    ]


def draw(rng):
    def log_int(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    task = rng.choice(["frame", "probe", "csr", "lists", "lists", "count", "count", "knn", "knn", "reorder", "batch"])
    c = {"task": task}
    if task == "batch":
        clouds = log_int(8, 96)
        return dict(c, clouds=clouds, n=max(clouds * 12_000, log_int(500_000, 12_000_000)), leaf=rng.choice([32, 64, 128]),
                    prec=rng.choice(["fp32", "fp64"]), per=log_int(200, 3_000), kmax=rng.choice([24, 64, 100]))
    top = {"frame": 250_000, "probe": 3_000_000, "csr": 3_000_000, "lists": 10_000_000, "count": 10_000_000,
           "knn": 8_000_000, "reorder": 40_000_000}[task]
    n = log_int(50_000, top)
    c.update(cloud=rng.choice(["box", "tile", "sweep"] if task in ("reorder", "csr", "knn") else ["box", "tile"]), n=n,
             enc="morton" if task == "frame" else rng.choice(["morton", "hilbert"]))
    if task == "reorder":
        return c
    c["leaf"] = rng.choice([16, 32, 64, 128, 128])
    if task == "frame":
        return dict(c, k=log_int(5, 30))
    c["prec"] = rng.choice(["fp32", "fp32", "fp64"])
    if task == "probe":
        return dict(c, radius=round(rng.uniform(0.5, 3.0), 3), nq=log_int(1, 1_000), k=log_int(1, 60))
    if task == "knn":
        k = log_int(1, 250)
        return dict(c, k=k, nq=min(n, int(3e7 / (k + 4))))
    c["kernel"] = rng.choice(["sphere", "sphere", "sphere", "circle", "cube", "square"])
    c["algo"] = rng.choice(["neighbors", "prune", "struct", "struct"])
    # a column of the box holds far more points than a ball, and the sweep is dense near its trajectory
    flat = c["kernel"] in ("circle", "square") and c["cloud"] == "box"
    lo, hi = (0.05, 0.4) if c["cloud"] == "sweep" else (0.3, 1.0 if flat else 2.5)
    c["radius"] = round(math.exp(rng.uniform(math.log(lo), math.log(hi))), 3)
    if task == "csr":
        return dict(c, nq=log_int(100, 1_500 if c["cloud"] == "sweep" else 20_000))
    if task == "lists":
        return dict(c, nq=min(n, log_int(10_000, 1_000_000), int(1.5e8 / _mean_neighbours(c))))
    return c


# ---------------------------------------------------------------- clouds
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _uniform(g, n, lo=0.0, hi=1.0):
    return torch.rand(n, generator=g, device=DEV, dtype=torch.float64).mul_(hi - lo).add_(lo)


def _normal(g, n, sd):
    return torch.randn(n, generator=g, device=DEV, dtype=torch.float64).mul_(sd)


def _pack(x, y, z):
    return torch.stack((x, y, z), dim=1).mul_(1000.0).round_().div_(1000.0)


def _box(n, seed):
    g = _gen(seed)
    side = 100.0 * (n / 1e6) ** (1.0 / 3.0)
    return _pack(_uniform(g, n, 0, side), _uniform(g, n, 0, side), _uniform(g, n, 0, side / 5))


def _tile(n, seed, x0=651000.0, y0=6861000.0):
    """The benchmark's tile: ground of 8 sinusoids, 15 % of the points on roofs and walls of 2000 box buildings
    per km^2, 20 % in 4000 Gaussian vegetation blobs per km^2 (sigma 2 m)."""
    g = _gen(seed)
    ext = 1000.0 * math.sqrt(n / 50e6)
    w, th, lam, phi = torch.rand(4, 8, generator=g, device=DEV, dtype=torch.float64).cpu()
    w = (0.2 + 0.8 * w) * (14.0 / (0.2 + 0.8 * w).sum())
    kx, ky = (2 * math.pi * f(2 * math.pi * th) / (40.0 + 560.0 * lam) for f in (torch.cos, torch.sin))
    waves = list(zip(w.tolist(), kx.tolist(), ky.tolist(), (2 * math.pi * phi).tolist()))

    def ground(x, y):
        z = torch.zeros_like(x)
        for a, p, q, f in waves:
            z += a * torch.sin(x * p + y * q + f)
        return z

    pick = _uniform(g, n)
    x, y = _uniform(g, n, 0, ext), _uniform(g, n, 0, ext)
    z = ground(x, y) + _normal(g, n, 0.05)
    blobs = max(1, round(4000 * ext * ext / 1e6))
    bx, by = _uniform(g, blobs, 0, ext), _uniform(g, blobs, 0, ext)
    bz = ground(bx, by) + _uniform(g, blobs, 3, 15)
    veg = pick < 0.20
    m = int(veg.sum())
    at = torch.randint(blobs, (m,), generator=g, device=DEV)
    x[veg], y[veg], z[veg] = bx[at] + _normal(g, m, 2.0), by[at] + _normal(g, m, 2.0), bz[at] + _normal(g, m, 2.0)
    houses = max(1, round(2000 * ext * ext / 1e6))
    hx, hy = _uniform(g, houses, 0, ext), _uniform(g, houses, 0, ext)
    hw, hd, hh = _uniform(g, houses, 10, 40), _uniform(g, houses, 10, 40), _uniform(g, houses, 5, 30)
    base = ground(hx, hy)
    built = (pick >= 0.20) & (pick < 0.35)
    m = int(built.sum())
    at = torch.randint(houses, (m,), generator=g, device=DEV)
    u, v, t = _uniform(g, m, -0.5, 0.5), _uniform(g, m, -0.5, 0.5), _uniform(g, m)
    roof = _uniform(g, m) < hw[at] * hd[at] / (hw[at] * hd[at] + 2 * (hw[at] + hd[at]) * hh[at])
    edge = torch.where(v < 0, -0.5, 0.5)  # walls: half on the sides along x, half on those along y
    along = _uniform(g, m) < 0.5
    x[built] = hx[at] + hw[at] * torch.where(roof | along, u, edge)
    y[built] = hy[at] + hd[at] * torch.where(roof, v, torch.where(along, edge, u))
    z[built] = base[at] + hh[at] * torch.where(roof, torch.ones_like(t), t)
    lim = ext - 0.001
    return _pack(x.clamp_(0, lim).add_(x0), y.clamp_(0, lim).add_(y0), z)


def _sweep(n, seed):
    g = _gen(seed)
    length = 5000.0 * n / 400e6
    s = _uniform(g, n, 0, length)
    d = 1.0 / (1.0 - _uniform(g, n, 0, 1.0 - 1.0 / 80.0))  # density ~ 1/d^2 on [1, 80] m
    side = torch.where(_uniform(g, n) < 0.5, -1.0, 1.0).to(torch.float64)
    z = _normal(g, n, 0.02)
    pick = _uniform(g, n)
    wall = pick < 0.2
    d = torch.where(wall, 12.0 + 3.0 * torch.floor(s / 20.0).remainder(3.0), d)
    z = torch.where(wall, _uniform(g, n, 0, 15), z)
    pole = (pick >= 0.2) & (pick < 0.23)
    z = torch.where(pole, _uniform(g, n, 0, 6), z)
    d = torch.where(pole, 6.0 + 0.1 * _uniform(g, n), d)
    s = torch.where(pole, torch.floor(s / 25.0) * 25.0 + 0.1 * _uniform(g, n), s)
    bend = 40.0 * torch.sin(s / 200.0)
    return _pack(651000.0 + s, 6861000.0 + bend + side * d, z)


def _cloud(case, seed):
    return {"box": _box, "tile": _tile, "sweep": _sweep}[case["cloud"]](case["n"], seed)


# ---------------------------------------------------------------- the library's device entry points
def _check(ctx, rc):
    if rc != 0:
        raise A.OctError(f"status {rc}: {ctx.L.oct_last_error(ctx.h)}")


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _set_points(ctx, xyz):
    """A device cloud (n x 3 float64) becomes the context's cloud."""
    ctx.n = xyz.shape[0]
    _check(ctx, ctx.L.oct_set_points_dev(ctx.h, _ptr(xyz), ctx.n, 24))


def _built(case, xyz):
    ctx = A.Octree(0)
    torch.cuda.synchronize()  # the context has a stream of its own
    _set_points(ctx, xyz)
    ctx.sort_points(ENCODERS[case["enc"]], fetch=False)
    ctx.build(case["leaf"])
    return ctx


def _list_words(case):
    """Room for the result lists, in 32-bit words, as a program that calls again and again sets it aside."""
    mean = _mean_neighbours(case)
    per = 0.25 * mean + 64 if case["algo"] == "struct" else 2 * mean + 16
    return int(case["nq"] * per)


def _batch_shape(case, seed):
    """Cloud sizes and the queries: radius (cloud, index, r), kNN (cloud, index, k)."""
    rng = np.random.default_rng(seed)
    sizes = np.exp(rng.uniform(np.log(1e4), np.log(4e6), case["clouds"]))
    sizes = np.maximum(1e4, sizes * (case["n"] / sizes.sum())).astype(np.int64)
    cloud = np.repeat(np.arange(case["clouds"], dtype=np.uint32), case["per"])
    idx = (rng.uniform(0, 1, len(cloud)) * sizes[cloud]).astype(np.uint32)
    knn = np.arange(len(cloud)) % 5 == 4
    radii = rng.uniform(0.5, 3.0, len(cloud)).astype(np.float32).astype(np.float64)
    k = rng.integers(8, case["kmax"] + 1, len(cloud)).astype(np.uint32)
    return sizes, (cloud[~knn], idx[~knn], radii[~knn]), (cloud[knn], idx[knn], k[knn])


def _batch_cloud(i, n, seed):
    return (_box if i % 2 else _tile)(int(n), 1000 * seed + i)


# ---------------------------------------------------------------- prepare, run, work
def prepare(case, seed):
    s = {"case": case}
    task = case["task"]
    if task == "batch":
        sizes, r, k = _batch_shape(case, seed)
        b = A.Batch(0)
        for i, n in enumerate(sizes):
            b.add(_batch_cloud(i, n, seed).cpu().numpy(), A.ENC_MORTON, case["leaf"])
        b.queries(*r, *k, kmax=case["kmax"])
        s["batch"] = b
        return s
    xyz = _cloud(case, seed)
    n = case["n"]
    if task == "frame":
        s["xyz"] = xyz.cpu().numpy()
        s["ctx"] = A.Octree(0)
        s["idx"] = torch.empty((n, case["k"]), dtype=torch.int32, device=DEV)
        s["d2"] = torch.empty((n, case["k"]), dtype=torch.float32, device=DEV)
        return s
    if task == "reorder":
        s["xyz"], s["ctx"] = xyz, A.Octree(0)
        g = _gen(seed + 1)
        s["records"] = torch.randint(-2**31, 2**31 - 1, (n, 8), generator=g, device=DEV, dtype=torch.int32)
        s["sorted"] = torch.empty_like(s["records"])
        return s
    if task == "probe":
        g = _gen(seed + 1)
        at = torch.randint(n, (case["nq"],), generator=g, device=DEV)
        s["centers"] = (xyz[at] + 0.2 * torch.rand((case["nq"], 3), generator=g, device=DEV, dtype=torch.float64)).cpu().numpy()
    s["ctx"] = ctx = _built(case, xyz)
    del xyz
    if task == "csr":
        nq = case["nq"]
        s["idx"] = np.random.default_rng(seed).integers(0, n, nq).astype(np.uint32)
        s["counts"], s["offsets"] = np.zeros(nq, np.uint32), np.zeros(nq + 1, np.uint64)
        s["entries"] = np.zeros(_list_words(case), np.uint32)
    elif task == "count":
        # a program that searches every point tunes the search on its cloud once
        ctx.autotune_radius(KERNELS[case["kernel"]], ALGOS[case["algo"]], PRECS[case["prec"]], case["radius"])
        s["counts"] = torch.empty(n, dtype=torch.int32, device=DEV)
    elif task == "knn":
        ctx.autotune_knn(case["k"], PRECS[case["prec"]])
        s["first"] = (n - case["nq"]) // 2
        s["idx"] = torch.empty((case["nq"], case["k"]), dtype=torch.int32, device=DEV)
        s["d2"] = torch.empty((case["nq"], case["k"]), dtype=torch.float32, device=DEV)
    elif task == "lists":
        nq = case["nq"]
        s["idx"] = torch.arange((n - nq) // 2, (n - nq) // 2 + nq, dtype=torch.int32, device=DEV)
        s["counts"] = torch.empty(nq, dtype=torch.int32, device=DEV)
        s["offsets"] = torch.empty(nq + 1, dtype=torch.int64, device=DEV)
        s["entries"] = torch.zeros(_list_words(case), dtype=torch.int32, device=DEV)
    return s


def run(s):
    c = s["case"]
    task = c["task"]
    if task == "batch":
        b = s["batch"]
        b.pipeline(A.K_SPHERE, A.A_STRUCT, PRECS[c["prec"]])
        counts, idx, d2 = b.pipeline_results()
        return {"counts": counts.view(np.int32), "idx": idx, "d2": d2}
    ctx = s["ctx"]
    if task == "frame":
        ctx.set_points(s["xyz"])
        center, radii, _, _ = ctx.sort_points(ENCODERS[c["enc"]], fetch=False)
        ctx.build(c["leaf"])
        ctx.knn_dev(c["k"], A.PREC_FP32, idx_ptr=s["idx"].data_ptr(), d2_ptr=s["d2"].data_ptr())
        ctx.synchronize()
        return {"center": center, "radii": radii, "idx": s["idx"], "d2": s["d2"]}
    if task == "reorder":
        _set_points(ctx, s["xyz"])
        center, radii, _, _ = ctx.sort_points(ENCODERS[c["enc"]], fetch=False)
        ctx.gather_records_dev(s["records"].data_ptr(), s["sorted"].data_ptr(), 32)
        return {"center": center, "radii": radii, "records": s["sorted"]}
    if task == "probe":
        counts, _ = ctx.radius(A.K_SPHERE, A.A_STRUCT, PRECS[c["prec"]], centers=s["centers"], radius=c["radius"])
        idx, d2, _ = ctx.knn(c["k"], PRECS[c["prec"]], centers=s["centers"])
        return {"counts": counts.view(np.int32), "idx": idx, "d2": d2}
    if task == "csr":
        kernel, algo, prec, at = KERNELS[c["kernel"]], ALGOS[c["algo"]], PRECS[c["prec"]], lambda a: ctypes.c_void_p(a.ctypes.data)
        _check(ctx, ctx.L.oct_radius(ctx.h, kernel, algo, prec, None, at(s["idx"]), None, float(c["radius"]), c["nq"], 1,
                                     at(s["counts"]), None))
        _check(ctx, ctx.L.oct_radius_fetch(ctx.h, at(s["offsets"]), at(s["entries"]), s["entries"].size))
        return {k: s[k].view(np.int64 if k == "offsets" else np.int32) for k in ("counts", "offsets", "entries")}
    if task == "lists":
        total = ctypes.c_uint64(0)
        _check(ctx, ctx.L.oct_radius_lists_noalloc(
            ctx.h, KERNELS[c["kernel"]], ALGOS[c["algo"]], PRECS[c["prec"]], _ptr(s["idx"]), float(c["radius"]), c["nq"],
            _ptr(s["counts"]), _ptr(s["offsets"]), _ptr(s["entries"]), s["entries"].numel(), ctypes.byref(total)))
        return {"counts": s["counts"], "offsets": s["offsets"], "entries": s["entries"], "total": total.value}
    if task == "count":
        _check(ctx, ctx.L.oct_radius_dev(ctx.h, KERNELS[c["kernel"]], ALGOS[c["algo"]], PRECS[c["prec"]], None,
                                         float(c["radius"]), ctx.n, _ptr(s["counts"]), None))
        ctx.synchronize()
        return {"counts": s["counts"]}
    ctx.knn_dev(c["k"], PRECS[c["prec"]], first=s["first"], nq=c["nq"], idx_ptr=s["idx"].data_ptr(), d2_ptr=s["d2"].data_ptr())
    ctx.synchronize()
    return {"idx": s["idx"], "d2": s["d2"]}


def _mean_neighbours(case):
    r, kernel = case["radius"], case["kernel"] if "kernel" in case else "sphere"
    area = math.pi * r * r if kernel in ("sphere", "circle") else 4 * r * r
    if case["cloud"] == "tile":
        return 50 * area
    if case["cloud"] == "sweep":
        return 20_000 * area
    return 5 * (area * 4 / 3 * r if kernel == "sphere" else area * 2 * r if kernel == "cube"
                else area * 20.0 * (case["n"] / 1e6) ** (1.0 / 3.0))


def work(case):
    task = case["task"]
    if task == "batch":
        nr, nk = case["clouds"] * case["per"] * 0.8, case["clouds"] * case["per"] * 0.2
        kmean = (8 + case["kmax"]) / 2
        return {"bytes": 24 * case["n"] + nr * 20 + nk * (12 + 12 * case["kmax"]), "flops": 8 * (nr * 50 * math.pi * 3 + nk * kmean)}
    n = case["n"]
    if task == "reorder":  # points and records in; keys, sorted cloud and records out
        return {"bytes": n * (24 + 32 + 8 + 24 + 32), "flops": 12 * n}
    if task == "frame":
        return {"bytes": n * (24 + 8 * case["k"]), "flops": n * (12 + 8 * case["k"])}
    if task == "probe":
        return {"bytes": case["nq"] * (24 * _mean_neighbours(case) + 24 + 4 + 12 * case["k"]),
                "flops": 8 * case["nq"] * (_mean_neighbours(case) + case["k"])}
    if task == "knn":  # the queries are a run of the cloud: its points once, k results each
        return {"bytes": case["nq"] * (24 + 8 * case["k"]), "flops": 8 * case["nq"] * case["k"]}
    nq = case.get("nq", n)
    m = _mean_neighbours(case)
    out = 0 if task == "count" else m * (8 / 10 if case["algo"] == "struct" else 4)  # ranges of about 10 points
    return {"bytes": nq * (24 + 4 + (8 if task != "count" else 0) + out), "flops": 8 * nq * m}


# ---------------------------------------------------------------- exact values in 64 bits
def _box_of(xyz):
    lo, hi = xyz.min(0).values, xyz.max(0).values
    return (lo + (hi - lo) / 2), (hi - lo) / 2


def _morton_order(xyz):
    """Stable order of the points by their Morton key (21 bits per axis over the bounding box)."""
    c, r = _box_of(xyz)
    q = (((xyz - c) + r) / (2.0 * r) * 2097152.0).to(torch.int64).clamp_(0, 2097151)
    key = torch.zeros(len(xyz), dtype=torch.int64, device=xyz.device)
    for bit in range(21):
        for a in range(3):
            key |= ((q[:, a] >> bit) & 1) << (3 * bit + a)
    return torch.sort(key, stable=True).indices


def _nearest(points, centers, k):
    """The k smallest squared distances of each centre, ascending."""
    out = torch.empty((len(centers), k), dtype=torch.float64, device=points.device)
    step = max(1, int(1.5e8 // len(points)))
    for i in range(0, len(centers), step):
        d = torch.zeros((len(centers[i:i + step]), len(points)), dtype=torch.float64, device=points.device)
        for a in range(3):
            d += (centers[i:i + step, a, None] - points[None, :, a]).square_()
        out[i:i + step] = torch.topk(d, k, dim=1, largest=False, sorted=True).values
    return out


def exact(case, seed):
    task = case["task"]
    if task == "batch":
        sizes, _, (kc, ki, kk) = _batch_shape(case, seed)
        d2 = torch.full((len(kc), case["kmax"]), float("nan"), dtype=torch.float64)
        for i, n in enumerate(sizes):
            xyz = _batch_cloud(i, n, seed)
            xyz = xyz[_morton_order(xyz)]
            rows = np.nonzero(kc == i)[0]
            if len(rows):
                d2[torch.from_numpy(rows)] = _nearest(xyz, xyz[torch.from_numpy(ki[rows].astype(np.int64)).to(DEV)], case["kmax"]).cpu()
        d2[torch.arange(case["kmax"])[None, :] >= torch.from_numpy(kk.astype(np.int64))[:, None]] = float("nan")
        return {"counts": None, "idx": None, "d2": d2}
    if task == "frame":
        xyz = _cloud(case, seed)
        center, radii = _box_of(xyz)
        sx = xyz[_morton_order(xyz)]
        return {"center": center, "radii": radii, "idx": None, "d2": _nearest(sx, sx, case["k"])}
    if task == "reorder":
        center, radii = _box_of(_cloud(case, seed))
        return {"center": center, "radii": radii, "records": None}
    if task == "probe":
        xyz = _cloud(case, seed)
        g = _gen(seed + 1)
        at = torch.randint(case["n"], (case["nq"],), generator=g, device=DEV)
        centers = xyz[at] + 0.2 * torch.rand((case["nq"], 3), generator=g, device=DEV, dtype=torch.float64)
        return {"counts": None, "idx": None, "d2": _nearest(xyz, centers, case["k"])}
    return None  # whole numbers, or (kNN of millions of points) far beyond a few seconds of exhaustive search
