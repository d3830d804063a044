"""The calls that this framework is timed on: neighbour searches, the fused
search + features pipelines, the CSR feature functions and the host-array
Python API, from a thousand points to ten million.

A case is a dict of plain values.  "op" names the call, "scene" the kind of
cloud, "n" its points, "k" the neighbours (or the most neighbours of a radius
search).  Clouds are made on the GPU from the seed alone, in shuffled order (a
scan is not stored in spatial order); device calls write into buffers that the
program keeps, as a pipeline over a stream of clouds does.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import point_geometric_features_amd as pgeof
from point_geometric_features_amd import capi

DEV = "cuda"
F_EPS = 1e-3  # the epsilon of the feature formulas


# ------------------------------------------------------------------ cases ----
def listed():
    return [
        # the smallest call in use: labels of a few points carried over from a
        # subsampled cloud (queries differ from the data), device arrays
        {"name": "knn_1k", "op": "knn", "scene": "cube", "n": 1000, "m": 257, "k": 10},
        # 10,000 points uniform in the unit cube, kNN CSR and features in one
        # call: the README example's size, where launches and latency count
        {"name": "fused_10k_k20", "op": "fused", "scene": "cube", "n": 10_000, "k": 20},
        # a LiDAR tile of the middling size of a serving stream
        {"name": "fused_100k_k20", "op": "fused", "scene": "lidar", "n": 100_003, "k": 20},
        # the headline: a 10 M-point LiDAR scene, kNN + features
        {"name": "fused_10m_k20", "op": "fused", "scene": "lidar", "n": 10_000_000, "k": 20},
        # larger neighbourhoods on a scene of 4 M points, an odd number of rows
        {"name": "fused_4m_k50", "op": "fused", "scene": "lidar", "n": 4_000_001, "k": 50},
        # knn_search of the upstream benchmark: 1 M points uniform in
        # [0, 200)^3, k = 50, indices and squared distances
        {"name": "knn_1m_k50", "op": "knn", "scene": "wide", "n": 1_000_000, "m": 0, "k": 50},
        # radius_search of the upstream benchmark: the same cloud, r = 0.2,
        # at most 30 (nearly every row holds its own point only)
        {"name": "radius_1m", "op": "radius", "scene": "wide", "n": 1_000_000, "k": 30, "r": 0.2},
        # radius CSR and features at four scales in one call, LiDAR, 2 M points
        {"name": "multiscale_2m", "op": "multiscale", "scene": "lidar", "n": 2_000_000, "k": 64, "r": 0.5},
        # kNN of 100 and the features at the eigentropy-optimal k, on planes,
        # lines and blobs far from the origin
        {"name": "optimal_1m", "op": "optimal", "scene": "precision", "n": 1_000_000, "k": 100},
        # compute_features on a ragged CSR that the caller has (rows of up to
        # 40 neighbours, some below k_min)
        {"name": "features_3m", "op": "features", "scene": "clusters", "n": 3_000_017, "k": 40, "k_min": 5},
        # the selected features of float64 host points (the README example's
        # radius, cap and features at its point density)
        {"name": "selected_200k", "op": "selected", "scene": "cube", "n": 200_000, "k": 20, "r": 0.2},
        # the two calls of a program that holds numpy arrays: knn_search, then
        # compute_features on its CSR, PCIe copies included
        {"name": "host_100k_k20", "op": "host", "scene": "lidar", "n": 100_000, "k": 20},
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["knn", "fused", "fused", "radius", "multiscale", "optimal", "features", "selected", "host"])
    if op == "knn":
        k = _size(rng, 1, 64)
        n = _size(rng, 1000, 2_000_000)
        m = rng.choice([0, _size(rng, 200, 1_000_000)])
        return {"op": op, "scene": rng.choice(["cube", "wide", "lidar"]), "n": n, "m": m, "k": k}
    if op == "fused":
        k = _size(rng, 8, 64)
        return {"op": op, "scene": rng.choice(["cube", "lidar"]), "n": _size(rng, 5000, 100_000_000 // k), "k": k}
    if op == "radius":
        # at the wide scene's density and the lidar scene's: from a point or
        # none in the ball to more than the cap
        scene = rng.choice(["wide", "lidar"])
        r = rng.uniform(0.2, 6.0) if scene == "wide" else rng.uniform(0.1, 0.6)
        return {"op": op, "scene": scene, "n": _size(rng, 10_000, 2_000_000), "k": _size(rng, 8, 64), "r": r}
    if op == "multiscale":
        return {"op": op, "scene": "lidar", "n": _size(rng, 50_000, 2_000_000), "k": _size(rng, 40, 100),
                "r": rng.uniform(0.3, 0.6)}
    if op == "optimal":
        return {"op": op, "scene": rng.choice(["lidar", "precision"]), "n": _size(rng, 50_000, 1_000_000),
                "k": _size(rng, 30, 100)}
    if op == "features":
        return {"op": op, "scene": "clusters", "n": _size(rng, 20_000, 5_000_000), "k": _size(rng, 10, 60),
                "k_min": rng.randint(4, 8)}
    if op == "selected":
        return {"op": op, "scene": "cube", "n": _size(rng, 20_000, 1_000_000), "k": _size(rng, 10, 40),
                "r": rng.uniform(0.15, 0.25)}
    return {"op": op, "scene": rng.choice(["cube", "lidar"]), "n": _size(rng, 10_000, 300_000), "k": _size(rng, 8, 50)}


# ----------------------------------------------------------------- clouds ----
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=DEV, dtype=torch.float64)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float64)


def _pick(g, n, weights):
    """n object numbers, objects taken in proportion to their weights."""
    edges = torch.cumsum(weights, 0)
    return torch.searchsorted(edges, _rand(g, n) * edges[-1]).clamp_(max=len(weights) - 1)


def _lidar(n, g):
    """A street scene at the density of 10 M points on 200 m x 200 m: half the
    points ground, then walls, poles and trunks, and vegetation."""
    extent = max(5.0, 200.0 * math.sqrt(n / 10_000_000))
    area = (extent / 200.0) ** 2
    n_wall, n_cyl, n_blob = n // 5, n // 10, n // 5
    n_ground = n - n_wall - n_cyl - n_blob
    ground = torch.cat([_rand(g, n_ground, 2) * extent, 0.02 * _randn(g, n_ground, 1)], 1)

    objects = max(1, round(40 * area))
    length, height = 5 + 25 * _rand(g, objects), 2 + 8 * _rand(g, objects)
    at, angle = _rand(g, objects, 2) * extent, math.pi * _rand(g, objects)
    i = _pick(g, n_wall, length * height)
    d = torch.stack([torch.cos(angle), torch.sin(angle)], 1)[i]
    nrm = torch.stack([-d[:, 1], d[:, 0]], 1)
    xy = at[i] + d * (_rand(g, n_wall) * length[i])[:, None] + nrm * (0.01 * _randn(g, n_wall))[:, None]
    wall = torch.cat([xy, (_rand(g, n_wall) * height[i])[:, None]], 1)

    objects = max(1, round(400 * area))
    radius, height = 0.1 + 0.4 * _rand(g, objects), 2 + 6 * _rand(g, objects)
    at = _rand(g, objects, 2) * extent
    i = _pick(g, n_cyl, radius * height)
    a, r = 2 * math.pi * _rand(g, n_cyl), radius[i] + 0.005 * _randn(g, n_cyl)
    pole = torch.stack([at[i, 0] + r * torch.cos(a), at[i, 1] + r * torch.sin(a), _rand(g, n_cyl) * height[i]], 1)

    objects = max(1, round(1000 * area))
    at = torch.cat([_rand(g, objects, 2) * extent, 2 + 10 * _rand(g, objects, 1)], 1)
    sigma = 0.3 + 1.2 * _rand(g, objects)
    i = _pick(g, n_blob, torch.ones_like(sigma))
    blob = at[i] + sigma[i][:, None] * _randn(g, n_blob, 3)
    return torch.cat([ground, wall, pole, blob])


def _precision(n, g):
    """Exact planes (level and tilted), exact lines and blobs, 1e5 from the origin."""
    n_tilt, n_line, n_blob = n // 4, n // 5, (3 * n) // 10
    n_level = n - n_tilt - n_line - n_blob
    spread = torch.tensor([200.0, 200.0, 20.0], dtype=torch.float64, device=DEV)

    def centres(points, per):
        objects = max(1, points // per)
        return _rand(g, objects, 3) * spread, torch.randint(objects, (points,), generator=g, device=DEV)

    at, i = centres(n_level, 2500)
    level = torch.cat([at[i, :2] + 5 * _rand(g, n_level, 2) - 2.5, torch.round(at[i, 2:] * 10) / 10], 1)
    at, i = centres(n_tilt, 2500)
    axes = torch.linalg.qr(_randn(g, len(at), 3, 3).cpu())[0].to(DEV)
    uv = 5 * _rand(g, n_tilt, 2) - 2.5
    tilt = at[i] + uv[:, :1] * axes[i, :, 0] + uv[:, 1:] * axes[i, :, 1]
    at, i = centres(n_line, 1000)
    along = torch.nn.functional.normalize(_randn(g, len(at), 3), dim=1)
    line = at[i] + (10 * _rand(g, n_line, 1) - 5) * along[i]
    at, i = centres(n_blob, 1000)
    blob = at[i] + (0.2 + 0.8 * _rand(g, len(at)))[i][:, None] * _randn(g, n_blob, 3)
    return torch.cat([level, tilt, line, blob]) + torch.tensor([1e5, 1e5, 0.0], dtype=torch.float64, device=DEV)


def _cloud(scene, n, g):
    if scene == "cube":
        xyz = _rand(g, n, 3)
    elif scene == "wide":
        xyz = 200.0 * _rand(g, n, 3)
    elif scene == "lidar":
        xyz = _lidar(n, g)
    else:
        xyz = _precision(n, g)
    return xyz[torch.randperm(n, generator=g, device=DEV)].float().contiguous()


def _cluster_csr(n, k, g):
    """A cloud of patches of 64 points and, for every point, a ragged list of
    1 to k neighbours out of its patch, the point itself first."""
    patches = (n + 63) // 64
    side = math.ceil(math.sqrt(patches))
    pid = torch.arange(patches, device=DEV)
    at = torch.stack([(pid % side).double(), (pid // side).double(), _rand(g, patches)], 1)
    bumps = torch.tensor([1.0, 1.0, 0.1], dtype=torch.float64, device=DEV)
    local = (at[:, None, :] + _rand(g, patches, 64, 3) * bumps).reshape(-1, 3)[:n]
    where = torch.randperm(n, generator=g, device=DEV)  # row of point p of the patch order
    xyz = torch.empty(n, 3, device=DEV)
    xyz[where] = local.float()
    row_of = torch.empty(n, dtype=torch.int64, device=DEV)
    row_of[where] = torch.arange(n, device=DEV)  # patch position of a row
    count = torch.randint(1, k + 1, (n,), generator=g, device=DEV)
    ptr = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    ptr[1:] = torch.cumsum(count, 0)
    rows = torch.repeat_interleave(torch.arange(n, device=DEV), count)
    nth = torch.arange(len(rows), device=DEV) - ptr[rows]
    pos = row_of[rows]
    start = torch.randint(1, 64, (n,), generator=g, device=DEV)  # an odd walk of the patch: no point twice
    to = (pos // 64) * 64 + (pos % 64 + nth * (2 * (start[rows] % 32) + 1)) % 64
    nn = where[torch.where(to < n, to, pos)]
    return xyz, nn.int(), ptr.int()


# ---------------------------------------------------------------- prepare ----
SCALES = [10, 20, 50, 100]
SELECTED = ("Verticality", "Curvature")


def _empty(*shape, dtype=torch.int32):
    return torch.zeros(*shape, dtype=dtype, device=DEV)


def prepare(case, seed):
    g = _gen(seed)
    op, n, k = case["op"], case["n"], case["k"]
    s = {"case": case}
    if op == "features":
        s["xyz"], s["nn"], s["ptr"] = _cluster_csr(n, k, g)
        return s
    if op == "selected":
        # 400 points per unit volume, as 10,000 in the README's cloud at its radius
        s["xyz"] = (_rand(g, n, 3) * (n / 400.0) ** (1.0 / 3.0)).cpu().numpy()
        s["features"] = [getattr(pgeof.EFeatureID, f) for f in SELECTED]
        return s
    s["xyz"] = _cloud(case["scene"], n, g)
    if op == "host":
        s["xyz"] = s["xyz"].cpu().numpy()
        s["ptr"] = (np.arange(n + 1, dtype=np.int64) * k).astype(np.uint32)
    elif op == "knn" and case["m"]:
        # queries in and around the data's box
        lo, hi = s["xyz"].amin(0), s["xyz"].amax(0)
        s["query"] = (lo + (hi - lo) * (1.1 * _rand(g, case["m"], 3) - 0.05)).float().contiguous()
    elif op == "fused":
        s["nn"], s["ptr"] = _empty(n * k), _empty(n + 1)
        s["feat"] = _empty(n, 11, dtype=torch.float32)
        s["ws"] = torch.empty(capi.knn_workspace_size(n, n, k), dtype=torch.uint8, device=DEV)
    elif op == "multiscale":
        s["nn"], s["ptr"] = _empty(n * k), _empty(n + 1)
        s["feat"] = _empty(n, len(SCALES), 11, dtype=torch.float32)
        s["ws"] = torch.empty(capi.radius_multiscale_workspace_size(n, k, len(SCALES)), dtype=torch.uint8, device=DEV)
    elif op == "optimal":
        s["nn"], s["ptr"] = _empty(n * k), _empty(n + 1)
        s["feat"] = _empty(n, 12, dtype=torch.float32)
        s["ws"] = torch.empty(capi.knn_optimal_workspace_size(n, k), dtype=torch.uint8, device=DEV)
    return s


# -------------------------------------------------------------------- run ----
def run(s):
    case = s["case"]
    op, k = case["op"], case["k"]
    xyz = s["xyz"]
    if op == "knn":
        idx, d2 = pgeof.knn_search(xyz, s.get("query", xyz), k)
        return {"idx": idx.view(torch.int32), "d2": d2}
    if op == "radius":
        idx, d2 = pgeof.radius_search(xyz, xyz, case["r"], k)
        return {"idx": idx, "d2": d2}
    if op == "fused":
        capi.knn_features_device(xyz, k, s["nn"], s["ptr"], s["feat"], workspace=s["ws"])
        return {"nn": s["nn"], "ptr": s["ptr"], "feat": s["feat"]}
    if op == "multiscale":
        capi.radius_multiscale_device(xyz, case["r"], k, SCALES, s["nn"], s["ptr"], s["feat"], workspace=s["ws"])
        return {"nn": s["nn"], "ptr": s["ptr"], "feat": s["feat"]}
    if op == "optimal":
        capi.knn_optimal_device(xyz, k, s["nn"], s["ptr"], s["feat"], k_min=10, workspace=s["ws"])
        return {"nn": s["nn"], "ptr": s["ptr"], "feat": s["feat"]}
    if op == "features":
        return {"feat": pgeof.compute_features(xyz, s["nn"], s["ptr"], case["k_min"])}
    if op == "selected":
        return {"feat": pgeof.compute_features_selected(xyz, case["r"], k, s["features"])}
    idx, d2 = pgeof.knn_search(xyz, xyz, k)
    return {"idx": idx, "d2": d2, "feat": pgeof.compute_features(xyz, idx.reshape(-1), s["ptr"])}


# ------------------------------------------------------------------- work ----
def work(case):
    """Compulsory traffic (points read once, every output written once) and
    arithmetic: 8 operations per returned distance, 21 per neighbour of a
    covariance, about 300 per eigensolve and its features."""
    op, n, k = case["op"], case["n"], case["k"]
    if op == "knn":
        m = case["m"] or n
        return {"bytes": 12 * n + (12 * m if case["m"] else 0) + 8 * m * k, "flops": 8 * m * k}
    if op == "radius":
        return {"bytes": 12 * n + 8 * n * k, "flops": 8 * n}
    if op == "fused":
        return {"bytes": 12 * n + 4 * n * k + 4 * n + 44 * n, "flops": n * (29 * k + 300)}
    if op == "multiscale":
        # rows are as full as the density and the cap allow: half the cap counted
        return {"bytes": 12 * n + 2 * n * k + 4 * n + 44 * 4 * n, "flops": n * (29 * (k // 2) + 3 * 300)}
    if op == "optimal":
        return {"bytes": 12 * n + 4 * n * k + 4 * n + 48 * n, "flops": n * (29 * k + 60 * (k - 9) + 300)}
    if op == "features":
        return {"bytes": 12 * n + 2 * n * (k + 1) + 4 * n + 44 * n, "flops": n * (21 * (k + 1) // 2 + 300)}
    if op == "selected":
        return {"bytes": 24 * n + 16 * n, "flops": n * (29 * k + 300)}
    return {"bytes": 12 * n + 8 * n * k + 12 * n + 4 * n * k + 4 * n + 44 * n, "flops": n * (29 * k + 300)}


# ------------------------------------------------------------------ exact ----
def _sq32(q, p):
    """float32 squared distances of every pair, each product and sum rounded."""
    d = q[:, None, 0] - p[None, :, 0]
    s = d * d
    for a in (1, 2):
        d = q[:, None, a] - p[None, :, a]
        s += d * d
    return s


def _neighbours(xyz, query, k):
    """The k nearest rows by the float32 distance, brute force."""
    step = max(1, min(len(query), 200_000_000 // len(xyz)))
    return torch.cat([torch.topk(_sq32(query[i:i + step], xyz), k, dim=1, largest=False, sorted=True)[1]
                      for i in range(0, len(query), step)])


def _d2(xyz, query, idx):
    d = query.double()[:, None, :] - xyz.double()[idx]
    return (d * d).sum(-1)


def _eigh3(c):
    """Eigenpairs (ascending) of symmetric 3x3 matrices by cyclic Jacobi."""
    a = c.clone()
    v = torch.eye(3, dtype=torch.float64, device=c.device).expand_as(a).clone()
    for _ in range(12):
        for p, q in ((0, 1), (0, 2), (1, 2)):
            apq = a[:, p, q]
            small = apq.abs() < 1e-300
            theta = (a[:, q, q] - a[:, p, p]) / (2 * torch.where(small, torch.ones_like(apq), apq))
            t = torch.where(theta >= 0, 1.0, -1.0) / (theta.abs() + torch.sqrt(theta * theta + 1))
            t = torch.where(small, torch.zeros_like(t), t)
            co = 1 / torch.sqrt(t * t + 1)
            si = t * co
            for m in (a, v):
                x, y = m[:, :, p].clone(), m[:, :, q].clone()
                m[:, :, p], m[:, :, q] = co[:, None] * x - si[:, None] * y, si[:, None] * x + co[:, None] * y
            x, y = a[:, p, :].clone(), a[:, q, :].clone()
            a[:, p, :], a[:, q, :] = co[:, None] * x - si[:, None] * y, si[:, None] * x + co[:, None] * y
    val, order = torch.sort(torch.diagonal(a, dim1=1, dim2=2), dim=1, stable=True)
    return val, torch.gather(v, 2, order[:, None, :].expand(-1, 3, 3))


def _features(xyz, nn, ptr, k_min):
    """The 11 features of every CSR row in 64 bits."""
    ptr = ptr.long()
    n, dev = len(ptr) - 1, nn.device
    count = ptr[1:] - ptr[:-1]
    rows = torch.repeat_interleave(torch.arange(n, device=dev), count)
    at = xyz.double()[nn.long()]
    inv = 1.0 / count.clamp(min=1).double()
    mean = torch.zeros(n, 3, dtype=torch.float64, device=dev).index_add_(0, rows, at) * inv[:, None]
    at = at - mean[rows]
    cov = torch.empty(n, 3, 3, dtype=torch.float64, device=dev)
    for p in range(3):
        for q in range(p, 3):
            cov[:, p, q] = torch.zeros(n, dtype=torch.float64, device=dev).index_add_(0, rows, at[:, p] * at[:, q]) * inv
            cov[:, q, p] = cov[:, p, q]
    del at, rows
    out = torch.empty(n, 11, dtype=torch.float64, device=dev)
    for i in range(0, n, 1 << 20):
        val, vec = _eigh3(cov[i:i + (1 << 20)])
        val = val.clamp(min=0.0)
        s0, s1, s2 = (val[:, j].sqrt() for j in (0, 1, 2))  # ascending, as the formulas take them
        normal = vec[:, :, 2]
        normal = torch.where(normal[:, 2:] < 0, -normal, normal)
        u = (val[:, None, :] * vec.abs()).sum(2)
        upright = torch.where(s0 > 0, u[:, 2] / u.norm(dim=1).clamp(min=1e-300), torch.zeros_like(s0))
        out[i:i + (1 << 20)] = torch.stack(
            [(s0 - s1) / (s0 + F_EPS), (s1 - s2) / (s0 + F_EPS), s2 / (s0 + F_EPS), upright,
             normal[:, 0], normal[:, 1], normal[:, 2], s0, (s0 * s1 + 1e-6).sqrt(),
             (s0 * s1 * s2 + 1e-9) ** (1.0 / 3.0), s2 / (s0 + s1 + s2 + F_EPS)], 1)
    out[count < k_min] = 0.0
    return out


def exact(case, seed):
    """run()'s outputs in 64 bits, where brute force can give the neighbours."""
    op, n, k = case["op"], case["n"], case["k"]
    if op == "features":
        s = prepare(case, seed)
        return {"feat": _features(s["xyz"], s["nn"], s["ptr"], case["k_min"])}
    if op not in ("knn", "fused", "host") or n * (case.get("m") or n) > 11_000_000_000:
        return None
    g = _gen(seed)
    xyz = _cloud(case["scene"], n, g)
    query = xyz
    if case.get("m"):
        lo, hi = xyz.amin(0), xyz.amax(0)
        query = (lo + (hi - lo) * (1.1 * _rand(g, case["m"], 3) - 0.05)).float().contiguous()
    idx = _neighbours(xyz, query, k)
    out = {"d2": _d2(xyz, query, idx)}
    if op == "knn":
        return {"idx": None, **out}
    feat = _features(xyz, idx.reshape(-1), torch.arange(n + 1, device=DEV) * k, 1)
    return {"nn": None, "ptr": None, "feat": feat} if op == "fused" else {"idx": None, **out, "feat": feat}
