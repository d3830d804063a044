"""kNN with one wave per query against the lane-per-query search and the oracle.

The wave kernel serves k <= 108; wave_k_max = 0 sends the same call to the
general path, which must give the same indices and squared distances bit for
bit, and the fused features the bits of compute_features on that CSR.
"""
import numpy as np
import pytest
import torch

import point_geometric_features_amd as pgeof
from oracle import oracle as O
from point_geometric_features_amd import capi, scenes

pytestmark = pytest.mark.gpu


class _Knobs:
    def __init__(self, **kw):
        self.kw = kw

    def __enter__(self):
        self.old = {k: capi.get_tuning(k) for k in self.kw}
        for k, v in self.kw.items():
            capi.set_tuning(k, v)

    def __exit__(self, *exc):
        for k, v in self.old.items():
            capi.set_tuning(k, v)


def _both(data, query, k, **knobs):
    with _Knobs(**knobs):
        gi, gd = pgeof.knn_search(data, query, k)
    with _Knobs(wave_k_max=0):
        ri, rd = pgeof.knn_search(data, query, k)
    np.testing.assert_array_equal(gi, ri)
    np.testing.assert_array_equal(gd, rd)
    return gi, gd


def _fused(xyz, k):
    x = torch.from_numpy(xyz).cuda()
    nn = torch.empty(len(xyz) * k, dtype=torch.int32, device="cuda")
    ptr = torch.empty(len(xyz) + 1, dtype=torch.int32, device="cuda")
    f = torch.empty((len(xyz), 11), dtype=torch.float32, device="cuda")
    d = torch.empty(len(xyz) * k, dtype=torch.float32, device="cuda")
    capi.knn_features_device(x, k, nn, ptr, f, sqr_dist=d)
    torch.cuda.synchronize()
    return nn.cpu().numpy().view(np.uint32).reshape(-1, k), d.cpu().numpy().reshape(-1, k), f.cpu().numpy()


# row classes of the kernel end at 12, 27, 54 and 108 (109: the general path)
@pytest.mark.parametrize("k", [1, 11, 12, 13, 16, 27, 28, 32, 48, 54, 55, 64, 65, 96, 108, 109])
@pytest.mark.parametrize("scene", ["lidar", "cube"])
def test_row_classes(scene, k):
    xyz = scenes.lidar_scene(40_003, seed=k, extent=18.0) if scene == "lidar" else scenes.uniform_cube(40_003, seed=k)
    gi, gd = _both(xyz, xyz, k)
    rows = np.random.default_rng(k).choice(len(xyz), 500, replace=False)
    oi, od = O.knn(xyz, xyz[rows], k, kdtree=True)
    np.testing.assert_array_equal(gi[rows], oi)
    np.testing.assert_array_equal(gd[rows], od)
    fi, fd, f = _fused(xyz, k)
    np.testing.assert_array_equal(fi, gi)
    np.testing.assert_array_equal(fd, gd)
    nn, ptr = scenes.knn_csr(gi)
    np.testing.assert_array_equal(f, pgeof.compute_features(xyz, nn, ptr))


@pytest.mark.parametrize("n", [1, 2, 3, 63, 64, 65, 257, 1000])
def test_small_clouds(n):
    xyz = scenes.uniform_cube(n, seed=n)
    for k in sorted({1, min(n, 5), min(n, 64), min(n, 100)}):
        gi, gd = _both(xyz, xyz, k)
        oi, od = O.knn(xyz, xyz, k, kdtree=False)
        np.testing.assert_array_equal(gi, oi)
        np.testing.assert_array_equal(gd, od)


def _clouds():
    rng = np.random.default_rng(5)
    lattice = np.stack(np.meshgrid(*[np.arange(12)] * 3, indexing="ij"), -1).reshape(-1, 3).astype(np.float32)
    dense = rng.normal(0, 0.05, size=(20_000, 3))
    far = rng.uniform(-50, 50, size=(300, 3))
    line = np.zeros((5000, 3))
    line[:, 0] = rng.uniform(0, 100, 5000)
    return {
        "lattice": np.concatenate([lattice, lattice[::-1] * np.float32(2)]),
        "one_point": np.full((3000, 3), 7.25, np.float32),
        "few_values": rng.integers(0, 3, size=(6000, 3)).astype(np.float32),
        "outliers": np.concatenate([dense, far]).astype(np.float32),
        "one_far": np.concatenate([rng.normal(0, 0.1, size=(4000, 3)), [[900.0, -700.0, 300.0]]]).astype(np.float32),
        "line": line.astype(np.float32),
        "plane_far": (np.c_[rng.uniform(0, 30, (15_000, 2)), np.zeros(15_000)] + [1e5, 1e5, 0]).astype(np.float32),
        "spike": np.concatenate([rng.uniform(0, 1, (9000, 3)), 0.5 + 1e-4 * rng.normal(size=(9000, 3))]).astype(np.float32),
    }


@pytest.mark.parametrize("name", ["lattice", "one_point", "few_values", "outliers", "one_far", "line", "plane_far",
                                  "spike"])
@pytest.mark.parametrize("k", [9, 20, 50, 100])
def test_shapes(name, k):
    """Ties at the k-th place, duplicates, isolated points (cubes that grow),
    regions too full for the registers, flat and far clouds."""
    xyz = np.ascontiguousarray(_clouds()[name])
    gi, gd = _both(xyz, xyz, k)
    rows = np.random.default_rng(k).choice(len(xyz), 300, replace=False)
    rows[-1] = len(xyz) - 1
    oi, od = O.knn(xyz, xyz[rows], k, kdtree=False)
    np.testing.assert_array_equal(gi[rows], oi)
    np.testing.assert_array_equal(gd[rows], od)


@pytest.mark.parametrize("k", [5, 20, 40, 80])
def test_queries_off_the_data(k):
    rng = np.random.default_rng(k)
    data = scenes.lidar_scene(30_001, seed=k, extent=15.0)
    q = rng.uniform(-200, 220, size=(3001, 3)).astype(np.float32)
    q[::2] = rng.uniform(-1, 16, size=(1501, 3)).astype(np.float32)
    q[7] = [np.nan, 0, 0]
    q[8] = [0, np.inf, 0]
    gi, gd = _both(data, q, k)
    assert (gi[7] == 0xFFFFFFFF).all() and np.isinf(gd[8]).all()
    ok = np.setdiff1d(np.arange(len(q)), [7, 8])
    oi, od = O.knn(data, q[ok], k, kdtree=False)
    np.testing.assert_array_equal(gi[ok], oi)
    np.testing.assert_array_equal(gd[ok], od)


def test_data_that_is_not_finite():
    xyz = scenes.uniform_cube(3000, seed=3)
    xyz[10] = [np.nan, 0.5, 0.5]
    xyz[20] = [np.inf, 0.5, 0.5]
    q = scenes.uniform_cube(300, seed=4)
    _both(xyz, q, 20)
    small = xyz[:30].copy()  # rows that need the points without a finite distance
    _both(small, q, 28)


@pytest.mark.parametrize("knobs", [{"grid_levels": 1}, {"grid_levels": 4}, {"grid_levels": 3, "grid_level_ratio": 4},
                                   {"knn_occupancy": 0.05, "grid_cells_per_point": 32}, {"knn_occupancy": 3.0},
                                   {"grid_cells_per_point": 1, "grid_levels": 1}],
                         ids=lambda d: ",".join(f"{k}={v}" for k, v in d.items()))
@pytest.mark.parametrize("k", [20, 60])
def test_grids(knobs, k):
    xyz = scenes.lidar_scene(50_000, seed=29, extent=20.0)
    _both(xyz, xyz, k, **knobs)


# ------------------------------------------------------------------ radius ----
def _radius_both(data, query, r, cap, **knobs):
    with _Knobs(**knobs):
        gi, gd = pgeof.radius_search(data, query, r, cap)
    with _Knobs(wave_k_max=0):
        ri, rd = pgeof.radius_search(data, query, r, cap)
    np.testing.assert_array_equal(gi, ri)
    np.testing.assert_array_equal(gd, rd)
    return gi, gd


# from a point or none in the ball (a query per lane) to more than the cap
@pytest.mark.parametrize("r", [0.01, 0.05, 0.15, 0.4, 1.5])
@pytest.mark.parametrize("cap", [1, 12, 13, 30, 54, 64, 108, 109])
def test_radius(r, cap):
    xyz = scenes.lidar_scene(30_001, seed=cap, extent=15.0)
    gi, gd = _radius_both(xyz, xyz, r, cap)
    rows = np.random.default_rng(cap).choice(len(xyz), 300, replace=False)
    oi, od, _ = O.radius(xyz, xyz[rows], r, cap, kdtree=True)
    np.testing.assert_array_equal(gi[rows], oi)
    np.testing.assert_array_equal(gd[rows], od)


@pytest.mark.parametrize("name", ["lattice", "one_point", "few_values", "outliers", "one_far", "plane_far", "spike"])
@pytest.mark.parametrize("r,cap", [(1.0, 20), (0.3, 60), (2.0, 100)])
def test_radius_shapes(name, r, cap):
    xyz = np.ascontiguousarray(_clouds()[name])
    _radius_both(xyz, xyz, r, cap)


# 2, 8, 32 and 64 queries per wave; sparse ones (one per lane, up to 16 hits)
# are shared by the waves of 64 queries, the last wave being short
@pytest.mark.parametrize("n", [4_099, 16_421, 65_601, 2_097_219])
@pytest.mark.parametrize("hits", [2, 12, 30])
def test_radius_waves(n, hits):
    xyz = scenes.uniform_cube(n, seed=hits)
    xyz[n // 2 : n // 2 + 40] = xyz[0]  # a dense spot among them
    edge = float(np.ptp(xyz[:, 0]))
    _radius_both(xyz, xyz, edge * float(np.cbrt(hits / (4.19 * n))), 30)


# two lanes per query: 16 to 32 hits, caps below and above them, a last half
# of 1, 31, 32 or 33 queries, one and two waves per 64 queries
@pytest.mark.parametrize("n", [65_569, 65_599, 65_632, 65_633, 2_097_153])
@pytest.mark.parametrize("hits,cap", [(14, 21), (14, 22), (20, 30), (20, 64), (24, 100), (30, 31)])
def test_radius_pairs(n, hits, cap):
    rng = np.random.default_rng(hits)
    side = 40 if n < 1_000_000 else 127
    at = np.stack(np.unravel_index(np.arange(n) % side**3, (side,) * 3), 1)  # jittered lattice: even density
    xyz = (at + rng.uniform(-0.3, 0.3, (n, 3))).astype(np.float32)
    xyz[n // 3 : n // 3 + 50] = xyz[5]  # and a spot of 50
    data = xyz[rng.permutation(n)].copy()
    density = n / side**3
    _radius_both(data, data, float(np.cbrt(hits / (4.19 * density))), cap)


@pytest.mark.parametrize("r", [0.0, 1e-30, np.inf, -0.5])
def test_radius_values(r):
    xyz = scenes.uniform_cube(2000, seed=8)
    xyz[1] = xyz[0]
    xyz[5] = [np.nan, 0, 0]
    q = np.concatenate([xyz, scenes.uniform_cube(100, seed=9) * np.float32(5) - np.float32(2)])
    q[11] = [np.inf, 0, 0]
    _radius_both(xyz, np.ascontiguousarray(q), r, 40)


def test_radius_queries_off_the_data():
    rng = np.random.default_rng(3)
    data = scenes.lidar_scene(20_001, seed=2, extent=12.0)
    q = rng.uniform(-30, 50, size=(3001, 3)).astype(np.float32)
    q[::2] = rng.uniform(-1, 13, size=(1501, 3)).astype(np.float32)
    for r in (0.3, 8.0):
        _radius_both(data, q, r, 50)


@pytest.mark.parametrize("knobs", [{"grid_levels": 1}, {"grid_levels": 2}, {"radius_cell_factor": 0.2},
                                   {"radius_cell_factor": 1.5}, {"grid_cells_per_point": 1}],
                         ids=lambda d: ",".join(f"{k}={v}" for k, v in d.items()))
def test_radius_grids(knobs):
    xyz = scenes.lidar_scene(50_000, seed=29, extent=20.0)
    _radius_both(xyz, xyz, 0.35, 50, **knobs)


@pytest.mark.parametrize("r", [0.05, 0.5])
def test_radius_csr(r):
    xyz = scenes.lidar_scene(60_000, seed=6, extent=25.0)
    x = torch.from_numpy(xyz).cuda()
    out = []
    for kmax in (108, 0):
        with _Knobs(wave_k_max=kmax):
            nn = torch.zeros(len(xyz) * 64, dtype=torch.int32, device="cuda")
            ptr = torch.empty(len(xyz) + 1, dtype=torch.int32, device="cuda")
            nnz = capi.radius_csr_device(x, r, 64, nn, ptr)
            out.append((nnz, nn.cpu().numpy(), ptr.cpu().numpy()))
    assert out[0][0] == out[1][0]
    np.testing.assert_array_equal(out[0][1], out[1][1])
    np.testing.assert_array_equal(out[0][2], out[1][2])


# the grid's levels are built at once or after level 0 (65,536 points), with 4
# or 16 points per thread (262,144), and few queries stay unsorted (8,192)
@pytest.mark.parametrize("n", [65_535, 65_536, 65_537, 262_144, 262_145])
@pytest.mark.parametrize("m", [8_192, 8_193])
@pytest.mark.parametrize("levels", [1, 2, 3, 4])
def test_grid_builds(n, m, levels):
    data = scenes.lidar_scene(n, seed=levels, extent=40.0)
    q = np.ascontiguousarray(data[np.random.default_rng(m).permutation(n)[:m]] + np.float32(0.01))
    _both(data, q, 12, grid_levels=levels)
    rows = slice(0, 400)
    oi, od = O.knn(data, q[rows], 12, kdtree=True)
    with _Knobs(grid_levels=levels):
        gi, gd = pgeof.knn_search(data, q, 12)
    np.testing.assert_array_equal(gi[rows], oi)
    np.testing.assert_array_equal(gd[rows], od)


def test_fused_row_offsets():
    for n, k in ((1, 1), (63, 20), (4097, 108), (4097, 109)):
        x = torch.from_numpy(scenes.uniform_cube(n, seed=n)).cuda()
        k = min(k, n)
        nn = torch.empty(n * k, dtype=torch.int32, device="cuda")
        ptr = torch.full((n + 1,), -1, dtype=torch.int32, device="cuda")
        f = torch.empty((n, 11), dtype=torch.float32, device="cuda")
        capi.knn_features_device(x, k, nn, ptr, f)
        np.testing.assert_array_equal(ptr.cpu().numpy(), np.arange(n + 1) * k)


def test_queries_far_from_a_large_cloud():
    """Balls that grow from far outside the grid must not take the whole cloud
    at once (they would hold every point of it)."""
    data = scenes.lidar_scene(300_000, seed=5, extent=60.0)
    q = np.random.default_rng(1).uniform(-3000, 3000, size=(200, 3)).astype(np.float32)
    gi, gd = _both(data, q, 16)
    oi, od = O.knn(data, q, 16, kdtree=True)
    np.testing.assert_array_equal(gi, oi)
    np.testing.assert_array_equal(gd, od)
