"""The general search (a lane per query with a heap) where calls of k <= 108
take the wave-per-query one: its knobs, heap layouts and passes with
wave_k_max = 0, against the oracle."""
import numpy as np
import pytest
import torch

import point_geometric_features_amd as pgeof
from oracle import oracle as O
from point_geometric_features_amd import capi, scenes

from tests.test_gpu_search import _KNOB_SETS

pytestmark = pytest.mark.gpu


class _Knobs:
    def __init__(self, **knobs):
        self.knobs = knobs

    def __enter__(self):
        self.old = {k: capi.get_tuning(k) for k in self.knobs}
        for k, v in self.knobs.items():
            capi.set_tuning(k, v)

    def __exit__(self, *exc):
        for k, v in self.old.items():
            capi.set_tuning(k, v)


def _fused(xyz, k):
    x, n = torch.from_numpy(xyz).cuda(), len(xyz)
    out = [torch.empty(n * k, dtype=torch.int32, device="cuda"), torch.empty(n + 1, dtype=torch.int32, device="cuda"),
           torch.empty(n, 11, device="cuda")]
    ws = torch.empty(capi.knn_workspace_size(n, n, k), dtype=torch.uint8, device="cuda")
    capi.knn_features_device(x, k, *out, workspace=ws)
    return out[0].cpu().numpy().view(np.uint32).reshape(n, k), out[2].cpu().numpy()


def _cloud(n=50_000):
    return scenes.lidar_scene(n, seed=29, extent=20.0)


@pytest.fixture(scope="module")
def oracle_rows():
    xyz = _cloud()
    return {k: O.knn(xyz, xyz, k, kdtree=True) for k in (16, 50)}


@pytest.mark.parametrize("knobs", [*_KNOB_SETS, {"near_first": 0}, {"near_first": 1}, {"heap_tail": 2},
                                   {"heap_tail": 2, "staging": 2}],
                         ids=lambda d: ",".join(f"{k}={v}" for k, v in d.items()))
@pytest.mark.parametrize("k", [16, 50])
def test_knobs(knobs, k, oracle_rows):
    xyz = _cloud()
    with _Knobs(wave_k_max=0, **knobs):
        gi, gd = pgeof.knn_search(xyz, xyz, k)
        nn, f = _fused(xyz, k)
    oi, od = oracle_rows[k]
    np.testing.assert_array_equal(gi, oi)
    np.testing.assert_array_equal(gd, od)
    np.testing.assert_array_equal(nn, oi)
    ptr = (np.arange(len(xyz) + 1) * k).astype(np.uint32)
    np.testing.assert_array_equal(f, pgeof.compute_features(xyz, nn.reshape(-1), ptr))


@pytest.mark.parametrize("knobs", [{}, {"heap_tail": 0}, {"staging": 1}, {"lds_budget": 4096}, {"near_first": 0}],
                         ids=lambda d: ",".join(f"{k}={v}" for k, v in d.items()) or "default")
@pytest.mark.parametrize("cap", [24, 64])
def test_radius_knobs(knobs, cap):
    xyz = _cloud()
    oi, od, _ = O.radius(xyz, xyz, 0.3, cap, kdtree=True)
    with _Knobs(wave_k_max=0, **knobs):
        gi, gd = pgeof.radius_search(xyz, xyz, 0.3, cap)
    np.testing.assert_array_equal(gi, oi)
    np.testing.assert_array_equal(gd, od)


@pytest.mark.parametrize("heap_tail", [1, 2])
@pytest.mark.parametrize("k", [22, 50])
def test_lattice_ties(k, heap_tail):
    """Keys that differ by index only, sifted through the heaps' tails."""
    xyz = np.stack(np.meshgrid(*[np.arange(18)] * 3), -1).reshape(-1, 3).astype(np.float32)
    xyz = xyz[np.random.default_rng(0).permutation(len(xyz))]
    oi, od = O.knn(xyz, xyz, k, kdtree=False)
    with _Knobs(wave_k_max=0, heap_tail=heap_tail):
        gi, gd = pgeof.knn_search(xyz, xyz, k)
        nn, _ = _fused(xyz, k)
    np.testing.assert_array_equal(gi, oi)
    np.testing.assert_array_equal(gd, od)
    np.testing.assert_array_equal(nn, oi)


@pytest.mark.parametrize("r,cap", [(1.0, 1), (1.0, 12), (1.0, 21), (1.0, 22), (1.0, 30), (0.3, 60)])
@pytest.mark.parametrize("name", ["lattice", "one_point", "one_far", "plane"])
def test_radius_shapes(name, r, cap):
    """Radius searches on both sides of cap 21, where the wave search begins."""
    rng = np.random.default_rng(1)
    xyz = {"lattice": np.floor(rng.random((6000, 3)) * 10), "one_point": np.full((3000, 3), 2.5),
           "one_far": np.concatenate([rng.random((5000, 3)) * 4, [[1e4, 0, 0]]]),
           "plane": rng.random((6000, 3)) * [20, 20, 0]}[name].astype(np.float32)
    q = xyz[:400]
    oi, od, _ = O.radius(xyz, q, r, cap, kdtree=False)
    gi, gd = pgeof.radius_search(xyz, q, r, cap)
    np.testing.assert_array_equal(gi, oi)
    np.testing.assert_array_equal(gd, od)


@pytest.mark.parametrize("n", [65_569, 65_633, 2_097_153])
@pytest.mark.parametrize("hits,cap", [(14, 22), (20, 30), (24, 100), (30, 31)])
def test_radius_pairs(n, hits, cap):
    """Balls of about `hits` points in a volume, rows of the last and first
    queries of a group against the oracle."""
    xyz = scenes.uniform_cube(n, seed=hits)
    r = float((hits / n / (4 / 3 * np.pi)) ** (1 / 3))
    x = torch.from_numpy(xyz).cuda()
    gi, gd = (a.cpu().numpy() for a in pgeof.radius_search(x, x, r, cap))
    rows = np.r_[0:15, n - 15 : n, np.random.default_rng(3).integers(0, n, 20)]
    oi, od, _ = O.radius(xyz, np.ascontiguousarray(xyz[rows]), r, cap, kdtree=False)
    np.testing.assert_array_equal(gi[rows], oi)
    np.testing.assert_array_equal(gd[rows], od)


def test_autotune_times_no_knob_set_twice():
    """Sets that differ only in knobs that the chosen search reads not are one
    candidate: row staging of a radius search by wave with its features after
    it, staging and LDS heaps of a kNN by wave."""
    x = torch.from_numpy(_cloud(20_000)).cuda()
    try:
        sets = capi.autotune("radius_multiscale", x, 40, radius=0.3, k_scales=[10, 40], reps=1)["candidates"]
        seen = [tuple(v for name, v in s.items() if name != "staging") for s in sets if s["fuse_multiscale"] == 0]
        assert len(seen[1:]) == len(set(seen[1:])) == 4
        sets = capi.autotune("knn_features", x, 20, reps=1)["candidates"][1:]
        seen = [tuple(v for name, v in s.items() if name not in ("staging", "lds_budget")) for s in sets]
        assert len(seen) == len(set(seen))
        with _Knobs(wave_k_max=0):
            general = capi.autotune("radius_multiscale", x, 40, radius=0.3, k_scales=[10, 40], reps=1)["candidates"]
        assert sum(s["fuse_multiscale"] == 0 for s in general[1:]) == 8
    finally:
        capi.autotune_clear()
