"""CSR feature kernels: rows whose lengths are multiples of four (every kNN
CSR with k a multiple of 4), read four indices per load without shifts."""
import time

import numpy as np
import pytest
import torch

import point_geometric_features_amd as pgeof
from oracle import oracle as O
from point_geometric_features_amd import capi, scenes

from tests.parity import assert_features_close

pytestmark = pytest.mark.gpu


def test_waves_of_whole_and_mixed_rows():
    """128 rows of 0, 4, .. 68 entries (waves of whole quads) at every 4-byte
    offset, against the oracle and, bit for bit, against the same rows in
    waves that a row of 5 makes mixed."""
    xyz = scenes.lidar_scene(5_000, seed=78, extent=8.0)
    idx, _ = pgeof.knn_search(xyz, xyz, 70)
    lens = np.tile(np.arange(18) * 4, 8)[:128]
    rows = [idx[100 + n, :m] for n, m in enumerate(lens)]
    sc = [4, 8, 20, 33, 68]

    def run(rows, shift):
        nn = np.concatenate([idx[0, :shift], *rows]).astype(np.uint32)
        ptr = np.r_[0, np.cumsum([shift, *map(len, rows)])].astype(np.uint32)
        ptr = ptr[1:]  # the entries in front belong to no row
        return (pgeof.compute_features(xyz, nn, ptr), pgeof.compute_features_multiscale(xyz, nn, ptr, sc),
                pgeof.compute_features_optimal(xyz, nn, ptr, 3, 2, 5))

    whole = run(rows, 0)
    nn = np.concatenate(rows).astype(np.uint32)
    ptr = np.r_[0, np.cumsum(lens)].astype(np.uint32)
    assert_features_close(whole[0], O.compute_features(xyz, nn, ptr), O.eigvals_csr_np(xyz, nn, ptr), "whole quads")
    for shift in (1, 2, 3):
        for a, b in zip(run(rows, shift), whole):
            np.testing.assert_array_equal(a, b)
    mixed = [r for n, row in enumerate(rows) for r in ([idx[7, :5], row] if n % 16 == 0 else [row])]
    keep = [n for n, r in enumerate(mixed) if len(r) != 5]
    for a, b in zip(run(mixed, 0), whole):
        np.testing.assert_array_equal(a[keep], b)


def test_aligned_rows_time():
    """6 M rows of 20 against their first 16 entries, in turns: 1.14 times as
    long with aligned 16-byte loads, 1.12 with unaligned ones and no shifts,
    1.20 when every group of four was shifted.  The limit lies at 1.165."""
    n = 6_000_000
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    x = torch.rand(n, 3, generator=g, device="cuda")
    x[:, 2] *= 0.01
    nn = torch.empty(n * 20, dtype=torch.int32, device="cuda")
    ptr = torch.empty(n + 1, dtype=torch.int32, device="cuda")
    f = torch.empty(n, 11, device="cuda")
    capi.knn_features_device(x, 20, nn, ptr, f)
    nn16 = nn.view(n, 20)[:, :16].reshape(-1).contiguous()
    ptr16 = (torch.arange(n + 1, device="cuda") * 16).int()

    def ms(nn, ptr):
        torch.cuda.synchronize()
        t = time.perf_counter()
        for _ in range(3):
            pgeof.compute_features(x, nn, ptr)
        torch.cuda.synchronize()
        return time.perf_counter() - t

    ratio = np.median([ms(nn, ptr) / ms(nn16, ptr16) for _ in range(12)])
    print(f"rows of 20 over rows of 16: {ratio:.3f}")
    assert ratio < 1.165
