"""The knob of the wave-per-query search: its default, its limits and its
place in the header's list."""
import os

import pytest

from point_geometric_features_amd import capi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_wave_k_max():
    assert capi.get_tuning("wave_k_max") == 108.0
    try:
        capi.set_tuning("wave_k_max", 0)
        assert capi.get_tuning("wave_k_max") == 0.0
        with pytest.raises(ValueError):
            capi.set_tuning("wave_k_max", -1.0)
    finally:
        capi.set_tuning("wave_k_max", 108)
    with open(os.path.join(ROOT, "include", "pgeof_hip.h")) as f:
        assert '"wave_k_max"' in f.read()
