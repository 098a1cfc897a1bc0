"""Grids that no launch can hold are refused by the argument checks."""

from __future__ import annotations

import ctypes

from kda_bt16 import _hip


def test_recurrence_refuses_more_pairs_than_a_grid_holds():
    a = _hip.KdaBt16Args()
    a.abi_version = _hip.ABI_VERSION
    a.T, a.K, a.V, a.scale, a.lower_bound = 1, 128, 128, 0.1, -5.0
    f = _hip.lib().kda_recurrent_fwd_hip
    a.B, a.H, a.HV = 1 << 24, 1, 1  # 256 threads each: 2^32
    assert f(ctypes.byref(a), None) == -2
    a.B, a.H, a.HV = 1 << 20, 16, 16
    assert f(ctypes.byref(a), None) == -2
    a.B = (1 << 20) - 1  # no tensors
    assert f(ctypes.byref(a), None) == -1
