"""The kept call plans against the library's own answers (no GPU needed)."""
import ctypes

import pytest

from memory_efficient_attn_layer_amd import _lib


@pytest.mark.parametrize("which", [_lib.MEA_PASS_FWD, _lib.MEA_PASS_BWD, _lib.MEA_PASS_BWD_TABLES])
@pytest.mark.parametrize("B,T,T_max,T_ws", [(2, 77, 77, 77), (1, 500, 130, 500), (1, 64, 96, 96), (0, 8, 8, 8)])
def test_plan_matches_the_library(which, B, T, T_max, T_ws):
    lib = _lib.load()
    for b16 in (False, True):
        d, n = _lib.plan(B, T, 96, 2, 64, T_max, 1e-6, 0, b16, which, T_ws)
        assert (d.B, d.T, d.C, d.H, d.N, d.T_max, d.N_active, d.tables_bf16) == (B, T, 96, 2, 64, T_max, 0, int(b16))
        assert n == lib.mea_workspace_bytes(ctypes.byref(_lib.desc(B, T, 96, 2, 64, T_ws, 1e-6, 0, b16)), which)
    d, n = _lib.decode_plan(max(B, 1), T, 96, 2, 64, 1e-6, 0)
    assert n == lib.mea_decode_workspace_bytes(ctypes.byref(d)) > 0
