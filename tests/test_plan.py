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


def test_workspaces_hold_what_the_kernels_touch():
    """No rows for an O that only a caller's o_save takes; no fp32 weight
    gradients where one token split writes them as bf16."""
    lib = _lib.load()
    d = _lib.desc(4, 4096, 1024, 16, 64, 4096, 1e-6)
    act, weights = 4 * 4096 * 1024 * 2, 4 * 1024 * 1024 * 2
    fwd = lib.mea_workspace_bytes(ctypes.byref(d), _lib.MEA_PASS_FWD)
    assert 4 * act + weights < fwd < 4 * act + weights + act // 2  # q, k, v, sig and the packed weights
    B, T, C, HN = 1, 256, 2048, 2048
    d = _lib.desc(B, T, C, 16, 128, T, 1e-6)
    bwd = lib.mea_workspace_bytes(ctypes.byref(d), _lib.MEA_PASS_BWD)
    known = 7 * T * HN * 2 + (4 + 4 + 1) * HN * C * 2 + T * C * 4  # rows, three weight layouts, the tiled dx's sums
    assert known < bwd < known + HN * C * 4
