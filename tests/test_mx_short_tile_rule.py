"""That MX calls with a short last tile (I % 128 != 0) have no weight copies, and that the calls which the large-tile kernels cannot
address are still taken (by the general kernel)."""

import ctypes

import pytest

from test_cabi import _valid_args


@pytest.mark.parametrize("I,col_tiles", [(32, 1), (480, 4), (512, 4), (544, 5), (640, 5), (2880, 23)])
def test_copies_are_of_whole_column_tiles_only(I, col_tiles):
    """Where I is no multiple of 128 the weights are read in place (and a call is planned whatever their alignment)."""
    from nkilib import _native as nv

    L = nv.lib()
    H, E = 1024, 4
    for dt, slice_bytes in ((nv.DT_FP8, 32768), (nv.DT_FP4_E2M1, 16384)):
        a = _valid_args(nv, nv.KIND_MXFP8, 129, H, I, E, 128, 8, dt)
        nbytes = lambda which: L.moe_kmajor_weights_bytes(ctypes.byref(a), which)
        whole = I % 128 == 0
        assert nbytes(0) == (E * col_tiles * (H // 128) * slice_bytes if whole else 0)
        assert nbytes(1) == (E * (H // 256) * col_tiles * slice_bytes if whole and dt == nv.DT_FP4_E2M1 else 0)
        a.gate_up_proj_weight = ctypes.c_void_p(4096 + 4)
        assert (nbytes(0) > 0) == whole and L.moe_blockwise_workspace_bytes(ctypes.byref(a)) > 0


def test_calls_past_the_offsets_are_taken_for_short_tiles_only():
    from nkilib import _native as nv

    L = nv.lib()
    ws = lambda a: L.moe_blockwise_workspace_bytes(ctypes.byref(a))
    big = lambda I: _valid_args(nv, nv.KIND_MXFP8, 2**32 // 7168 + 1, 7168, I, 256, 128, 766, nv.DT_FP8)
    assert ws(big(2048)) == 0 and ws(big(2080)) > 0
