"""GPU parity of the tile loop that takes both operands through LDS (csrc/mx_wide.hpp) against the oracle: one expert, so
that the token count is the chunk's row count, at the edges of every row-tile class (8 .. 20 row tiles, odd numbers of row
tiles per wave among them, a second chunk behind a full one), K loops of odd and of single slices (the down stage of
I = 128), short last intermediate tiles, every format and both weight orders.  Tolerances are those of test_gpu_moe.py."""

import numpy as np
import pytest

from helpers import dense_case, from_bf16_tensor, mx_case
from oracle import moe as omoe
from test_gpu_moe import REF_MX_CLAMPS, _check, _golden_dense, _golden_mx_options, _run_dense, _run_fp8_row, _run_mx_options

pytestmark = pytest.mark.gpu

# 8, 10, 12, 14, 16, 18, 20 row tiles, each at its last row or one past the class below, and two chunks
ROWS = [128, 129, 192, 193, 224, 256, 257, 288, 289, 320, 577]


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("I", [128, 640])
def test_wide_mx(rows, I):
    c = mx_case(rows, 512, I, 1, 1, 128, seed=41, skip_token=True, bias=True, weight_format="e4m3", random_codes=True)
    o = from_bf16_tensor(_run_mx_options(c, 3, REF_MX_CLAMPS, False))
    _check(o[0, :rows], _golden_mx_options(c, 3, REF_MX_CLAMPS)[:rows], f"wide mx rows={rows} I={I}")


@pytest.mark.parametrize("rows,fmt,copies", [(200, "e5m2", True), (300, "e5m2", False), (320, "e4m3", False), (193, "e4m3", False),
                                              (128, "e2m1", True), (256, "e2m1", False), (320, "e2m1", True), (577, "e2m1", False)])
def test_wide_mx_formats_and_layouts(rows, fmt, copies):
    from nkilib.core.moe.moe_cte import _launch

    c = mx_case(rows, 1024, 384, 1, 1, 128, seed=42, bias=False, weight_format=fmt, random_codes=True)
    was = _launch.mx_weight_copies
    try:
        _launch.mx_weight_copies = copies
        o = from_bf16_tensor(_run_mx_options(c, 0, {}, False))
    finally:
        _launch.mx_weight_copies = was
    _check(o[0, :rows], _golden_mx_options(c, 0, {})[:rows], f"wide mx {fmt} rows={rows} copies={copies}")


@pytest.mark.parametrize("rows", [128, 256, 257, 320, 577])
@pytest.mark.parametrize("I,fp8w,mode", [(64, False, 1), (320, True, 2), (512, False, 0)])
def test_wide_bf16(rows, I, fp8w, mode):
    c = dense_case(rows, 512, I, 1, 1, 128, seed=43, bias=fp8w, quant=fp8w, hidden_std=1.0)
    o = from_bf16_tensor(_run_dense(c, impl="shard_on_i", mode=mode, fp8_weights=fp8w))
    _check(o[:rows], _golden_dense(c, mode=mode, fp8_weights=fp8w)[:rows], f"wide bf16 rows={rows} I={I}")


@pytest.mark.parametrize("rows,I", [(128, 128), (256, 384), (320, 640), (577, 512)])
def test_wide_fp8_row(rows, I):
    c = dense_case(rows, 512, I, 1, 1, 128, seed=44, quant=True, bias=True, hidden_std=1.0)
    rec, out = _run_fp8_row(c, np.ones((1, 512), np.float32), act=3)
    import torch

    raw = rec.view(torch.uint8).cpu().numpy()
    g = omoe.moe_blockwise_fp8_row_ref(raw[:, :512], raw[:, 512:].copy().view(np.float32).reshape(-1), c["aff"], c["gate_up_q"],
                                       c["down_q"], c["gate_up_scale"], c["down_scale"], c["tp2id"], c["b2e"], c["B"],
                                       gate_up_proj_bias=c["gate_up_bias"], down_proj_bias=c["down_bias"],
                                       activation_function=3, expert_affinities_scaling_mode=1)
    o = from_bf16_tensor(out)
    _check((o[:rows, 0] if o.ndim == 3 else o[:rows]), g[:rows], f"wide fp8 row rows={rows} I={I}")
