"""GPU parity of the large-tile kernels where a launch's last round of tiles is cut into pieces by rows (a launch of few tiles,
or few of them behind full rounds), at the edges of the row-tile counts: 128 / 129 rows (not cut / cut), pieces that the last
one does not need, 256 / 257, 288 / 289 and 320 rows, and two rounds in turns.  Tolerances are those of test_gpu_moe.py."""

import numpy as np
import pytest

from helpers import dense_case, from_bf16_tensor, mx_case
from oracle import moe as omoe
from test_gpu_moe import REF_MX_CLAMPS, _check, _golden_dense, _golden_mx_options, _run_dense, _run_fp8_row, _run_mx_options

pytestmark = pytest.mark.gpu

ROWS = [128, 129, 193, 225, 257, 289, 320, 321]


@pytest.mark.parametrize("T", ROWS)
@pytest.mark.parametrize("fmt", ["e4m3", "e2m1"])
def test_pieces_mx(T, fmt):
    c = mx_case(T, 512, 384, 1, 1, 128, seed=61, bias=True, weight_format=fmt)
    o = from_bf16_tensor(_run_mx_options(c, 3, REF_MX_CLAMPS, False))
    _check(o[0, :T], _golden_mx_options(c, 3, REF_MX_CLAMPS)[:T], f"pieces mx {fmt} T={T}")


@pytest.mark.parametrize("T", ROWS)
def test_pieces_dense(T):
    c = dense_case(T, 512, 200, 1, 1, 128, seed=62, bias=True, hidden_std=1.0)
    o = from_bf16_tensor(_run_dense(c, act=0, mode=1)).reshape(T + 1, -1, 512)[:, 0]  # (with or without the second plane)
    _check(o[:T], _golden_dense(c, act=0, mode=1)[:T], f"pieces bf16 T={T}")


@pytest.mark.parametrize("T", [130, 290])
def test_pieces_fp8_row(T):
    c = dense_case(T, 512, 256, 1, 1, 128, seed=63, quant=True, bias=True, hidden_std=1.0)
    rec, out = _run_fp8_row(c, np.ones((1, 512), np.float32), act=3, clamps={})
    import torch

    raw = rec.view(torch.uint8).cpu().numpy()
    g = omoe.moe_blockwise_fp8_row_ref(raw[:, :512], raw[:, 512:].copy().view(np.float32).reshape(-1), c["aff"],
                                       c["gate_up_q"], c["down_q"], c["gate_up_scale"], c["down_scale"], c["tp2id"],
                                       c["b2e"], c["B"], gate_up_proj_bias=c["gate_up_bias"],
                                       down_proj_bias=c["down_bias"], activation_function=3)
    _check(from_bf16_tensor(out).reshape(T + 1, -1, 512)[:T, 0], g[:T], f"pieces fp8 row T={T}")


def test_rounds_in_turns():
    """16 experts of about 200 rows over 18 column tiles: 36 items on every XCD, a full round of 32 and 4 that are cut."""
    c = mx_case(1600, 512, 2304, 16, 2, 128, seed=64)
    o = from_bf16_tensor(_run_mx_options(c, 0, None, False))
    _check(o[0, :1600], _golden_mx_options(c, 0, None)[:1600], "two rounds mx")
    again = from_bf16_tensor(_run_mx_options(c, 0, None, False))
    assert np.array_equal(o, again)
