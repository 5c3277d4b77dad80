"""GPU parity of the tile loop that takes both operands through LDS (csrc/mx_wide.hpp) against the oracle: one expert, so
that the token count is the chunk's row count, at the edges of every row-tile class (8 .. 20 row tiles, odd numbers of row
tiles per wave among them, a second chunk behind a full one), K loops of odd and of single slices (the down stage of
I = 128), short last intermediate tiles, every format and both weight orders; several experts of different chunk counts, so
that a workgroup goes from tile to tile of several classes; ROW records on aligned copies of their codes.  Tolerances are
those of test_gpu_moe.py."""

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


def _of_tokens(c, tokens):
    """The same layer over some of its tokens."""
    T, B, mask = len(tokens), c["B"], c["mask"][tokens]
    tp, b2e = [], []
    for e in range(c["E"]):
        rows = np.nonzero(mask[:, e])[0]
        n = -(-len(rows) // B)
        tp.append(np.pad(rows, (0, n * B - len(rows)), constant_values=T))
        b2e += [e] * n
    rows = np.append(tokens, c["T"])
    return dict(c, T=T, T1=T + 1, N=len(b2e), hidden=c["hidden"][rows], aff=c["aff"][rows], mask=mask,
                tp2id=np.concatenate(tp).astype(np.int32), b2e=np.array(b2e, np.int32))


# Experts of 2 to 2188 rows.  A row's bits do not depend on the rows that share its chunk, so the layer equals that of 100
# (bf16: 500) tokens at a time, whose chunks are of other classes (MX: most run the loop of up to 64 rows).  Against the
# oracle the 2-norm counts: an intermediate block whose maximum lies at a power of two may re-quantise with twice the step,
# which moved one row of 3000 by 4 % of its norm, 2.3 % of the largest value, and the 2-norm of the layer stayed at 0.0015;
# 0.008 leaves room for thirty such rows (0.04 * sqrt(30 / 3000) = 0.004) over what roundings give.
def _ragged(c, layer, golden, per):
    o = layer(c)[:3000]
    for i in range(0, 3000, per):
        part = layer(_of_tokens(c, np.arange(i, i + per)))[:per]
        assert np.array_equal(part.view(np.uint32), o[i:i + per].view(np.uint32)), i
    g = golden(c)[:3000]
    assert np.linalg.norm(o - g) <= 8e-3 * np.linalg.norm(g)


@pytest.mark.parametrize("fmt,alpha", [("e4m3", 0.3), ("e2m1", 0.3), ("e5m2", 1.0)])
def test_wide_mx_ragged_experts(fmt, alpha):
    c = mx_case(3000, 1024, 512, 8, 2, 128, seed=45, bias=True, weight_format=fmt, random_codes=True, alpha=alpha)
    _ragged(c, lambda c: from_bf16_tensor(_run_mx_options(c, 3, REF_MX_CLAMPS, False))[0],
            lambda c: _golden_mx_options(c, 3, REF_MX_CLAMPS), 100)


@pytest.mark.parametrize("alpha,fp8w", [(0.3, False), (1.0, True)])
def test_wide_bf16_ragged_experts(alpha, fp8w):
    c = dense_case(3000, 512, 320, 8, 2, 128, seed=46, bias=True, quant=fp8w, hidden_std=1.0, alpha=alpha)
    _ragged(c, lambda c: from_bf16_tensor(_run_dense(c, impl="shard_on_i", fp8_weights=fp8w)),
            lambda c: _golden_dense(c, fp8_weights=fp8w), 500)


@pytest.mark.parametrize("T,I,E,k,mode,skip", [(300, 512, 4, 2, 1, False), (700, 448, 3, 2, 2, False), (300, 512, 4, 2, 0, True),
                                               (100, 640, 2, 1, 2, True)])
def test_fp8_row_records_on_aligned_copies(T, I, E, k, mode, skip):
    """split_rows (csrc/capi.hip) counts the rows that a table of so many blocks is made for: with blocks of padding behind
    its own a small layer runs on copies of the records' codes and scales.  The same bits as on the records."""
    import torch
    from nkilib.core.moe.moe_cte import QuantizationConfig, SkipMode, moe_cte
    from nkilib.core.rmsnorm import RmsNormQuantKernelArgs, rmsnorm_quant_kernel
    from nkilib.core.utils.common_types import ExpertAffinityScaleMode
    from helpers import bf16_tensor, f32_tensor, i32_tensor, u8_tensor
    from test_gpu_moe import _spec

    dev = torch.device("cuda:0")
    H, B = 512, 128
    c = dense_case(T, H, I, E, k, B, seed=47, quant=True, bias=True, hidden_std=1.0, skip_token=skip)
    rec = rmsnorm_quant_kernel(bf16_tensor(c["hidden"], dev), bf16_tensor(np.ones((1, H), np.float32), dev),
                               RmsNormQuantKernelArgs())
    weights = (u8_tensor(c["gate_up_q"], dev).view(torch.float8_e4m3fn), u8_tensor(c["down_q"], dev).view(torch.float8_e4m3fn))
    scales = QuantizationConfig(f32_tensor(c["gate_up_scale"], dev), f32_tensor(c["down_scale"], dev))
    kw = dict(gate_and_up_proj_bias=bf16_tensor(c["gate_up_bias"], dev), down_proj_bias=bf16_tensor(c["down_bias"], dev),
              expert_affinities_scaling_mode=ExpertAffinityScaleMode(mode), skip_dma=SkipMode(skip, False))
    aff, outs = bf16_tensor(c["aff"].reshape(-1, 1), dev), []
    more = 2 ** 36 // (B * H * I) + 1  # (rows * H * I >= 2^36)
    for extra in (0, more):
        tp = np.concatenate([np.asarray(c["tp2id"]).reshape(-1), np.full(extra * B, -1 if skip else T)])
        b2e = np.concatenate([np.asarray(c["b2e"]).reshape(-1), np.full(extra, E - 1)])
        outs.append(moe_cte(rec, aff, *weights, i32_tensor(tp, dev), i32_tensor(b2e, dev), B, _spec("shard_on_block"),
                            quantization_config=scales, **kw))
    torch.cuda.synchronize()
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))
    raw = rec.view(torch.uint8).cpu().numpy()
    g = omoe.moe_blockwise_fp8_row_ref(raw[:, :H], raw[:, H:].copy().view(np.float32).reshape(-1), c["aff"], c["gate_up_q"],
                                       c["down_q"], c["gate_up_scale"], c["down_scale"], c["tp2id"], c["b2e"], B,
                                       gate_up_proj_bias=c["gate_up_bias"], down_proj_bias=c["down_bias"],
                                       skip_token=skip, expert_affinities_scaling_mode=mode)
    _check(from_bf16_tensor(outs[1])[:T, 0], g[:T], f"fp8 row, aligned copies, T={T} I={I} mode={mode}")
