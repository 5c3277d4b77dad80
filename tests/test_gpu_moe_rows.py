"""GPU parity of the few-rows expert kernel (csrc/bwmm_rows.hip) against the oracle at the edges of its instances: one,
two and four row tiles (16 / 17, 32 / 33, 64 / 65 tokens), passes over more rows than an instance multiplies, K loops
shorter than the waves that split them, short last intermediate tiles, both column groupings (few and many 64-column
groups), every weight format and the options of the epilogues.  Tolerances are those of test_gpu_moe.py."""

import numpy as np
import pytest

from helpers import dense_case, from_bf16_tensor, mx_case
from oracle import moe as omoe
from test_gpu_moe import (REF_MX_CLAMPS, _check, _golden_dense, _golden_mx_options, _run_dense, _run_fp8_row,
                          _run_mx_options)

pytestmark = pytest.mark.gpu

CL = dict(gate_clamp_upper_limit=0.8, gate_clamp_lower_limit=-0.7, up_clamp_upper_limit=0.9, up_clamp_lower_limit=-0.5)


@pytest.mark.parametrize("T,H,I,E,k,act,mode,bias,skip,fp8w", [
    (1, 256, 128, 4, 2, 0, 1, False, False, False),     # four K slices for four waves; one slice each in the down stage
    (16, 512, 384, 8, 2, 0, 1, True, True, False),      # one full row tile; a short last intermediate tile (768 bytes of K)
    (17, 512, 128, 4, 4, 3, 2, True, False, False),     # two row tiles; Swish, PRE_SCALE; two K slices for four waves
    (33, 2560, 1152, 16, 4, 0, 1, False, False, True),  # four row tiles; 128-column workgroups in both stages; fp8 weights
    (40, 512, 1152, 16, 4, 0, 1, True, True, False),    # the same from a short K, bf16 weights
    (64, 512, 256, 3, 2, 1, 0, True, True, False),      # GELU, NO_SCALE
    (65, 512, 128, 8, 2, 0, 1, False, False, False),    # more tokens than a pass has rows
    (256, 512, 256, 8, 2, 2, 1, True, False, False),    # experts of more than 64 rows: a second pass
])
def test_rows_dense(T, H, I, E, k, act, mode, bias, skip, fp8w):
    c = dense_case(T, H, I, E, k, 128, seed=31, skip_token=skip, bias=bias, quant=fp8w, hidden_std=1.0)
    o = from_bf16_tensor(_run_dense(c, act=act, mode=mode, clamps=CL, fp8_weights=fp8w))[:, 0]
    g = _golden_dense(c, act=act, mode=mode, clamps=CL, fp8_weights=fp8w)
    _check(o[:T], g[:T], f"few rows bf16 T={T} H={H} I={I}")


@pytest.mark.parametrize("T,H,I,E,k,mode", [(5, 512, 512, 4, 2, 2), (24, 2560, 1152, 16, 2, 1), (50, 512, 640, 2, 2, 1)])
def test_rows_fp8_row(T, H, I, E, k, mode):
    c = dense_case(T, H, I, E, k, 128, seed=32, quant=True, bias=True, hidden_std=1.0)
    rec, out = _run_fp8_row(c, np.ones((1, H), np.float32), mode=mode, clamps=CL, act=3)
    import torch

    raw = rec.view(torch.uint8).cpu().numpy()
    g = omoe.moe_blockwise_fp8_row_ref(raw[:, :H], raw[:, H:].copy().view(np.float32).reshape(-1), c["aff"], c["gate_up_q"],
                                       c["down_q"], c["gate_up_scale"], c["down_scale"], c["tp2id"], c["b2e"], c["B"],
                                       gate_up_proj_bias=c["gate_up_bias"], down_proj_bias=c["down_bias"],
                                       activation_function=3, expert_affinities_scaling_mode=mode, **CL)
    _check(from_bf16_tensor(out)[:T, 0], g[:T], f"few rows fp8 row T={T}")


@pytest.mark.parametrize("T,H,I,E,k,fmt,skip", [
    (1, 512, 128, 8, 4, "e4m3", False),
    (16, 1024, 640, 4, 2, "e4m3", True),     # a short last intermediate tile
    (17, 512, 512, 2, 2, "e4m3", False),
    (32, 2560, 1152, 16, 4, "e5m2", False),  # 128-column workgroups in the down stage
    (8, 512, 384, 4, 2, "e2m1", True),       # 4-bit weights: both stages
    (60, 1024, 512, 2, 2, "e2m1", False),    # ... the down stage alone, four row tiles
])
@pytest.mark.parametrize("copies", [True, False])
def test_rows_mx(T, H, I, E, k, fmt, skip, copies):
    """With the weights' copies in read order and from the reference layout in place."""
    from nkilib.core.moe.moe_cte import _launch

    c = mx_case(T, H, I, E, k, 128, seed=33, skip_token=skip, bias=True, weight_format=fmt, random_codes=True)
    was = _launch.mx_weight_copies
    try:
        _launch.mx_weight_copies = copies
        o = from_bf16_tensor(_run_mx_options(c, 3, REF_MX_CLAMPS, False))
    finally:
        _launch.mx_weight_copies = was
    _check(o[0, :T], _golden_mx_options(c, 3, REF_MX_CLAMPS)[:T], f"few rows mx {fmt} T={T} H={H} I={I} copies={copies}")


@pytest.mark.parametrize("kind,T", [("bf16", 20), ("bf16", 200), ("mx", 1), ("mx", 150)])
def test_clock_probe_is_filled(kind, T):
    """The gate/up and the down GEMM each store their workgroup 0's cycles and 100 MHz ticks, whichever kernel they are."""
    import torch
    from nkilib.core.moe.moe_cte import _launch

    probe = torch.full((4,), -1, dtype=torch.int64, device="cuda:0")
    _launch.gemm_clock_probe = probe
    try:
        if kind == "mx":
            _run_mx_options(mx_case(T, 512, 512, 4, 2, 128, seed=38, bias=True, random_codes=True), 3, REF_MX_CLAMPS, False)
        else:
            _run_dense(dense_case(T, 512, 256, 4, 2, 128, seed=38, hidden_std=1.0))
        torch.cuda.synchronize()
    finally:
        _launch.gemm_clock_probe = None
    cycles, ticks = probe[0::2].tolist(), probe[1::2].tolist()
    assert all(t > 0 for t in ticks) and all(c > 0 for c in cycles), probe.tolist()


def test_mx_copies_follow_the_block_scales():
    """A scale changed in place, or another scale tensor with the same weights, must reach the result."""
    import torch
    from nkilib import synthetic as syn
    from nkilib.core.moe.moe_cte import _launch
    from nkilib.core.moe.moe_tkg import moe_tkg
    from nkilib.core.utils.common_types import ExpertAffinityScaleMode

    dev = torch.device("cuda:0")
    T, H, I, E, k = 4, 512, 256, 4, 2
    gu, gs, d, ds = syn.mx_expert_weights(E, H, I, 0.05, dev, seed=5)
    ids, aff = syn.route(T, E, k, dev, seed=5)
    x = syn.hidden_states(T, H, dev, seed=5)[:T].contiguous()

    def layer(scale):
        return moe_tkg(x, gu, d, aff[:T].contiguous(), ids, False, expert_gate_up_weights_scale=scale,
                       expert_down_weights_scale=ds, expert_affinities_scaling_mode=ExpertAffinityScaleMode.POST_SCALE)

    def plain(scale):
        _launch.mx_weight_copies = False
        try:
            return layer(scale)
        finally:
            _launch.mx_weight_copies = True

    assert torch.equal(layer(gs), plain(gs))
    other = gs + 1
    assert torch.equal(layer(other), plain(other)) and not torch.equal(layer(other), layer(gs))
    gs.add_(1)
    assert torch.equal(layer(gs), layer(other))


@pytest.mark.parametrize("T", [4, 150])  # the few-rows and the large-tile kernels
@pytest.mark.parametrize("fp4", [False, True])
def test_mx_scales_are_read_by_every_call(T, fp4):
    """The kept copies hold weights alone: scales written past torch's version counter, scale tensors that did not exist
    when the copies were made, and scales updated between the replays of a recorded graph all reach the result, and none
    of them makes the copies anew."""
    import torch
    from nkilib import synthetic as syn
    from nkilib.core.moe.moe_cte import _launch
    from nkilib.core.moe.moe_tkg import moe_tkg
    from nkilib.core.utils.common_types import ExpertAffinityScaleMode

    dev = torch.device("cuda:0")
    H, I, E, k = 512, 256, 4, 2
    gu, gs, d, ds = syn.mx4_expert_weights(E, H, I, dev, seed=6) if fp4 else syn.mx_expert_weights(E, H, I, 0.05, dev, seed=6)
    ids, aff = syn.route(T, E, k, dev, seed=6)
    x = syn.hidden_states(T, H, dev, seed=6)[:T].contiguous()
    aff = aff[:T].contiguous()

    def layer(gs, ds):
        return moe_tkg(x, gu, d, aff, ids, False, expert_gate_up_weights_scale=gs, expert_down_weights_scale=ds,
                       expert_affinities_scaling_mode=ExpertAffinityScaleMode.POST_SCALE)

    def plain(gs, ds):
        _launch.mx_weight_copies = False
        try:
            return layer(gs, ds)
        finally:
            _launch.mx_weight_copies = True

    _launch.clear_kmajor_weight_cache()
    gs0, ds0 = torch.zeros_like(gs), torch.zeros_like(ds)
    layer(gs0, ds0)  # (the copies are made here, before the scales are there)
    (copies,) = _launch._kmajor.values()
    first = layer(gs, ds)
    assert first.abs().sum() > 0 and torch.equal(first, plain(gs, ds))
    gs.data.add_(1)
    ds.data.sub_(1)
    assert torch.equal(layer(gs, ds), plain(gs, ds)) and not torch.equal(layer(gs, ds), first)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = layer(gs, ds)
    for step in range(3):
        if step:
            gs.add_(1)
            ds.add_(1)
        want = plain(gs, ds)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), step
    assert list(_launch._kmajor.values()) == [copies]


@pytest.mark.parametrize("T", [1, 20, 150])  # the few-rows and the large-tile kernels
@pytest.mark.parametrize("act", [0, 3])
def test_nan_rows_stay_nan_under_an_upper_gate_clamp(T, act):
    """The clamps of the models that clamp (gate from above, up from both sides): a token that is not a number must not
    come out as one, and no other token may be touched by it."""
    c = dense_case(T, 512, 256, 4, 2, 128, seed=36, bias=True, hidden_std=1.0)
    clamps = dict(gate_clamp_upper_limit=0.8, up_clamp_upper_limit=0.9, up_clamp_lower_limit=-0.5)
    want = from_bf16_tensor(_run_dense(c, act=act, mode=1, clamps=clamps))[:T, 0]
    c["hidden"][0] = np.nan
    o = from_bf16_tensor(_run_dense(c, act=act, mode=1, clamps=clamps))[:T, 0]
    assert np.isnan(o[0]).all()
    assert np.array_equal(o[1:], want[1:])


@pytest.mark.parametrize("T", [20, 150])  # the few-rows and the large-tile kernels
@pytest.mark.parametrize("I,fp8w", [(36, False), (130, False), (202, True), (264, False)])
def test_padded_intermediate_dense(T, I, fp8w):
    """Intermediate sizes that fill neither a column tile of 128 nor a K slice of 64 (and rows of weights that are not
    aligned to four elements): the padding columns must add nothing, biases and scales keep their columns."""
    c = dense_case(T, 512, I, 4, 2, 128, seed=34, bias=True, quant=fp8w, hidden_std=1.0)
    o = from_bf16_tensor(_run_dense(c, act=1, mode=1, clamps=CL, fp8_weights=fp8w))[:, 0]
    _check(o[:T], _golden_dense(c, act=1, mode=1, clamps=CL, fp8_weights=fp8w)[:T], f"padded bf16 T={T} I={I}")


@pytest.mark.parametrize("T", [20, 150])
@pytest.mark.parametrize("I", [36, 130, 203, 256])
def test_infinite_rows_with_a_padded_intermediate(T, I):
    """An infinity times weights that are all positive is an infinity in every output: the columns that pad the weights,
    zeros, must not make it something else (256 fills its tiles: no padding)."""
    c = dense_case(T, 512, I, 4, 2, 128, seed=37, hidden_std=1.0)
    c["gate_up_w"], c["down_w"] = np.abs(c["gate_up_w"]) + 2.0 ** -7, np.abs(c["down_w"]) + 2.0 ** -7
    want = from_bf16_tensor(_run_dense(c, act=0, mode=1))[:T, 0]
    c["hidden"][0] = np.abs(c["hidden"][0])
    c["hidden"][0, 5] = np.inf
    o = from_bf16_tensor(_run_dense(c, act=0, mode=1))[:T, 0]
    assert np.isposinf(o[0]).all()
    assert np.array_equal(o[1:], want[1:])


@pytest.mark.parametrize("T", [20, 150])
@pytest.mark.parametrize("I", [36, 264])
def test_padded_intermediate_fp8_row(T, I):
    c = dense_case(T, 512, I, 4, 2, 128, seed=35, quant=True, bias=True, hidden_std=1.0)
    rec, out = _run_fp8_row(c, np.ones((1, 512), np.float32), clamps=CL, act=3)
    import torch

    raw = rec.view(torch.uint8).cpu().numpy()
    g = omoe.moe_blockwise_fp8_row_ref(raw[:, :512], raw[:, 512:].copy().view(np.float32).reshape(-1), c["aff"],
                                       c["gate_up_q"], c["down_q"], c["gate_up_scale"], c["down_scale"], c["tp2id"],
                                       c["b2e"], c["B"], gate_up_proj_bias=c["gate_up_bias"], down_proj_bias=c["down_bias"],
                                       activation_function=3, **CL)
    _check(from_bf16_tensor(out)[:T, 0], g[:T], f"padded fp8 row T={T} I={I}")
