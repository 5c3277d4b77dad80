"""GPU parity of the MX kinds on the general tiled kernel, which takes the calls of a short last tile (I % 128 != 0) whose tensors
lie closer than the other kernels' loads are aligned to: 16 bytes for the weights and activations, 4 for scales, biases and
affinities.  Tolerances are those of test_gpu_moe.py."""

import numpy as np
import pytest

from helpers import bf16_tensor, from_bf16_tensor, i32_tensor, mx_case, u8_tensor
from test_gpu_moe import REF_MX_CLAMPS, _check, _golden_mx_options

pytestmark = pytest.mark.gpu


def _at(t, offset):
    """The same values, `offset` bytes behind an aligned address."""
    import torch

    n = t.numel() * t.element_size()
    room = torch.zeros(n + 256, dtype=torch.uint8, device=t.device)
    room[offset: offset + n].copy_(t.contiguous().view(torch.uint8).reshape(-1))
    out = room[offset: offset + n].view(t.dtype).view(t.shape)
    assert out.data_ptr() % 16 == offset % 16
    return out


@pytest.mark.parametrize("T,I,fmt,moved,offset", [
    (300, 96, "e4m3", "gate_up", 4),
    (300, 544, "e5m2", "gate_up", 8),
    (300, 608, "e2m1", "gate_up", 8),
    (20, 160, "e2m1", "down", 4),       # (few rows)
    (300, 1056, "e4m3", "down", 8),
    (300, 96, "e5m2", "down", 4),
    (300, 96, "e2m1", "codes", 4),      # MXFP8 codes and their scales (bf16 hidden states there are refused by the quantiser)
    (300, 544, "e4m3", "codes", 8),
    (300, 544, "e4m3", "gate_up_s", 1),
    (300, 96, "e4m3", "down_s", 2),
    (300, 544, "e2m1", "gate_up_bias", 2),
    (300, 96, "e5m2", "down_bias", 2),
    (20, 544, "e4m3", "aff", 2),
])
def test_tensors_off_their_alignment(T, I, fmt, moved, offset):
    import torch
    from nkilib.core.moe.moe_cte import _launch
    from nkilib.core.moe.moe_cte.bwmm_shard_on_block_mx import bwmm_shard_on_block_mx
    from nkilib.core.subkernels.rmsnorm_mx_quantize_tkg import rmsnorm_mx_quantize
    from nkilib.core.utils.common_types import ActFnType
    from oracle.numerics import pack_e2m1_x4

    H, E, k, B = 1024, 8, 2, 128
    dev = torch.device("cuda:0")
    c = mx_case(T, H, I, E, k, B, seed=71, bias=True, weight_format=fmt, random_codes=True)
    t = {n: u8_tensor(c[n], dev) for n in ("gate_up_s", "down_s")}
    t |= {n: bf16_tensor(c[n], dev) for n in ("gate_up_bias", "down_bias", "hidden")}
    t["aff"] = bf16_tensor(c["aff"].reshape(-1, 1), dev)
    for name, q in (("gate_up", "gate_up_q"), ("down", "down_q")):
        if fmt == "e2m1":
            t[name] = torch.from_numpy(pack_e2m1_x4(c[q]).view(np.int16)).to(dev)
        else:
            t[name] = u8_tensor(c[q], dev).view(torch.float8_e5m2 if fmt == "e5m2" else torch.float8_e4m3fn)
    t["xs"] = None
    if moved == "codes":
        t["hidden"], t["xs"] = rmsnorm_mx_quantize(t["hidden"], None, do_norm=False)

    def run():
        clocks = torch.zeros(4, dtype=torch.int64, device=dev)  # (the general kernel writes none)
        _launch.gemm_clock_probe = clocks
        try:
            out = bwmm_shard_on_block_mx[2](
                t["hidden"], t["aff"], t["gate_up"], t["down"], i32_tensor(c["tp2id"], dev), i32_tensor(c["b2e"], dev),
                gate_and_up_proj_bias=t["gate_up_bias"], down_proj_bias=t["down_bias"], gate_up_proj_scale=t["gate_up_s"],
                down_proj_scale=t["down_s"], block_size=B, activation_function=ActFnType.Swish, hidden_states_scale=t["xs"],
                **REF_MX_CLAMPS)
        finally:
            _launch.gemm_clock_probe = None
        return from_bf16_tensor(out)[0, :T], clocks.cpu().tolist()

    golden = _golden_mx_options(c, 3, REF_MX_CLAMPS)[:T]
    aligned, clocks = run()
    assert all(clocks)
    _check(aligned, golden, f"mx aligned {fmt} I={I}")
    for name in (("hidden", "xs") if moved == "codes" else (moved,)):
        t[name] = _at(t[name], offset)
    out, clocks = run()
    assert not any(clocks), "the general kernel takes this call"
    _check(out, golden, f"mx general kernel {fmt} I={I}, {moved} at {offset}")
