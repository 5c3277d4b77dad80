"""GPU parity of the MX kinds where the last intermediate tile holds no multiple of 32 partitions (I % 128 != 0): the last
column tile of the gate/up stage and the last K slice of the down stage are 8, 16 or 24 partitions of their 32, in the
few-rows kernel and both tile loops of the large-tile kernels.  Tolerances are those of test_gpu_moe.py."""

import numpy as np
import pytest

from helpers import from_bf16_tensor, mx_case
from test_gpu_moe import REF_MX_CLAMPS, _check, _golden_mx_options, _run_mx_options

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,I,E,k,fmt", [
    (1, 512, 32, 4, 2, "e4m3"),       # few rows; 8 partitions in all, one K slice
    (20, 512, 480, 4, 2, "e4m3"),     # two row tiles; a full slice grid but 8 partitions
    (7, 1024, 608, 4, 2, "e2m1"),     # 4-bit weights; 24 partitions behind a full intermediate tile
    (9, 512, 544, 4, 2, "e5m2"),      # 8, 16 and 24 of them, 8-bit weights
    (20, 512, 576, 4, 2, "e4m3"),
    (31, 1024, 608, 4, 2, "e4m3"),
    (40, 512, 192, 4, 1, "e4m3"),     # chunks of up to 64 rows: weights through registers
    (40, 512, 160, 3, 1, "e2m1"),     # (its down stage on the few-rows kernel)
    (100, 512, 544, 8, 2, "e4m3"),    # the same, behind a full intermediate tile
    (100, 512, 576, 8, 2, "e5m2"),
    (100, 1024, 608, 8, 2, "e4m3"),
    (100, 512, 160, 8, 2, "e2m1"),
    (100, 512, 544, 8, 2, "e2m1"),
    (100, 1024, 608, 8, 2, "e2m1"),
    (300, 1024, 96, 4, 2, "e4m3"),    # chunks past 64 rows: both operands through LDS
    (600, 512, 1120, 2, 1, "e4m3"),   # ... of more than 256 rows
    (500, 512, 544, 2, 1, "e2m1"),
    (300, 512, 832, 4, 2, "e5m2"),
])
def test_short_tiles(T, H, I, E, k, fmt):
    # (Another seed for the smallest: with 32 intermediate values in all, one that an exponential's last bit moves across the
    # tie between two e4m3 codes changes by 1/16, and a row of outputs by up to that share of its largest term.  Seed 51 has
    # such a value, 3.2e-2 off against the oracle in this kernel and in the general kernel alike.)
    c = mx_case(T, H, I, E, k, 128, seed=61 if I == 32 else 51, bias=True, weight_format=fmt, random_codes=True)
    rows = c["mask"].sum(axis=0)
    assert T != 100 or (rows.max() <= 64 and rows.min() > 0)
    want = _golden_mx_options(c, 3, REF_MX_CLAMPS)[:T]
    o = from_bf16_tensor(_run_mx_options(c, 3, REF_MX_CLAMPS, False))
    _check(o[0, :T], want, f"mx short tiles {fmt} T={T} I={I}")
    if I > 512:
        # what stands in the down weights past the last partition is nothing's input: the bits do not change with it
        worst = 0x7 if fmt == "e2m1" else 0x7f  # the largest 4-bit value; not a number in both 8-bit formats
        c["down_q"][:, I % 512 // 4:, I // 512] = worst
        c["down_s"][:, I % 512 // 32:, I // 512] = 255  # no number either
        assert np.array_equal(from_bf16_tensor(_run_mx_options(c, 3, REF_MX_CLAMPS, False)), o)


@pytest.mark.parametrize("T", [20, 300])  # the few-rows and the large-tile kernels
def test_infinite_rows_with_a_short_tile(T):
    """A row whose activations overflow reaches the columns that the last tile does not have as well: its own outputs may be
    anything, every other row keeps its bits."""
    c = mx_case(T, 512, 96, 4, 2, 128, seed=52, weight_format="e4m3")
    want = from_bf16_tensor(_run_mx_options(c, 0, None, False))
    c["hidden"][0] = 3e38
    o = from_bf16_tensor(_run_mx_options(c, 0, None, False))
    assert np.array_equal(o[0, 1:T], want[0, 1:T])


@pytest.mark.parametrize("fmt", ["e4m3", "e2m1"])
@pytest.mark.parametrize("T", [20, 300])  # the few-rows and the large-tile kernels
def test_weights_are_read_as_they_are(T, fmt):
    """A weight loader writes through ``param.data``, which torch's version counter does not see.  Where I is no multiple of
    128 the MX kinds keep nothing of the weights: the next call multiplies with what stands there now, and a call that is
    recorded as the first with its weights leaves nothing behind."""
    import torch
    from nkilib.core.moe.moe_cte import _launch
    from nkilib.core.moe.moe_cte.bwmm_shard_on_block_mx import bwmm_shard_on_block_mx
    from helpers import bf16_tensor, i32_tensor, u8_tensor
    from oracle.numerics import pack_e2m1_x4

    dev = torch.device("cuda:0")
    c, d = (mx_case(T, 512, 96, 4, 2, 128, seed=s, weight_format=fmt, random_codes=True) for s in (53, 54))

    def weights(case):
        if fmt == "e2m1":
            return [torch.from_numpy(pack_e2m1_x4(case[w]).view(np.int16)).to(dev) for w in ("gate_up_q", "down_q")]
        return [u8_tensor(case[w], dev).view(torch.float8_e4m3fn) for w in ("gate_up_q", "down_q")]

    args = [bf16_tensor(c["hidden"], dev), bf16_tensor(c["aff"].reshape(-1, 1), dev)]
    tables = [i32_tensor(c["tp2id"], dev), i32_tensor(c["b2e"], dev)]
    kw = dict(gate_up_proj_scale=u8_tensor(c["gate_up_s"], dev), down_proj_scale=u8_tensor(c["down_s"], dev), block_size=128)
    run = lambda w: bwmm_shard_on_block_mx[2](*args, *w, *tables, **kw)
    kept = len(_launch._kmajor)
    w, other = weights(c), weights(d)
    first, second = run(w), run(other)
    assert not torch.equal(first, second)
    for t, o in zip(w, other):
        raw = torch.uint8 if t.element_size() == 1 else torch.int16
        t.data.view(raw).copy_(o.view(raw))
    assert torch.equal(run(w), second)
    assert len(_launch._kmajor) == kept
