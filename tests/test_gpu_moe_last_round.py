"""GPU parity of the large-tile kernels where a launch's last round of tiles is cut into pieces by rows, in halves and in quarters, at
the edges of the row-tile counts: 128 / 129 rows (not cut / cut), pieces that the last one does not need, 256 / 257, 288 / 289
and 320 rows, with activation checkpoints, and two rounds in turns.  A launch's size follows from the number of blocks its table
has, so the same layer with and without empty blocks behind its own is cut or not: both give the same bits.  (Which launch is
cut how: large_tile_queues.py.)  Tolerances are those of test_gpu_moe.py."""

import numpy as np
import pytest

import large_tile_queues as lq
from helpers import dense_case, from_bf16_tensor, mx_case
from oracle import moe as omoe
from test_gpu_moe import (REF_MX_CLAMPS, _check, _golden_dense, _golden_mx_options, _run_checkpointed, _run_dense, _run_fp8_row,
                          _run_mx_options)

pytestmark = pytest.mark.gpu

B = 128
ROWS = [128, 129, 193, 225, 256, 257, 289, 320, 321]
# H, I, the blocks of the table that is cut, how: three and two column tiles (gate/up and down) on 32 workgroups, or ten
SIZES = [(512, 384, 64, 2), (2560, 1280, 16, 1)]


def with_blocks(c, blocks):
    """The case with this many blocks: no empty ones behind its own, or more of them."""
    c = dict(c)
    real = ((c["tp2id"] >= 0) & (c["tp2id"] < c["T"])).reshape(-1, B).any(axis=1)
    own = int(np.flatnonzero(real)[-1]) + 1
    c["N"] = own if blocks is None else blocks
    c["tp2id"] = np.concatenate([c["tp2id"].reshape(-1)[: own * B], np.full((c["N"] - own) * B, c["T"], np.int32)]).astype(np.int32)
    c["b2e"] = np.concatenate([c["b2e"].reshape(-1)[:own], np.full(c["N"] - own, c["E"] - 1)]).astype(np.int32)
    return c


def check_cuts(T, size, ckpt=False):
    """One expert of T rows: the table without further blocks is not cut, the one with them is, unless the tiles have no more
    than 128 rows."""
    H, I, blocks, shift = size
    tp2id, own = np.concatenate([np.arange(T), np.full(-T % B, T)]).astype(np.int32), -(-T // B)
    for n in (own, blocks):
        queues = lq.queues_of(lq.chunks_of(np.concatenate([tp2id, np.full((n - own) * B, T, np.int32)]), np.zeros(n, np.int32), B, 1, T, ckpt), ckpt)
        for gx in (I // 128, H // 256):
            cuts = lq.launch_cuts(queues, gx, n)
            tall = any(c[1] > 128 for q in queues[1] for _, c in q)
            assert cuts == {0} if n == own or not tall else shift in cuts, (T, size, n, gx, cuts)
    return blocks


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("T", ROWS)
@pytest.mark.parametrize("fmt", ["e4m3", "e5m2", "e2m1"])
def test_pieces_mx(T, fmt, size):
    blocks = check_cuts(T, size)
    c = mx_case(T, *size[:2], 1, 1, B, seed=61, bias=True, weight_format=fmt, random_codes=True)
    cut = _run_mx_options(with_blocks(c, blocks), 3, REF_MX_CLAMPS, False)
    _check(from_bf16_tensor(cut)[0, :T], _golden_mx_options(c, 3, REF_MX_CLAMPS)[:T], f"pieces mx {fmt} T={T}")
    whole = _run_mx_options(with_blocks(c, None), 3, REF_MX_CLAMPS, False)
    assert np.array_equal(from_bf16_tensor(cut)[0, :T], from_bf16_tensor(whole)[0, :T])


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("T", ROWS)
def test_pieces_dense(T, size):
    blocks = check_cuts(T, size)
    H, I = size[:2]
    c = dense_case(T, H, I, 1, 1, B, seed=62, bias=True, hidden_std=1.0)
    rows = lambda t: from_bf16_tensor(t).reshape(T + 1, -1, H)[:T, 0]  # (with or without the second plane)
    cut = rows(_run_dense(with_blocks(c, blocks), act=0, mode=1))
    _check(cut, _golden_dense(c, act=0, mode=1)[:T], f"pieces bf16 T={T}")
    assert np.array_equal(cut, rows(_run_dense(with_blocks(c, None), act=0, mode=1)))


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("T", [129, 225, 256, 289, 320])
def test_pieces_checkpoints(T, size):
    """(one padding row more than T)"""
    blocks = check_cuts(T, size, True)
    H, I = size[:2]
    c = dense_case(T, H, I, 1, 1, B, seed=65, bias=True, hidden_std=1.0)
    outs = {}
    for n in (None, blocks):
        cn = with_blocks(c, n)
        outs[n] = [from_bf16_tensor(o) for o in _run_checkpointed(cn, "shard_on_i", act=3, mode=1)]
    own = with_blocks(c, None)
    golden = omoe.moe_blockwise_ref(c["hidden"], c["aff"], c["gate_up_w"], c["down_w"], own["tp2id"], own["b2e"], B,
                                    gate_up_proj_bias=c["gate_up_bias"], down_proj_bias=c["down_bias"], activation_function=3,
                                    skip_token=False, expert_affinities_scaling_mode=1, checkpoint_activation=True)
    for i, (name, g) in enumerate(zip(("output", "gate_up_activations_T", "down_activations"), golden)):
        n = T if i == 0 else own["N"]
        _check(outs[blocks][i][:n], g[:n], f"pieces checkpoint {name} T={T}")
        assert np.array_equal(outs[blocks][i][:n], outs[None][i][:n])


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("T", [129, 225, 257, 320])
def test_pieces_fp8_row(T, size):
    blocks = check_cuts(T, size)
    H, I = size[:2]
    c = dense_case(T, H, I, 1, 1, B, seed=63, quant=True, bias=True, hidden_std=1.0)
    import torch

    rec, out = _run_fp8_row(with_blocks(c, blocks), np.ones((1, H), np.float32), act=3, clamps={})
    raw = rec.view(torch.uint8).cpu().numpy()
    g = omoe.moe_blockwise_fp8_row_ref(raw[:, :H], raw[:, H:].copy().view(np.float32).reshape(-1), c["aff"],
                                       c["gate_up_q"], c["down_q"], c["gate_up_scale"], c["down_scale"], c["tp2id"],
                                       c["b2e"], c["B"], gate_up_proj_bias=c["gate_up_bias"],
                                       down_proj_bias=c["down_bias"], activation_function=3)
    rows = lambda t: from_bf16_tensor(t).reshape(T + 1, -1, H)[:T, 0]
    _check(rows(out), g[:T], f"pieces fp8 row T={T}")
    _, whole = _run_fp8_row(with_blocks(c, None), np.ones((1, H), np.float32), act=3, clamps={})
    assert np.array_equal(rows(out), rows(whole))


def test_rounds_in_turns():
    """16 experts of about 200 rows over 18 column tiles: 36 items on every XCD, a full round of 32 and 4 that are cut in quarters."""
    c = mx_case(1600, 512, 2304, 16, 2, 128, seed=64)
    queues = lq.queues_of(lq.chunks_of(c["tp2id"], c["b2e"], B, 16, 1600))
    assert all(lq.cut_of(q, queues[0], 18, 32) == (32, 2) for q in queues[1])
    o = from_bf16_tensor(_run_mx_options(c, 0, None, False))
    _check(o[0, :1600], _golden_mx_options(c, 0, None)[:1600], "two rounds mx")
    again = from_bf16_tensor(_run_mx_options(c, 0, None, False))
    assert np.array_equal(o, again)
