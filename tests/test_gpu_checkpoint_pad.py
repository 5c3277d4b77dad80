"""Activation checkpoints (csrc/combine.hip: ckpt_tail_kernel, and ckpt_pad_kernel for a layer issued stage by stage): the
rows of tokens, those behind an expert's last token and the blocks that do not run, every row against the oracle's; the same
bits whether the tables are the block build's own or copies of them, and from one call and from a call per stage; calls with
checkpoints follow tables that change.  Tolerances are those of test_gpu_moe.py."""

import numpy as np
import pytest

from helpers import bf16_tensor, dense_case, from_bf16_tensor, i32_tensor
from oracle import blocks as ob
from oracle import moe as omoe
from test_gpu_moe import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,I,E,k,B,skip,cond", [
    (300, 512, 256, 4, 2, 512, False, False),  # one block per expert, more rows of padding than of tokens; blocks past the experts
    (300, 512, 256, 4, 2, 512, False, True),   # the same with conditions: the blocks past the experts stay zero
    (40, 512, 128, 8, 2, 64, True, False),     # short blocks, pieces of eight rows with rows to keep
    (100, 256, 64, 4, 1, 33, False, True),     # odd blocks: element by element; I shorter than a column tile
    (300, 256, 160, 2, 1, 33, False, True),    # odd blocks in chunks of 150 rows, which go through five blocks each
    (600, 256, 128, 2, 1, 131, False, False),  # ... of 300 rows
    (700, 256, 128, 2, 1, 131, True, False),   # ... and a second chunk that begins within a block
    (700, 256, 128, 2, 1, 130, False, False),  # the same with even blocks, two rows to a store
    (256, 256, 96, 2, 1, 128, False, False),   # full blocks: the last run's only padding is whole blocks
    (9, 256, 128, 16, 1, 128, True, False),    # experts without a token
])
def test_checkpoint_padding(T, H, I, E, k, B, skip, cond, monkeypatch):
    import torch
    from nkilib.core.moe.moe_cte import SkipMode, _launch, build_token_blocks
    from nkilib.core.moe.moe_cte.bwmm_shard_on_block import run_dense_variant

    dev = torch.device("cuda:0")
    c = dense_case(T, H, I, E, k, B, seed=41, skip_token=skip, bias=True, hidden_std=1.0)
    ids = i32_tensor(ob.router_with_controlled_distribution(T, k, E).astype(np.int32), dev)
    args = (bf16_tensor(c["hidden"], dev), bf16_tensor(c["aff"].reshape(-1, 1), dev), bf16_tensor(c["gate_up_w"], dev),
            bf16_tensor(c["down_w"], dev))
    outs, stages = [], []
    for planned, by_stage in ((False, False), (True, False), (True, True)):
        tp, b2e, co = build_token_blocks(ids, E, B, c["N"], skip_token=skip)
        assert np.array_equal(tp.cpu().numpy(), c["tp2id"])
        if not planned:  # (copies: not the tables that the plan belongs to)
            tp, b2e, co = tp.clone(), b2e.clone(), co.clone()
        junk = [torch.full((c["N"] * B * max(2 * I, H),), float("nan"), dtype=torch.bfloat16, device=dev) for _ in range(2)]
        del junk  # the checkpoints are allocated over it
        monkeypatch.setattr(_launch, "stage_callback", stages.append if by_stage else None)
        outs.append(run_dense_variant(*args, B, tp, b2e, "TH", conditions=co if cond else None,
                                      gate_and_up_proj_bias=bf16_tensor(c["gate_up_bias"], dev),
                                      down_proj_bias=bf16_tensor(c["down_bias"], dev), skip_dma=SkipMode(skip, False),
                                      checkpoint_gate_up=True, checkpoint_down=True))
    torch.cuda.synchronize()
    assert stages == ["prep", "gate_up", "down", "combine"]
    g_out, g_gu, g_d = omoe.moe_blockwise_ref(
        c["hidden"], c["aff"], c["gate_up_w"], c["down_w"], c["tp2id"], c["b2e"], B,
        conditions=c["cond"] if cond else None, gate_up_proj_bias=c["gate_up_bias"], down_proj_bias=c["down_bias"],
        activation_function=0, skip_token=skip, expert_affinities_scaling_mode=1, checkpoint_activation=True)
    for out, gu, d in outs:
        _check(from_bf16_tensor(out)[:T], g_out[:T], "output")
        _check(from_bf16_tensor(gu), g_gu, "gate_up_activations_T")
        _check(from_bf16_tensor(d), g_d, "down_activations")
    for x, y, z in zip(*outs):
        assert torch.equal(x.view(torch.int16), y.view(torch.int16)) and torch.equal(x.view(torch.int16), z.view(torch.int16))


def test_checkpoints_follow_the_tables():
    """Tables of the block build that are overwritten past torch's version counter, or between the replays of a recorded
    graph: nothing that was derived from what they held before counts."""
    import torch
    from nkilib.core.moe.moe_cte import SkipMode, build_token_blocks
    from nkilib.core.moe.moe_cte.bwmm_shard_on_block import run_dense_variant

    dev = torch.device("cuda:0")
    T, H, I, E, k, B = 300, 512, 256, 4, 2, 128
    c = dense_case(T, H, I, E, k, B, seed=42, hidden_std=1.0)
    aff = torch.rand((T + 1, E), device=dev).to(torch.bfloat16).reshape(-1, 1)
    args = (bf16_tensor(c["hidden"], dev), aff, bf16_tensor(c["gate_up_w"], dev), bf16_tensor(c["down_w"], dev))
    rng = np.random.default_rng(42)
    # three routings, of other experts' loads each: the first two, two of the first three, and any
    ids = [i32_tensor(np.stack([rng.permutation(m)[:k] for _ in range(T)]).astype(np.int32), dev) for m in (2, 3, 4)]

    def layer(tp, b2e):
        return run_dense_variant(*args, B, tp, b2e, "TH", skip_dma=SkipMode(False, False), checkpoint_gate_up=True,
                                 checkpoint_down=True)

    tables = [[t.clone() for t in build_token_blocks(i, E, B, c["N"])[:2]] for i in ids]
    want = [layer(*t) for t in tables]
    assert not torch.equal(want[0][0], want[1][0]) and not torch.equal(want[1][0], want[2][0])
    tp, b2e, _ = build_token_blocks(ids[0], E, B, c["N"])

    def same(outs, n):
        return all(torch.equal(x.view(torch.int16), y.view(torch.int16)) for x, y in zip(outs, want[n]))

    assert same(layer(tp, b2e), 0)
    tp.data.copy_(tables[1][0])
    b2e.data.copy_(tables[1][1])
    assert same(layer(tp, b2e), 1)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = layer(tp, b2e)
    for n in (1, 2, 0):
        tp.copy_(tables[n][0])
        b2e.copy_(tables[n][1])
        layer(*tables[0])  # (eager work between the replays)
        graph.replay()
        torch.cuda.synchronize()
        assert same(outs, n), n


@pytest.mark.parametrize("N,B,first", [
    (1, 131200, 0),     # a block of the gate_up checkpoint of more than 4 GiB, two rows to a store
    (1, 131201, 0),     # the same, row by row
    (2, 65600, 65500),  # blocks of 2 GiB, a chunk that goes on into the second one
])
def test_gate_up_checkpoint_past_4_gib(N, B, first):
    """One expert, 200 tokens from slot `first` on, every other slot padding: each token's column equals that of the same
    tokens in a block of 256 rows (which the tests above compare with the oracle), each other slot's the padding row's."""
    import torch
    from nkilib.core.moe.moe_cte import SkipMode
    from nkilib.core.moe.moe_cte.bwmm_shard_on_block import run_dense_variant

    dev = torch.device("cuda:0")
    T, H, I = 200, 256, 8192
    g = torch.Generator(device=dev)
    g.manual_seed(43)

    def bf16(*shape, std=0.1):
        return (torch.randn(shape, generator=g, device=dev) * std).to(torch.bfloat16)

    x = bf16(T + 1, H, std=1.0)
    x[T] = 0
    aff = torch.ones((T + 1, 1), dtype=torch.bfloat16, device=dev)
    gu, dw, gu_b, d_b = bf16(1, H, 2, I), bf16(1, I, H), bf16(1, 2, I, std=0.5), bf16(1, H)

    def layer(n, b, at):
        tp = torch.full((n * b,), T, dtype=torch.int32, device=dev)
        tp[at:at + T] = torch.arange(T, dtype=torch.int32, device=dev)
        return run_dense_variant(x, aff, gu, dw, b, tp, torch.zeros(n, dtype=torch.int32, device=dev), "TH",
                                 gate_and_up_proj_bias=gu_b, down_proj_bias=d_b, skip_dma=SkipMode(False, False),
                                 checkpoint_gate_up=True)

    out0, want = layer(1, 256, 0)
    out, ck = layer(N, B, first)
    assert torch.equal(out.view(torch.int16), out0.view(torch.int16))
    want = want[0].view(torch.int16)                                             # [2, I, 256]
    for n in range(N):
        lo, hi = max(first - n * B, 0), min(first + T - n * B, B)                # the block's rows with tokens
        for gu_ in range(2):
            rows, w = ck[n, gu_].view(torch.int16), want[gu_]
            t0 = n * B + lo - first
            assert torch.equal(rows[:, lo:hi], w[:, t0:t0 + hi - lo]), (n, gu_, "tokens")
            assert bool((rows[:, :lo] == w[:, T:T + 1]).all()) and bool((rows[:, hi:] == w[:, T:T + 1]).all()), (n, gu_, "padding")


@pytest.mark.parametrize("N,B,I", [
    (1 << 18, 2, 2048),  # 2^24 pieces of 64 columns
    (1 << 23, 1, 8),     # so many blocks that the copies of the two checkpoints need a launch each
])
def test_checkpoints_of_very_many_blocks(N, B, I):
    """The first blocks hold 200 tokens, the others do not run: the same values as in one block of 256 rows, and zeros."""
    import torch
    from nkilib.core.moe.moe_cte import SkipMode
    from nkilib.core.moe.moe_cte.bwmm_shard_on_block import run_dense_variant

    dev = torch.device("cuda:0")
    T, H = 200, 256
    g = torch.Generator(device=dev)
    g.manual_seed(44)
    x, gu, dw = [(torch.randn(s, generator=g, device=dev) * 0.1).to(torch.bfloat16) for s in ((T + 1, H), (1, H, 2, I), (1, I, H))]
    x[T] = 0
    aff = torch.ones((T + 1, 1), dtype=torch.bfloat16, device=dev)

    def layer(n, b, active):
        tp = torch.full((n * b,), T, dtype=torch.int32, device=dev)
        tp[:T] = torch.arange(T, dtype=torch.int32, device=dev)
        cond = (torch.arange(n + 1, device=dev) < active).to(torch.int32)
        return run_dense_variant(x, aff, gu, dw, b, tp, torch.zeros(n, dtype=torch.int32, device=dev), "TH", conditions=cond,
                                 skip_dma=SkipMode(False, False), checkpoint_gate_up=True, checkpoint_down=True)

    out0, gu0, d0 = layer(1, 256, 1)
    out, gu1, d1 = layer(N, B, T // B)
    na = T // B
    assert torch.equal(out.view(torch.int16), out0.view(torch.int16))
    assert torch.equal(gu1[:na].permute(1, 2, 0, 3).reshape(2, I, T).view(torch.int16), gu0[0, :, :, :T].contiguous().view(torch.int16))
    assert torch.equal(d1[:na].reshape(T, H).view(torch.int16), d0[0, :T].view(torch.int16))
    assert not bool(gu1[na:].any()) and not bool(d1[na:].any())
