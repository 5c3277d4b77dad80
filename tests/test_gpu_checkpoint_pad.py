"""Activation checkpoints behind an expert's last token and in blocks that do not run (ckpt_pad_*_kernel): every row against
the oracle's without a plan, and the same bits with the block build's plan.  Tolerances are those of test_gpu_moe.py."""

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
    (256, 256, 96, 2, 1, 128, False, False),   # full blocks: the last run's only padding is whole blocks
    (9, 256, 128, 16, 1, 128, True, False),    # experts without a token
])
def test_checkpoint_padding(T, H, I, E, k, B, skip, cond):
    import torch
    from nkilib.core.moe.moe_cte import SkipMode, build_token_blocks
    from nkilib.core.moe.moe_cte.bwmm_shard_on_block import run_dense_variant

    dev = torch.device("cuda:0")
    c = dense_case(T, H, I, E, k, B, seed=41, skip_token=skip, bias=True, hidden_std=1.0)
    ids = i32_tensor(ob.router_with_controlled_distribution(T, k, E).astype(np.int32), dev)
    args = (bf16_tensor(c["hidden"], dev), bf16_tensor(c["aff"].reshape(-1, 1), dev), bf16_tensor(c["gate_up_w"], dev),
            bf16_tensor(c["down_w"], dev))
    outs = []
    for planned in (False, True):
        tp, b2e, co = build_token_blocks(ids, E, B, c["N"], skip_token=skip)
        assert np.array_equal(tp.cpu().numpy(), c["tp2id"])
        if not planned:  # (copies: not the tables that the plan belongs to)
            tp, b2e, co = tp.clone(), b2e.clone(), co.clone()
        junk = [torch.full((c["N"] * B * max(2 * I, H),), float("nan"), dtype=torch.bfloat16, device=dev) for _ in range(2)]
        del junk  # the checkpoints are allocated over it
        outs.append(run_dense_variant(*args, B, tp, b2e, "TH", conditions=co if cond else None,
                                      gate_and_up_proj_bias=bf16_tensor(c["gate_up_bias"], dev),
                                      down_proj_bias=bf16_tensor(c["down_bias"], dev), skip_dma=SkipMode(skip, False),
                                      checkpoint_gate_up=True, checkpoint_down=True))
    torch.cuda.synchronize()
    g_out, g_gu, g_d = omoe.moe_blockwise_ref(
        c["hidden"], c["aff"], c["gate_up_w"], c["down_w"], c["tp2id"], c["b2e"], B,
        conditions=c["cond"] if cond else None, gate_up_proj_bias=c["gate_up_bias"], down_proj_bias=c["down_bias"],
        activation_function=0, skip_token=skip, expert_affinities_scaling_mode=1, checkpoint_activation=True)
    for out, gu, d in outs:
        _check(from_bf16_tensor(out)[:T], g_out[:T], "output")
        _check(from_bf16_tensor(gu), g_gu, "gate_up_activations_T")
        _check(from_bf16_tensor(d), g_d, "down_activations")
    for x, y in zip(*outs):
        assert torch.equal(x.view(torch.int16), y.view(torch.int16))
