"""The bookkeeping of calls without a block plan (csrc/combine.hip): the single launch and the four launches, on either
side of the sizes that part them (2048 blocks, 4096 tokens), block sizes that are no multiples of a unit of 64 slots, a stop
condition in the middle.  Layers against the oracle at the tolerance of test_gpu_moe.py."""

import numpy as np
import pytest

from helpers import dense_case, from_bf16_tensor
from test_gpu_moe import _check, _golden_dense, _run_dense

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,B,E,k", [
    (4096, 4, 8, 2),   # 2055 blocks: four launches
    (4096, 5, 8, 2),   # 1643 blocks of five slots, every list place taken
    (4097, 64, 8, 2),  # a token too many for the single launch
    (4096, 65, 8, 2),  # two units per block, the second of a single slot
    (300, 512, 4, 4),
    (1, 128, 8, 2),
])
def test_layer_from_tables(T, B, E, k):
    c = dense_case(T, 256, 64, E, k, B, seed=51, hidden_std=1.0)
    o = from_bf16_tensor(_run_dense(c, impl="shard_on_i"))
    _check(o[:T], _golden_dense(c)[:T], f"tables T={T} B={B}")


def test_stop_condition():
    c = dense_case(700, 256, 64, 4, 2, 96, seed=52, hidden_std=1.0)
    cond = np.ones(c["N"] + 1, np.int32)
    cond[c["N"] - 3:] = 0
    o = from_bf16_tensor(_run_dense(c, impl="shard_on_i_hybrid", conditions=cond))
    _check(o[:700], _golden_dense(c, conditions=cond)[:700], "stop condition")
