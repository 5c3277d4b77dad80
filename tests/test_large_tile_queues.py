"""The walk of the large-tile GEMMs over their queues (large_tile_queues.py): every tile is done once, whole or in pieces that cover
its rows, in the order of the instances; and the cases of test_gpu_moe_last_round.py are cut as they say."""

import numpy as np
import pytest

import large_tile_queues as lq
import test_gpu_moe_last_round as last_round


def test_every_row_of_every_tile_once_and_in_instance_order():
    rng = np.random.default_rng(5)
    seen = set()
    for _ in range(400):
        E = int(rng.integers(1, 40))
        rows = rng.integers(0, int(rng.choice([40, 130, 330, 1200])), size=E)
        slot, chunks = 0, []
        for e, r in enumerate(rows.tolist()):
            n = 0 if r == 0 else 1 if r <= 320 else -(-(r - 320) // 256) + 1
            chunks += [(slot + 256 * i, 256 if i + 1 < n else r - 256 * i, e) for i in range(n)]
            slot += -(-r // 128) * 128
        if not chunks:
            continue
        pad_row = bool(rng.integers(2))
        interleave, queues = lq.queues_of(chunks, pad_row)
        assert sorted(c for q in queues for _, c in q) == sorted(chunks)
        gx = int(rng.integers(1, 30))
        W = lq.workgroups_per_xcd(gx, len(chunks))
        for q in queues:
            whole, shift = lq.cut_of(q, interleave, gx, W)
            seen.add(shift)
            left = {i: q[i // gx][1][1] for i in range(len(q) * gx)}
            for w in range(W):
                last = -1
                for what, item, *x in lq.items_of(w, q, interleave, gx, W):
                    rows_, cls = (left[item], x[0]) if what == "whole" else (x[1], x[2])
                    left[item] -= rows_
                    # (equal only within one run of whole items: a piece has an instance behind all of them)
                    assert cls > last or (what == "whole" and cls == last)
                    last = cls
                    assert lq.row_tiles(rows_) <= [20, 20, 20 if pad_row else 18, 18, 16, 16, 14, 12, 10, 8, 8, 4][cls]
            assert not any(left.values())
    assert seen == {0, 1, 2}


@pytest.mark.parametrize("size", last_round.SIZES)
@pytest.mark.parametrize("T", last_round.ROWS)
@pytest.mark.parametrize("ckpt", [False, True])
def test_cases_are_cut_as_they_say(T, size, ckpt):
    last_round.check_cuts(T, size, ckpt)
