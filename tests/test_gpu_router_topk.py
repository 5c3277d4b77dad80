"""GPU parity of the router top-k front end (through the C ABI) against oracle/router.py.

Bars: expert indices identical wherever the k-th and (k+1)-th logits are further apart than the fp32 GEMM's
reordering noise (1e-5; otherwise either expert is a correct answer) and in descending-logit order; logits within
bf16 rounding (output dtype) of the fp64-accumulated oracle; affinities max-abs-rel <= 1e-2 (bf16 output).
"""

import numpy as np
import pytest

from oracle import router as orr
from oracle.compare import max_abs_rel
from oracle.numerics import bf16_from_bits

pytestmark = pytest.mark.gpu


def _np(t):
    import torch

    if t.dtype == torch.bfloat16:
        return bf16_from_bits(t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16))
    return t.cpu().numpy()


@pytest.mark.parametrize(
    "T,H,E,k,act,pre,norm,bias,layout",
    [
        (300, 512, 64, 2, 1, True, False, True, 1),     # softmax over all experts, unmasked (reference default)
        (1000, 7168, 256, 8, 0, True, True, False, 1),  # DeepSeek-V3 shape: sigmoid, top-8, renormalised
        (257, 1024, 100, 4, 1, False, False, True, 0),  # activation after the selection, E not a multiple of 16, x [H, T]
        (64, 256, 512, 8, 0, False, False, False, 1),   # E = 512
        (5, 128, 8, 8, 1, True, True, True, 1),         # k == E, ragged T
    ],
)
def test_router_topk_matches_oracle(T, H, E, k, act, pre, norm, bias, layout):
    import torch
    from nkilib.core.router_topk import router_topk
    from nkilib.core.utils.common_types import RouterActFnType

    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(11)
    x = torch.empty((T, H), device=dev).uniform_(-1, 1, generator=g).to(torch.bfloat16)
    w = torch.empty((H, E), device=dev).uniform_(-0.1, 0.1, generator=g).to(torch.bfloat16)
    b = torch.empty((1, E), device=dev).uniform_(-0.5, 0.5, generator=g).to(torch.bfloat16) if bias else None
    xin = x if layout == 1 else x.t().contiguous()
    outs = router_topk[2](xin, w, b, None, None, None, RouterActFnType(act), k, layout, 0, router_pre_norm=pre,
                          norm_topk_prob=norm, return_eager_affi=True)
    torch.cuda.synchronize()
    logits, idx, aff, topk_aff = outs
    r = orr.router_topk_ref(_np(x), _np(w), None if b is None else _np(b).reshape(-1), act, k, router_pre_norm=pre,
                            norm_topk_prob=norm)
    lg = _np(logits)
    assert np.abs(lg - r["router_logits"]).max() <= 2 ** -8 * np.abs(r["router_logits"]).max() + 1e-6
    gap = orr.topk_gap(r["router_logits"], k)
    safe = gap > 1e-5
    gi = idx.cpu().numpy()
    assert safe.mean() > 0.95
    assert np.array_equal(np.sort(gi[safe], axis=1), np.sort(r["expert_index"][safe], axis=1))
    # order: descending logits (compare through the oracle's logits; equal logits may swap)
    picked = np.take_along_axis(r["router_logits"], gi.astype(np.int64), axis=1)
    assert (np.diff(picked, axis=1) <= 1e-5).all()
    a = _np(aff)
    err = max_abs_rel(a[safe], r["expert_affinities"][safe])
    print(f"router T={T} E={E} k={k}: affinity max-abs-rel {err:.2e}, {100 * (1 - safe.mean()):.2f}% near-ties", flush=True)
    assert err <= 1e-2
    ta = topk_aff.cpu().numpy()
    want = np.take_along_axis(r["expert_affinities"], gi.astype(np.int64), axis=1)
    assert np.abs(ta[safe] - want[safe]).max() <= 1e-5 + 1e-4 * np.abs(want).max()


@pytest.mark.parametrize("small_ws,unaligned", [(True, False), (False, False), (False, True)])
@pytest.mark.parametrize("aff_bf16", [False, True])
@pytest.mark.parametrize(
    "T,H,E,k,act,pre,norm,mask,bias",
    [
        (70, 512, 64, 2, 1, 1, 0, 0, True),     # softmax over all experts, unmasked
        (70, 512, 64, 2, 0, 1, 0, 0, False),    # sigmoid, unmasked
        (65, 1024, 200, 8, 1, 1, 0, 1, False),  # softmax, zeros outside the selected
        (130, 448, 256, 4, 0, 1, 1, 0, True),   # sigmoid, renormalised
        (33, 512, 100, 3, 1, 1, 1, 1, True),    # softmax, renormalised
        (129, 640, 300, 4, 1, 0, 0, 0, True),   # activation after the selection; more than 256 experts
        (1, 128, 17, 8, 0, 0, 0, 0, False),
    ],
)
def test_router_c_entry_matches_oracle(T, H, E, k, act, pre, norm, mask, bias, aff_bf16, small_ws, unaligned):
    """Every form through the C entry on both of its paths: with the small workspace, and for tokens that are not 16-byte
    aligned whatever the workspace, one launch walks K and selects; otherwise K is split over workgroups."""
    import torch
    from nkilib import _native as nv

    dev = torch.device("cuda:0")
    L = nv.lib()
    g = torch.Generator(device=dev).manual_seed(T + E)
    buf = torch.empty((T * H + 1,), dtype=torch.bfloat16, device=dev).uniform_(-1, 1, generator=g)
    x = (buf[1:] if unaligned else buf[:-1]).view(T, H)
    assert (x.data_ptr() % 16 != 0) == unaligned
    w = torch.empty((H, E), device=dev).uniform_(-0.1, 0.1, generator=g).to(torch.bfloat16)
    b = torch.empty((E,), device=dev).uniform_(-0.5, 0.5, generator=g) if bias else None
    size = L.moe_router_topk_workspace_bytes(H, E) if small_ws else L.moe_router_topk_workspace_bytes_for(T, H, E)
    ws = torch.full((size,), 255, dtype=torch.uint8, device=dev)
    logits = torch.empty((T, E), device=dev)
    idx = torch.empty((T, k), dtype=torch.int32, device=dev)
    aff = torch.full((T + 1, E), 7.0, dtype=torch.bfloat16 if aff_bf16 else torch.float32, device=dev)
    topk = torch.empty((T, k), device=dev)
    nv.check(L.moe_router_topk(nv.ptr(x), nv.ptr(w), nv.ptr(b), nv.DT_FP32, T, H, E, k, act, pre, norm, mask, 1,
                               nv.ptr(logits), nv.DT_FP32, nv.ptr(idx), nv.ptr(aff),
                               nv.DT_BF16 if aff_bf16 else nv.DT_FP32, nv.ptr(topk), nv.ptr(ws), size,
                               nv.stream_ptr(dev)), "router")
    torch.cuda.synchronize()
    r = orr.router_topk_ref(_np(x), _np(w), None if b is None else b.cpu().numpy(), act, k, router_pre_norm=bool(pre),
                            norm_topk_prob=bool(norm))
    # (the bound on the logits is that of the next test)
    bound = 8 * H ** 0.5 * 2.0 ** -24 * (np.abs(_np(x)) @ np.abs(_np(w)) + 0.5) + 1e-6
    assert (np.abs(_np(logits) - r["router_logits"]) <= bound).all()
    srt = -np.sort(-r["router_logits"], axis=1)
    safe = (srt[:, :k] - srt[:, 1:k + 1]).min(axis=1) > 2 * bound.max()
    assert safe.mean() > 0.5
    gi = idx.cpu().numpy()
    assert np.array_equal(gi[safe], r["expert_index"][safe])
    want = r["expert_affinities"].copy()
    if mask:  # (the oracle has no such option: zeros outside the selected experts)
        keep = np.zeros_like(want, dtype=bool)
        np.put_along_axis(keep, r["expert_index"].astype(np.int64), True, axis=1)
        want[~keep] = 0
    # both activations follow the logits with a relative slope of at most 1, quotients with twice that, and once more where
    # they are renormalised; exponents of up to 16 are rounded by 2^-20 on either side; bf16 rounds by 2^-8 of the value
    rel = 4 * bound.max() + 2.0 ** -18
    assert (np.abs(_np(aff)[:T] - want)[safe] <= (rel + (2.0 ** -8 if aff_bf16 else 0)) * np.abs(want)[safe]).all()
    assert not _np(aff)[T].any()
    sel = np.take_along_axis(want, gi.astype(np.int64), axis=1)
    assert (np.abs(topk.cpu().numpy() - sel)[safe] <= rel * np.abs(sel)[safe]).all()


@pytest.mark.parametrize(
    "T,H,E,k",
    [
        (1, 128, 8, 2),       # one token, a single part of K
        (64, 7168, 256, 8),   # a full tile of 64 tokens, K in 16 parts
        (65, 7168, 256, 8),   # a second tile of one token
        (4097, 256, 200, 4),  # the first of the 128-token tiles of a group of 256, one token in the last tile
        (8193, 192, 100, 3),  # the same of a group of 128
        (129, 1024, 128, 6),  # a third tile of one token, experts in one group of 128
        (40, 1088, 100, 4),   # K steps that the parts do not share out evenly, padded experts
        (700, 896, 65, 3),    # one expert past the group of 64
        (33000, 192, 60, 2),  # more tiles than CUs: one part
        (200, 640, 260, 8),   # two groups of 256
    ],
)
def test_router_split_over_k_matches_the_unsplit_kernel(T, H, E, k):
    """The C entry with the small workspace (one workgroup per token tile) and with the one for K split over workgroups:
    the logits differ by the order of fp32 sums: H roundings of independent sign, each at most 2^-24 * sum |x w|, so
    sqrt(H) of these is a deviation of either side's sum, taken four times for both sides.  Where the logits around the
    selected ones are further apart than that the selections are equal."""
    import torch
    from nkilib import _native as nv

    dev = torch.device("cuda:0")
    L = nv.lib()
    g = torch.Generator(device=dev).manual_seed(T)
    x = torch.randn((T, H), generator=g, device=dev).to(torch.bfloat16)
    w = (torch.randn((H, E), generator=g, device=dev) * H ** -0.5).to(torch.bfloat16)
    b = torch.randn((E,), generator=g, device=dev)
    res = []
    for size in (L.moe_router_topk_workspace_bytes(H, E), L.moe_router_topk_workspace_bytes_for(T, H, E)):
        ws = torch.full((size,), 255, dtype=torch.uint8, device=dev)
        lg = torch.empty((T, E), device=dev)
        idx = torch.empty((T, k), dtype=torch.int32, device=dev)
        aff = torch.full((T + 1, E), 7.0, device=dev)
        nv.check(L.moe_router_topk(nv.ptr(x), nv.ptr(w), nv.ptr(b), nv.DT_FP32, T, H, E, k, 0, 1, 1, 1, 1, nv.ptr(lg),
                                   nv.DT_FP32, nv.ptr(idx), nv.ptr(aff), nv.DT_FP32, None, nv.ptr(ws), size,
                                   nv.stream_ptr(dev)), "router")
        torch.cuda.synchronize()
        res.append((lg, idx, aff))
    (l0, i0, a0), (l1, i1, a1) = res
    bound = 8 * H ** 0.5 * 2.0 ** -24 * (x.abs().float() @ w.abs().float()) + 1e-6
    assert ((l0 - l1).abs() <= bound).all()
    assert not a0[T].any() and not a1[T].any()
    srt = l0.sort(dim=1, descending=True).values
    gaps = (srt[:, :k] - srt[:, 1:k + 1]).min(dim=1).values if k < E else (srt[:, :k - 1] - srt[:, 1:k]).min(dim=1).values
    safe = gaps > bound.max()
    assert safe.float().mean() > 0.5
    assert torch.equal(i0[safe], i1[safe])
    assert (a0[:T][safe] - a1[:T][safe]).abs().max() <= 2 * bound.max()


def test_route_for_moe_feeds_the_block_build():
    """Masked table + ids from hidden states: zero outside the top-k, zero padding row, ids usable as they are."""
    import torch
    from nkilib.core.moe.moe_cte import build_token_blocks, get_n_blocks
    from nkilib.core.router_topk import route_for_moe
    from nkilib.core.utils.common_types import RouterActFnType

    dev = torch.device("cuda:0")
    T, H, E, k, B = 512, 1024, 32, 4, 128
    g = torch.Generator(device=dev).manual_seed(3)
    x = torch.randn((T + 1, H), generator=g, device=dev).to(torch.bfloat16)
    x[T] = 0
    w = (torch.randn((H, E), generator=g, device=dev) * 0.05).to(torch.bfloat16)
    ids, aff = route_for_moe(x, w, None, k, RouterActFnType.SIGMOID, norm_topk_prob=True)
    torch.cuda.synchronize()
    a = _np(aff)
    assert a.shape == (T + 1, E) and not a[T].any()
    assert ((a[:T] > 0).sum(axis=1) == k).all()
    np.testing.assert_allclose(a[:T].sum(axis=1), 1.0, atol=2e-2)
    rows = np.arange(T)[:, None]
    assert (a[rows, ids.cpu().numpy()] > 0).all()
    N = get_n_blocks(T, k, E, B, n_block_per_iter=2)
    tp2id, b2e, _ = build_token_blocks(ids, E, B, N, n_conditions=N + 2)
    assert int((tp2id.reshape(-1) < T).sum()) == T * k
