"""Backward launches with few workgroups (two wave pairs per key group in the dK/dV kernel), the causal spans of the
dense backward and the longest-first order of varlen launches, at the edges of their tiles, against the float64
oracle.  Gradients are compared relative to the largest gradient, as fp16 / bf16 gradients carry their own rounding:
1e-2 / 4e-2, the bars of the other 16-bit backward tests' scale."""
import numpy as np
import pytest
import torch

from _helpers import randn, to_np
from oracle import attention as ora

pytestmark = pytest.mark.gpu

DEV = "cuda"
TOL = {torch.float16: 1e-2, torch.bfloat16: 4e-2}


def _check(got, ref, dtype):
    for name, g, r in zip(("dq", "dk", "dv"), got, ref):
        g = to_np(g)
        assert np.all(np.isfinite(g)), name
        err = np.max(np.abs(g - r)) / max(1.0, np.max(np.abs(r)))
        assert err <= TOL[dtype], f"{name}: {err:.2e}"


# Key blocks of 64 (one wave pair per 32-row half of a 64-row tile): one block, its edges, rows short of a half tile.
@pytest.mark.parametrize("sq,sk", [(1, 1), (31, 64), (33, 65), (64, 127), (96, 128), (161, 130), (300, 257), (65, 400)])
@pytest.mark.parametrize("causal,window", [(False, (-1, -1)), (True, (-1, -1)), (True, (70, 0)), (False, (20, 33))])
@pytest.mark.parametrize("head_dim,hq,hk,dtype", [(128, 2, 2, torch.float16), (64, 6, 2, torch.bfloat16)])
def test_dense(sq, sk, causal, window, head_dim, hq, hk, dtype):
    from flash_attn_triton import flash_attn_func
    q, k, v = (randn((2, n, h, head_dim), i, dtype) for n, h, i in ((sq, hq, 1), (sk, hk, 2), (sk, hk, 3)))
    dout = randn((2, sq, hq, head_dim), 4, dtype)
    leaves = [t.to(DEV).requires_grad_() for t in (q, k, v)]
    out = flash_attn_func(*leaves, causal=causal, window_size=window)
    got = torch.autograd.grad(out, leaves, dout.to(DEV))
    ref = ora.attention_backward(to_np(q), to_np(k), to_np(v), to_np(dout), causal=causal, window_size=window)
    _check(got, ref[:3], dtype)


def _counts(batch, heads, causal):
    from flash_attn_triton import flash_attn_func
    s, d = 140, 64
    q, k, v, dout = (randn((batch, s, heads, d), i) for i in (11, 12, 13, 14))
    leaves = [t.to(DEV).requires_grad_() for t in (q, k, v)]
    got = torch.autograd.grad(flash_attn_func(*leaves, causal=causal), leaves, dout.to(DEV))
    ref = ora.attention_backward(to_np(q), to_np(k), to_np(v), to_np(dout), causal=causal)
    _check(got, ref[:3], torch.float16)


# 300 workgroups of 128 keys is the last count of the two-pair form (causal), 150 without a mask: both sides of them (140
# keys are two workgroups a head, so 300 and 302, 150 and 152), and group counts that do and do not fill the spans.
@pytest.mark.parametrize("batch,heads", [(1, 3), (20, 5), (30, 5), (151, 1), (60, 5), (61, 5), (25, 8)])
def test_causal_counts(batch, heads):
    _counts(batch, heads, True)


@pytest.mark.parametrize("batch,heads", [(15, 5), (19, 4)])
def test_full_counts(batch, heads):
    _counts(batch, heads, False)


# A varlen launch counts by its packed keys: 10 sequences of 1910 keys in all are 14 + 5 workgroups a head (the grid,
# sized for the longest, has 130): 285 and 304 (causal), 133 and 152 with 15, 16, 7 and 8 heads.
@pytest.mark.parametrize("heads,causal", [(15, True), (16, True), (7, False), (8, False)])
def test_varlen_workgroup_counts(heads, causal):
    from flash_attn_triton import flash_attn_varlen_func
    lengths, d = [30] * 4 + [1640] + [30] * 5, 64
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lengths)]), dtype=torch.int32)
    q, k, v, dout = (randn((int(cu[-1]), heads, d), i) for i in (31, 32, 33, 34))
    leaves = [t.to(DEV).requires_grad_() for t in (q, k, v)]
    out = flash_attn_varlen_func(*leaves, cu.to(DEV), cu.to(DEV), max(lengths), max(lengths), causal=causal)
    got = torch.autograd.grad(out, leaves, dout.to(DEV))
    ref = ora.attention_varlen_backward(to_np(q), to_np(k), to_np(v), to_np(dout), cu.numpy(), cu.numpy(), None, causal)
    _check(got, ref[:3], torch.float16)


# More than 64 sequences (ranked in blocks of 64), equal and zero lengths, K/V head counts around the 8 XCDs.
@pytest.mark.parametrize("lengths", [[5, 0, 130, 130, 64], list(range(1, 71)), [0, 0, 300], [40] * 66 + [200]])
@pytest.mark.parametrize("hq,hk,head_dim", [(4, 2, 128), (9, 9, 64), (8, 1, 64)])
@pytest.mark.parametrize("causal", [False, True])
def test_varlen(lengths, hq, hk, head_dim, causal):
    from flash_attn_triton import flash_attn_varlen_func
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lengths)]), dtype=torch.int32)
    T = int(cu[-1])
    q, k, v, dout = (randn((T, h, head_dim), i) for h, i in ((hq, 21), (hk, 22), (hk, 23), (hq, 24)))
    leaves = [t.to(DEV).requires_grad_() for t in (q, k, v)]
    out = flash_attn_varlen_func(*leaves, cu.to(DEV), cu.to(DEV), max(lengths), max(lengths), causal=causal)
    ref_out, _ = ora.attention_varlen(to_np(q), to_np(k), to_np(v), cu.numpy(), cu.numpy(), None, causal)
    assert np.max(np.abs(to_np(out) - ref_out)) <= 4e-3   # fp16 outputs up to 4: half an ulp is 2e-3 more than the bar
    got = torch.autograd.grad(out, leaves, dout.to(DEV))
    ref = ora.attention_varlen_backward(to_np(q), to_np(k), to_np(v), to_np(dout), cu.numpy(), cu.numpy(), None, causal)
    _check(got, ref[:3], torch.float16)
