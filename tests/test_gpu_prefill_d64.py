"""The head-dim-64 prefill kernel at the edges of its tiles (64 keys), row blocks (128 rows, 32 per wave), its three
runs of tiles (upper boundary, unmasked, lower boundary) and its launch forms, against the float64 oracle."""
import numpy as np
import pytest
import torch

from _helpers import ATOL, assert_close, randn, to_np
from oracle import attention as ora

pytestmark = pytest.mark.gpu

DEV = "cuda"
D = 64


def _cu(n):
    return torch.tensor(np.concatenate([[0], np.cumsum(n)]), dtype=torch.int32)


@pytest.mark.parametrize("sq,sk", [(1, 1), (31, 64), (64, 65), (127, 127), (128, 128), (129, 320), (300, 63), (33, 449),
                                   (257, 512)])
@pytest.mark.parametrize("causal,window,offset", [(False, (-1, -1), 0), (True, (-1, -1), 0), (True, (-1, -1), 70),
                                                  (True, (-1, -1), -40), (True, (100, -1), 30), (False, (64, 64), 0),
                                                  (False, (-1, 10), -5), (False, (0, 0), 0)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_dense_edges(sq, sk, causal, window, offset, dtype):
    from flash_attn_triton.triton_kernel.attention_kernel import dense_forward
    hq, hk = 4, 2
    q, k, v = (randn((2, n, h, D), s, dtype) for n, h, s in ((sq, hq, 1), (sk, hk, 2), (sk, hk, 3)))
    out, lse = dense_forward(q.to(DEV), k.to(DEV), v.to(DEV), softmax_scale=0.2, causal=causal, q_pos_offset=offset,
                             window_left=window[0], window_right=window[1], return_lse=True)
    ref, ref_lse, _ = ora.attention(to_np(q), to_np(k), to_np(v), softmax_scale=0.2, causal=causal,
                                    window_size=window, causal_offset=offset)
    assert_close(to_np(out.cpu()), ref, ATOL[dtype], "out", dtype)
    got = lse.cpu().numpy()
    assert np.array_equal(np.isneginf(got), np.isneginf(ref_lse))
    fin = np.isfinite(ref_lse)
    assert np.max(np.abs(got[fin] - ref_lse[fin]), initial=0.0) < 1e-3


@pytest.mark.parametrize("batch,heads", [(1, 3), (2, 12), (1, 8), (3, 24), (5, 8)])
def test_causal_work_items(batch, heads):
    # Group counts that do and do not split over the 8 XCDs and the spans of the causal order: every row block of
    # every head is computed.
    from flash_attn_triton import flash_attn_func
    s = 700
    q, k, v = (randn((batch, s, heads, D), i) for i in (5, 6, 7))
    out = to_np(flash_attn_func(q.to(DEV), k.to(DEV), v.to(DEV), causal=True).cpu())
    ref, _, _ = ora.attention(to_np(q), to_np(k), to_np(v), causal=True)
    assert_close(out, ref, ATOL[torch.float16], "out", torch.float16)


def test_max_moves():
    # Scores that keep rising by more than the rescale slack along the walk (towards lower keys), by less, and rows
    # whose first tiles hold very negative scores.
    from flash_attn_triton import flash_attn_func
    s = 320
    q, k, v = (randn((1, s, 1, D), i) for i in (11, 12, 13))
    ramp = torch.linspace(6.0, -6.0, s)[None, :, None, None]
    k = (k * 0.2 + ramp * torch.sign(q.mean(1, keepdim=True).float())).half()
    for sign in (1, -1):
        out = to_np(flash_attn_func((sign * q).to(DEV), k.to(DEV), v.to(DEV)).cpu())
        ref, _, _ = ora.attention(to_np(sign * q), to_np(k), to_np(v))
        # large scores: exp of an fp32 score of size up to 50 is off by 50 * 2^-24 * few, far below the fp16 bar
        assert_close(out, ref, ATOL[torch.float16], f"sign {sign}", torch.float16)


@pytest.mark.parametrize("page", [0, 16, 48, 24])   # 24: not whole 16-row groups, the general kernel
@pytest.mark.parametrize("used", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_varlen(page, used, dtype):
    from flash_attn_triton import flash_attn_varlen_func
    lq, lk, hq, hk = [1, 256, 0, 300, 63], [64, 300, 9, 65, 700], 4, 2
    uq, uk = ([1, 200, 0, 257, 63], [33, 300, 0, 64, 650]) if used else (None, None)
    q = randn((sum(lq), hq, D), 21, dtype)
    bt = None
    if page:
        counts = [-(-n // page) for n in lk]
        perm = torch.randperm(sum(counts), generator=torch.Generator().manual_seed(1))
        bt = torch.zeros((len(lk), max(counts)), dtype=torch.int32)
        at = 0
        for b, c in enumerate(counts):
            bt[b, :c] = perm[at:at + c]
            at += c
        k, v = randn((at, page, hk, D), 22, dtype), randn((at, page, hk, D), 23, dtype)
    else:
        k, v = randn((sum(lk), hk, D), 22, dtype), randn((sum(lk), hk, D), 23, dtype)
    dev = lambda t: None if t is None else torch.as_tensor(t, dtype=torch.int32).to(DEV)
    out = flash_attn_varlen_func(q.to(DEV), k.to(DEV), v.to(DEV), _cu(lq).to(DEV), _cu(lk).to(DEV), max(lq), max(lk),
                                 causal=True, block_table=None if bt is None else bt.to(DEV), seqused_q=dev(uq),
                                 seqused_k=dev(uk))
    cq, ck, cv, cuq, cuk = ora.compact_varlen(to_np(q), to_np(k), to_np(v), _cu(lq).numpy(), _cu(lk).numpy(), uq, uk,
                                              None if bt is None else bt.numpy())
    ref, _ = ora.attention_varlen(cq, ck, cv, cuq, cuk, None, True)
    assert_close(to_np(out.cpu()), ref, ATOL[dtype], "varlen", dtype)


@pytest.mark.parametrize("sq,hq,hk", [(33, 2, 2), (127, 1, 1), (32, 8, 2), (129, 2, 2), (50, 6, 2)])
@pytest.mark.parametrize("page", [0, 16, 256, 40])
@pytest.mark.parametrize("causal,window", [(False, (-1, -1)), (True, (-1, -1)), (True, (100, 0))])
def test_cache_chunk(sq, hq, hk, page, causal, window):
    from flash_attn_triton import flash_attn_with_kvcache
    lengths = [0, 5, 64, 65, 511, 1300]
    kw = {}
    if page:
        counts = [-(-n // page) for n in lengths]
        perm = torch.randperm(sum(counts) + 1, generator=torch.Generator().manual_seed(2))
        bt = torch.zeros((len(lengths), max(counts)), dtype=torch.int32)
        at = 0
        for b, c in enumerate(counts):
            bt[b, :c] = perm[at:at + c]
            at += c
        shape = (at + 1, page, hk, D)
        kw["block_table"] = bt
    else:
        shape = (len(lengths) + 1, 1400, hk, D)
        kw["cache_batch_idx"] = torch.tensor([3, 0, 6, 1, 2, 5], dtype=torch.int32)
        kw["cache_leftpad"] = torch.tensor([0, 9, 0, 64, 100, 100], dtype=torch.int32)
    q, kc, vc = randn((len(lengths), sq, hq, D), 31), randn(shape, 32), randn(shape, 33)
    sl = torch.tensor(lengths, dtype=torch.int32)
    out = flash_attn_with_kvcache(q.to(DEV), kc.to(DEV), vc.to(DEV), cache_seqlens=sl.to(DEV), causal=causal,
                                  window_size=window, **{n: t.to(DEV) for n, t in kw.items()})
    ref, _, _, _ = ora.attention_kvcache(to_np(q), to_np(kc), to_np(vc), cache_seqlens=lengths, causal=causal,
                                         window_size=window, **{n: t.numpy() for n, t in kw.items()})
    assert_close(to_np(out.cpu()), ref, ATOL[torch.float16], "chunk", torch.float16)
