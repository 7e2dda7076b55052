"""Chunks of queries against a KV cache, and paged varlen, at head dim 128 on the ping-pong kernel: the edges of its
row blocks (256 packed rows), key tiles (64), key splits, pages (8-row groups) and of the rule that selects it,
against the float64 oracle."""
import math

import numpy as np
import pytest
import torch

from _helpers import ATOL, assert_close, randn, to_np
from oracle import attention as ora

pytestmark = pytest.mark.gpu

DEV = "cuda"
D = 128


def _paged(lengths, page, hk, seed, dtype):
    """Shuffled pages; the slots past each sequence's last key hold NaN, which no result may see."""
    counts = [-(-n // page) for n in lengths]
    perm = torch.randperm(sum(counts) + 1, generator=torch.Generator().manual_seed(seed))
    kc = randn((sum(counts) + 1, page, hk, D), seed + 1, dtype)
    vc = randn((sum(counts) + 1, page, hk, D), seed + 2, dtype)
    bt = torch.zeros((len(lengths), max(max(counts), 1)), dtype=torch.int32)
    at = 0
    for b, (n, c) in enumerate(zip(lengths, counts)):
        bt[b, :c] = perm[at:at + c]
        at += c
        if n % page:
            kc[bt[b, c - 1], n % page:] = float("nan")
            vc[bt[b, c - 1], n % page:] = float("nan")
    return kc, vc, bt


def _clean(t):
    return np.nan_to_num(to_np(t), nan=0.0)


# Rows per KV head: 33 (the smallest), 255 / 256 / 257 (one row block, two), 3 * 100 with an odd group.
@pytest.mark.parametrize("sq,hq,hk", [(33, 2, 2), (255, 1, 1), (64, 8, 2), (257, 2, 2), (100, 6, 2)])
@pytest.mark.parametrize("page", [8, 24, 256, 20])   # 20: not whole 8-row groups, the general kernel
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [False, True])
def test_paged_chunk(sq, hq, hk, page, dtype, causal):
    from flash_attn_triton import flash_attn_with_kvcache
    # no key, fewer keys than queries, tile edges, several splits
    lengths = [0, 5, 64, 65, 511, 1300]
    kc, vc, bt = _paged(lengths, page, hk, 300 + sq, dtype)
    q = randn((len(lengths), sq, hq, D), 303, dtype)
    sl = torch.tensor(lengths, dtype=torch.int32)
    out = flash_attn_with_kvcache(q.to(DEV), kc.to(DEV), vc.to(DEV), cache_seqlens=sl.to(DEV),
                                  block_table=bt.to(DEV), causal=causal)
    ref, _, _, _ = ora.attention_kvcache(to_np(q), _clean(kc), _clean(vc), cache_seqlens=lengths,
                                         block_table=bt.numpy(), causal=causal)
    assert_close(to_np(out.cpu()), ref, ATOL[dtype], "paged chunk", dtype)


@pytest.mark.parametrize("causal,window", [(False, (-1, -1)), (True, (-1, -1)), (True, (100, 0)), (False, (37, 20))])
def test_batched_chunk_rows_leftpad_lse(causal, window):
    # Batched cache with row indices and left padding, strided q (a slice of a packed projection), LSE of every row.
    from flash_attn_triton import _native, flash_attn_with_kvcache
    B, cap, hq, hk, sq = 3, 1400, 8, 2, 70
    kc, vc = randn((5, cap, hk, D), 311), randn((5, cap, hk, D), 312)
    q = randn((B, sq, hq + 2 * hk, D), 313)[:, :, :hq]
    rows = torch.tensor([4, 0, 2], dtype=torch.int32)
    pads = torch.tensor([0, 17, 100], dtype=torch.int32)
    lens = torch.tensor([1400, 900, 1], dtype=torch.int32)
    kw = dict(cache_batch_idx=rows.to(DEV), cache_leftpad=pads.to(DEV), causal=causal, window_size=window)
    base = randn((B, sq, hq + 2 * hk, D), 313).to(DEV)
    qd, kd, vd = base[:, :, :hq], kc.to(DEV), vc.to(DEV)
    out = flash_attn_with_kvcache(qd, kd, vd, cache_seqlens=lens.to(DEV), **kw)
    ref, ref_lse, _, _ = ora.attention_kvcache(to_np(q), to_np(kc), to_np(vc), cache_seqlens=lens.numpy(),
                                               cache_batch_idx=rows.numpy(), cache_leftpad=pads.numpy(),
                                               causal=causal, window_size=window)
    assert_close(to_np(out.cpu()), ref, ATOL[torch.float16], "batched chunk", torch.float16)
    out2 = torch.full_like(out, float("nan"))
    lse = torch.full((B, hq, sq), float("nan"), device=DEV)
    _native.fwd_kvcache(qd, kd, vd, out2, lse, lens.to(DEV), None, rows.to(DEV), pads.to(DEV), cap,
                        1.0 / math.sqrt(D), causal, window[0], window[1], None)
    assert torch.equal(out, out2)
    got = lse.cpu().numpy()
    assert np.array_equal(np.isneginf(got), np.isneginf(ref_lse))
    fin = np.isfinite(ref_lse)
    assert np.max(np.abs(got[fin] - ref_lse[fin])) < 1e-3


def test_chunk_unchecked_arguments_stay_in_the_cache():
    # The kernel itself clamps lengths past the capacity and reads pages outside the cache as zeros (the Python layer
    # raises for both only after the launch).
    from flash_attn_triton import _native
    page, hk, hq, sq = 16, 1, 1, 40
    kc, vc = randn((4, page, hk, D), 321).to(DEV), randn((4, page, hk, D), 322).to(DEV)
    bt = torch.tensor([[0, 1 << 28, 2, -7]], dtype=torch.int32)
    q = randn((1, sq, hq, D), 323)
    out = torch.empty((1, sq, hq, D), dtype=torch.float16, device=DEV)
    _native.fwd_kvcache(q.to(DEV), kc, vc, out, None, torch.tensor([10 ** 6], dtype=torch.int32, device=DEV),
                        bt.to(DEV), None, None, 4 * page, 1.0 / math.sqrt(D), False, -1, -1, None)
    k = torch.cat([kc[0].cpu(), torch.zeros(page, hk, D).half(), kc[2].cpu(), torch.zeros(page, hk, D).half()])[None]
    v = torch.cat([vc[0].cpu(), torch.zeros(page, hk, D).half(), vc[2].cpu(), torch.zeros(page, hk, D).half()])[None]
    ref, _, _ = ora.attention(to_np(q), to_np(k), to_np(v))
    assert_close(to_np(out.cpu()), ref, ATOL[torch.float16], "clamped", torch.float16)


@pytest.mark.parametrize("page", [8, 16, 40])
@pytest.mark.parametrize("used", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_paged_varlen(page, used, dtype):
    from flash_attn_triton import flash_attn_varlen_func
    lq, lk, hq, hk = [1, 256, 0, 300, 63], [64, 300, 9, 65, 700], 4, 2
    uq, uk = ([1, 200, 0, 257, 63], [33, 300, 0, 64, 650]) if used else (None, None)
    kc, vc, bt = _paged(lk, page, hk, 330, dtype)
    cu = lambda n: torch.tensor(np.concatenate([[0], np.cumsum(n)]), dtype=torch.int32)
    q = randn((sum(lq), hq, D), 331, dtype)
    dev = lambda t: None if t is None else torch.as_tensor(t, dtype=torch.int32).to(DEV)
    out = flash_attn_varlen_func(q.to(DEV), kc.to(DEV), vc.to(DEV), cu(lq).to(DEV), cu(lk).to(DEV), max(lq), max(lk),
                                 causal=True, block_table=bt.to(DEV), seqused_q=dev(uq), seqused_k=dev(uk))
    cq, ck, cv, cuq, cuk = ora.compact_varlen(to_np(q), _clean(kc), _clean(vc), cu(lq).numpy(), cu(lk).numpy(), uq, uk,
                                              bt.numpy())
    ref, _ = ora.attention_varlen(cq, ck, cv, cuq, cuk, None, True)
    assert_close(to_np(out.cpu()), ref, ATOL[dtype], "paged varlen", dtype)
