"""Launches issued before the host has read the argument checks (fa_check_bounds / fa_check_wait): a failing check
raises before the call returns, the guarded kernels then write nothing, and a passing one changes no result."""
import numpy as np
import pytest
import torch

from _helpers import ATOL, assert_close, randn, to_np
from oracle import attention as ora

pytestmark = pytest.mark.gpu

DEV = "cuda"
D = 64


def _append_args(dtype=torch.float16, paged=False):
    B, hq, hk, cap, n = 3, 4, 2, 256, 2
    page = 64
    shape = (B * cap // page, page, hk, D) if paged else (B, cap, hk, D)
    a = dict(q=randn((B, n, hq, D), 1, dtype), k_cache=randn(shape, 2, dtype), v_cache=randn(shape, 3, dtype),
             k=randn((B, n, hk, D), 4, dtype), v=randn((B, n, hk, D), 5, dtype),
             cache_seqlens=torch.tensor([0, 100, 254], dtype=torch.int32))
    if paged:
        a["block_table"] = torch.randperm(B * cap // page, generator=torch.Generator().manual_seed(6)).reshape(B, -1).int()
    return a


def _tables(rows, dtype):
    ang = torch.arange(rows).float()[:, None] * (10000.0 ** (-torch.arange(0, D, 2).float() / D))[None, :]
    return ang.cos().to(dtype), ang.sin().to(dtype)


@pytest.mark.parametrize("what", ["length", "negative", "page", "host_page", "rotary", "leftpad"])
def test_rejected_append_leaves_the_cache(what):
    from flash_attn_triton import flash_attn_with_kvcache
    a = _append_args(paged=what in ("page", "host_page"))
    exc, match = ValueError, "do not fit"
    if what == "length":
        a["cache_seqlens"][1] = 255
    elif what == "negative":
        a["cache_seqlens"][0] = -1
    elif what in ("page", "host_page"):
        a["block_table"][2, 3] = 12
        exc, match = ValueError, "invalid physical page"
    elif what == "rotary":
        a["rotary_cos"], a["rotary_sin"] = _tables(255, torch.float16)
        exc, match = IndexError, "rotary"
    else:
        a["cache_leftpad"] = torch.tensor([0, 3, 1], dtype=torch.int32)
    # (host_page: a block table on the CPU, which is checked there)
    d = {n: t if what == "host_page" and n == "block_table" else t.to(DEV) for n, t in a.items()}
    for _ in range(2):
        with pytest.raises(exc, match=match):
            flash_attn_with_kvcache(**d, causal=True)
        torch.cuda.synchronize()
        assert torch.equal(d["k_cache"].cpu(), a["k_cache"]) and torch.equal(d["v_cache"].cpu(), a["v_cache"])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("table", [torch.float16, torch.bfloat16, torch.float32, torch.float64])
@pytest.mark.parametrize("paged,interleaved", [(False, True), (True, False)])
def test_append_rotary_table_types(dtype, table, paged, interleaved):
    from flash_attn_triton import flash_attn_with_kvcache
    a = _append_args(dtype, paged)
    cos, sin = _tables(256, table)
    d = {n: t.to(DEV) for n, t in a.items()}
    out = flash_attn_with_kvcache(**d, rotary_cos=cos.to(DEV), rotary_sin=sin.to(DEV), causal=True,
                                  rotary_interleaved=interleaved)
    np_a = {n: to_np(a[n]) for n in ("q", "k_cache", "v_cache")}
    rounded = [to_np(t.to(dtype)) for t in (cos, sin)]   # the tables enter in the input type
    ref, _, kref, vref = ora.attention_kvcache(
        np_a["q"], np_a["k_cache"], np_a["v_cache"], cache_seqlens=a["cache_seqlens"].numpy(),
        block_table=a["block_table"].numpy() if paged else None, causal=True, k_new=to_np(a["k"]), v_new=to_np(a["v"]),
        rotary_cos=rounded[0], rotary_sin=rounded[1], rotary_interleaved=interleaved)
    # fp32: the rotation and the softmax in fp32 (inputs of size 4, head dim 64): 5e-5 as for the other fp32 paths
    tol = 5e-5 if dtype == torch.float32 else 2 * ATOL[dtype]   # q and k are rounded once more after the rotation
    assert_close(to_np(out.cpu()), ref, tol, "out", dtype)
    # one rounding of the rotated k
    assert_close(to_np(d["k_cache"].cpu()), kref, 1e-6, "k cache", dtype)
    assert np.array_equal(to_np(d["v_cache"].cpu()), vref)


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("head_dim,dtype", [(128, torch.float16), (64, torch.bfloat16), (32, torch.float16),
                                            (16, torch.float16), (64, torch.float32)])
def test_varlen_guarded(grad, head_dim, dtype):
    from flash_attn_triton import flash_attn_varlen_func
    lens = [5, 0, 300, 33]
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32)
    q, k, v = (randn((sum(lens), 2, head_dim), i, dtype).to(DEV).requires_grad_(grad) for i in (11, 12, 13))
    # far out of range: an unguarded launch would leave the tensors
    for bad in ([0, 5, 5, 1 << 29, 338], [0, -(1 << 29), 5, 305, 338], [0, 5, 5, 305, 1 << 30]):
        for args in ((torch.tensor(bad, dtype=torch.int32), cu), (cu, torch.tensor(bad, dtype=torch.int32))):
            with pytest.raises(ValueError, match="cu_seqlens|max sequence"):
                flash_attn_varlen_func(q, k, v, args[0].to(DEV), args[1].to(DEV), 300, 300, causal=True)
    out = flash_attn_varlen_func(q, k, v, cu.to(DEV), cu.to(DEV), 300, 300, causal=True)
    ref, _ = ora.attention_varlen(to_np(q), to_np(k), to_np(v), cu.numpy(), cu.numpy(), None, True)
    assert_close(to_np(out), ref, 5e-5 if dtype == torch.float32 else ATOL[dtype], "out", dtype)
    if grad:
        out.sum().backward()
        assert all(torch.isfinite(t.grad).all() for t in (q, k, v))


def test_more_checks_than_one_launch_holds():
    from flash_attn_triton._checks import Deferred
    ts = [torch.arange(i, i + 300, dtype=torch.int32, device=DEV) for i in range(11)]
    seen = []
    for bad in (None, 0, 7, 8, 10):
        chk = Deferred()
        for i, t in enumerate(ts):
            chk.check_range(t, 0, i + 299 - (i == bad), ValueError(f"check {i}"))
            chk.check_range(t, i, None, ValueError("low"))   # the same array again: one reduction
        assert chk.ranges_only()
        if bad is None:
            chk.flush(lambda g: seen.append(g.tolist()), guarded=True)
        else:
            with pytest.raises(ValueError, match=f"check {bad}$"):
                chk.flush(lambda g: seen.append(g.tolist()), guarded=True)
        assert seen[-1] == [int(i == bad) for i in range(11)]


def test_check_behind_queued_work_and_launch_errors():
    # The checked values are produced by work still queued on the stream (a decode call checks on a second stream,
    # which has to wait for it), and a failing check goes before an error of the launch itself.
    from flash_attn_triton import flash_attn_with_kvcache
    from flash_attn_triton._checks import Deferred
    kc, vc, q = (randn((2, n, 2, D), i).to(DEV) for n, i in ((128, 21), (128, 22), (1, 23)))
    big = torch.randn(4096, 4096, device=DEV)
    lens = torch.full((2,), 1000, dtype=torch.int32, device=DEV)
    torch.cuda.synchronize()
    for value, ok in ((128, True), (129, False)):
        x = big
        for _ in range(8):
            x = x @ big * 1e-2
        lens.copy_((x[:2, 0] * 0).to(torch.int32) + value)
        if ok:
            assert torch.isfinite(flash_attn_with_kvcache(q, kc, vc, cache_seqlens=lens)).all()
        else:
            with pytest.raises(ValueError, match="valid lengths"):
                flash_attn_with_kvcache(q, kc, vc, cache_seqlens=lens)
        lens.fill_(1000)

    def fails():
        raise KeyError("launch")
    chk = Deferred()
    chk.check_range(lens, 0, 10, ValueError("check"))
    with pytest.raises(ValueError, match="check"):
        chk.flush(fails)
    chk.check_range(lens, 0, 1000, ValueError("check"))
    with pytest.raises(KeyError):
        chk.flush(fails)


def test_update_writes_lengths_without_work():
    # Nothing to append or rotate: the new lengths are written all the same, except with a failed guard.
    from flash_attn_triton import _native
    kc, q = torch.zeros((3, 16, 2, D), dtype=torch.float16, device=DEV), torch.zeros((3, 1, 2, D), dtype=torch.float16,
                                                                                   device=DEV)
    lens = torch.tensor([5, 0, 16], dtype=torch.int32, device=DEV)
    for flag in (0, 1):
        out = torch.full((3,), -7, dtype=torch.int32, device=DEV)
        guard = torch.tensor([0, flag], dtype=torch.int32, device=DEV)
        _native.kvcache_update(None, None, kc, kc, lens, None, None, None, 16, None, None, True, q, None, out, guard)
        assert out.tolist() == ([-7] * 3 if flag else [5, 0, 16])


def test_rejected_dropout_call_leaves_the_generator():
    from flash_attn_triton import flash_attn_varlen_func
    q = randn((20, 2, D), 41).to(DEV)
    good, bad = (torch.tensor(c, dtype=torch.int32, device=DEV) for c in ([0, 7, 20], [0, 7, 19]))
    torch.manual_seed(5)
    state = torch.get_rng_state()
    with pytest.raises(ValueError, match="cover"):
        flash_attn_varlen_func(q, q, q, bad, bad, 13, 13, dropout_p=0.5)
    assert torch.equal(torch.get_rng_state(), state)
    first = flash_attn_varlen_func(q, q, q, good, good, 13, 13, dropout_p=0.5)
    assert not torch.equal(torch.get_rng_state(), state)   # one draw per call that runs
    torch.manual_seed(5)
    assert torch.equal(flash_attn_varlen_func(q, q, q, good, good, 13, 13, dropout_p=0.5), first)
