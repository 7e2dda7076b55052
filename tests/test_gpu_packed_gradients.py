"""Gradients of the packed entry points: written in place as one packed tensor where the attention's backward can, stacked
otherwise, and equal to those of the unpacked calls bit for bit."""
import pytest
import torch

from _helpers import randn

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _cu(lengths):
    return torch.tensor([0] + lengths, dtype=torch.int32).cumsum(0).to(torch.int32).to(DEV)


@pytest.mark.parametrize("dtype,head_dim,heads", [(torch.float16, 64, 3), (torch.bfloat16, 128, 2), (torch.float32, 32, 2),
                                                  (torch.float16, 16, 2), (torch.float16, 256, 1)])
@pytest.mark.parametrize("form", ["qkv", "kv", "kv_cross", "varlen_qkv", "varlen_kv"])
def test_packed_equals_unpacked(dtype, head_dim, heads, form):
    import flash_attn_triton as fa
    lens = [70, 0, 33, 130]
    T, cu = sum(lens), _cu(lens)
    n = 3 if form.endswith("qkv") else 2
    lead = (T,) if form.startswith("varlen") else (2, 77)
    packed = randn(lead + (n, heads, head_dim), 1, dtype).to(DEV).requires_grad_()
    qlead = (2, 40) if form == "kv_cross" else lead
    q = None if n == 3 else randn(qlead + (heads, head_dim), 2, dtype).to(DEV).requires_grad_()
    dout = randn(qlead + (heads, head_dim), 3, dtype).to(DEV)
    leaves = [packed] if q is None else [q, packed]
    args = leaves + ([cu, max(lens)] if form == "varlen_qkv" else [cu, cu, max(lens), max(lens)] if form == "varlen_kv" else [])
    fn = {"qkv": fa.flash_attn_qkvpacked_func, "kv": fa.flash_attn_kvpacked_func, "kv_cross": fa.flash_attn_kvpacked_func,
          "varlen_qkv": fa.flash_attn_varlen_qkvpacked_func, "varlen_kv": fa.flash_attn_varlen_kvpacked_func}[form]
    out = fn(*args, causal=form != "kv_cross")
    got = torch.autograd.grad(out, leaves, dout)
    parts = [t.detach().clone().requires_grad_() for t in packed.detach().unbind(-3)]
    qkv = parts if q is None else [q.detach().clone().requires_grad_()] + parts
    if form.startswith("varlen"):
        ref = fa.flash_attn_varlen_func(*qkv, cu, cu, max(lens), max(lens), causal=True)
    else:
        ref = fa.flash_attn_func(*qkv, causal=form != "kv_cross")
    want = torch.autograd.grad(ref, qkv, dout)
    assert torch.equal(out, ref)
    assert torch.equal(got[-1], torch.stack(want[-n:], -3))
    assert got[-1].is_contiguous()
    if q is not None:
        assert torch.equal(got[0], want[0])


def test_other_gradient_routes():
    # A second use of the packed tensor (accumulated gradients), a non-contiguous input (copied first), and gradients
    # through an output that only part of the loss reaches.
    from flash_attn_triton import flash_attn_qkvpacked_func
    x = randn((2, 64, 3, 2, 64), 5).to(DEV).requires_grad_()
    w = randn((2, 64, 2, 64), 6).to(DEV)
    (g,) = torch.autograd.grad((flash_attn_qkvpacked_func(x) * w).sum(), x)
    ((flash_attn_qkvpacked_func(x) * w).sum() + x.float().square().sum()).backward()
    assert torch.allclose(x.grad.float(), g.float() + 2 * x.detach().float(), rtol=2e-3, atol=4e-3)
    y = x.detach().transpose(0, 1).contiguous().transpose(0, 1).requires_grad_()
    (gy,) = torch.autograd.grad((flash_attn_qkvpacked_func(y) * w).sum(), y)
    assert torch.equal(gy, g)
    z = x.detach().clone().requires_grad_()
    out = flash_attn_qkvpacked_func(z)
    (gz,) = torch.autograd.grad(out[:1].float().sum() * 0 + (out * w).sum(), z)
    assert torch.equal(gz, g)


@pytest.mark.parametrize("head_dim,dtype", [(128, torch.float16), (64, torch.bfloat16), (256, torch.float16),
                                            (32, torch.float32)])
def test_varlen_gradients_write_every_row(head_dim, dtype):
    # The gradient tensors are not cleared first: every row of every sequence is written, also of sequences without
    # queries or without keys.
    from flash_attn_triton.triton_kernel.attention_kernel import varlen_backward, varlen_forward
    lq, lk = [70, 0, 33, 1, 0, 40], [64, 50, 0, 1, 0, 130]
    cq, ck = _cu(lq), _cu(lk)
    q, do = (randn((sum(lq), 4, head_dim), i, dtype).to(DEV) for i in (7, 8))
    k, v = (randn((sum(lk), 2, head_dim), i, dtype).to(DEV) for i in (9, 10))
    kw = dict(softmax_scale=0.1, causal=True)
    out, lse = varlen_forward(q, k, v, cq, ck, 70, 130, return_lse=True, **kw)
    want = varlen_backward(q, k, v, out, do, lse, cq, ck, 70, 130, **kw)
    torch.use_deterministic_algorithms(True)   # empty tensors then hold NaN
    try:
        got = varlen_backward(q, k, v, out, do, lse, cq, ck, 70, 130, covered=True, **kw)
    finally:
        torch.use_deterministic_algorithms(False)
    for a, b in zip(got, want):
        assert torch.equal(a, b)
