"""An output whose gradient autograd leaves undefined (the function that consumed it returned None for it): q, k and v
still get gradients, of zeros.  The kernels are replaced by torch stand-ins, so this runs without a GPU."""
import pytest
import torch

from flash_attn_triton.triton_kernel import attention_kernel as ak


class _NoGradient(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x):
        return x * 2

    @staticmethod
    def backward(ctx, g):
        return None


@pytest.mark.parametrize("varlen", [False, True])
@pytest.mark.parametrize("passed", [False, True])
def test_undefined_output_gradient(monkeypatch, varlen, passed):
    def forward(q, k, v, *cu, **kw):
        return q + k + v, torch.zeros(q.shape[:-1])

    def backward(q, k, v, out, dout, lse, *cu, **kw):
        return dout * q, dout * k, dout * v

    kind = "varlen" if varlen else "dense"
    monkeypatch.setattr(ak, f"{kind}_forward", forward)
    monkeypatch.setattr(ak, f"{kind}_backward", backward)
    shape = (5, 2, 16) if varlen else (1, 5, 2, 16)
    q, k, v = (torch.randn(shape, generator=torch.Generator().manual_seed(i)).requires_grad_() for i in range(3))
    cu = torch.tensor([0, 5], dtype=torch.int32)
    out = (ak.varlen_attention(q, k, v, cu, cu, 5, 5, softmax_scale=1.0, causal=False) if varlen
           else ak.dense_attention(q, k, v, softmax_scale=1.0, causal=False))
    (out if passed else _NoGradient.apply(out)).sum().backward()
    for t in (q, k, v):
        assert torch.equal(t.grad, t.detach() if passed else torch.zeros_like(t))
