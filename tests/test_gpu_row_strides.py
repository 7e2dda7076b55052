"""Query rows further apart than 32-bit byte offsets reach (40 rows, 256 MiB from one to the next): dense, varlen, paged
varlen and KV-cache calls against the same call on contiguous queries."""
import pytest
import torch

from _helpers import ATOL, randn

pytestmark = pytest.mark.gpu

DEV = "cuda"
ROWS, STRIDE, PAGE = 40, 1 << 27, 16


def _far(x):
    """x [ROWS, H, D] with its rows STRIDE elements apart."""
    h, d = x.shape[1:]
    far = torch.empty((ROWS - 1) * STRIDE + h * d, dtype=x.dtype, device=DEV).as_strided((ROWS, h, d), (STRIDE, d, 1))
    return far.copy_(x)


@pytest.mark.parametrize("kind,head_dim", [("dense", 64), ("varlen", 64), ("paged", 64), ("paged", 128), ("cache", 64),
                                           ("cache", 128)])
def test_far_query_rows(kind, head_dim):
    from flash_attn_triton import flash_attn_func, flash_attn_varlen_func, flash_attn_with_kvcache
    keys, h = 80, 2
    q = randn((ROWS, h, head_dim), 1).to(DEV)
    if kind in ("paged", "cache"):
        k, v = (randn((keys // PAGE, PAGE, h, head_dim), i).to(DEV) for i in (2, 3))
    else:
        k, v = (randn((keys, h, head_dim), i).to(DEV) for i in (2, 3))
    cu_q, cu_k = (torch.tensor([0, n], dtype=torch.int32, device=DEV) for n in (ROWS, keys))
    table = torch.tensor([[3, 0, 4, 1, 2]], dtype=torch.int32, device=DEV)

    def call(q):
        if kind == "dense":
            return flash_attn_func(q[None], k[None], v[None])[0]
        if kind == "cache":
            return flash_attn_with_kvcache(q[None], k, v, cache_seqlens=cu_k[1:], block_table=table)[0]
        return flash_attn_varlen_func(q, k, v, cu_q, cu_k, ROWS, keys, causal=True,
                                      block_table=table if kind == "paged" else None)

    near, far = call(q), call(_far(q))
    # two kernels, each within the fp16 bar of the exact result
    assert (near.float() - far.float()).abs().max().item() <= 2 * ATOL[torch.float16]
