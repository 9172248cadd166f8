"""The one-launch prompt store of LogoKVCache against its row copies: prompts
below, at and above the ring, 64-token blocks and one past, both head dims, and
the layouts that stay on the copies."""

import pytest
import torch

from logo_amd.ops.decode import LogoKVCache

pytestmark = pytest.mark.gpu


def _cache(B, H, D, T, dtype=torch.bfloat16, window=128):
    c = LogoKVCache(2, B, H, D, T + 7, window=window, dtype=dtype, device="cuda")
    for ts in (c.local_k, c.local_v, c.global_k, c.global_v):
        for t in ts:
            t.fill_(-3.0)
    return c


def _all(c):
    return [*c.local_k, *c.local_v, *c.global_k, *c.global_v]


@pytest.mark.parametrize("B,H,D,T,window,dtype", [
    (1, 1, 128, 1, 128, torch.bfloat16), (2, 3, 64, 64, 128, torch.bfloat16), (2, 2, 128, 129, 128, torch.bfloat16),
    (1, 4, 128, 130, 128, torch.float16), (3, 2, 64, 1000, 0, torch.bfloat16), (2, 16, 128, 3001, 128, torch.bfloat16)])
def test_store_is_the_row_copies(gpu, B, H, D, T, window, dtype):
    g = torch.Generator().manual_seed(T)
    rows = [torch.randn(B, T, H, D, generator=g).to(dtype).cuda().transpose(1, 2) for _ in range(4)]
    a, b = _cache(B, H, D, T, dtype, window), _cache(B, H, D, T, dtype, window)
    assert a._store_fused(1, *rows)
    b._store_rows(1, slice(None), *rows)
    for x, y in zip(_all(a), _all(b)):
        assert torch.equal(x, y)
    c = _cache(B, H, D, T, dtype, window)
    c.prefill(1, *rows)
    for x, y in zip(_all(c), _all(b)):
        assert torch.equal(x, y)


def test_other_layouts_stay_on_the_copies(gpu):
    rows = [torch.randn(2, 70, 2, 64, device="cuda").bfloat16().transpose(1, 2) for _ in range(4)]
    c = _cache(2, 2, 64, 70)
    assert not c._store_fused(0, *(r.contiguous() for r in rows))   # head-major rows
    assert not c._store_fused(0, *(r.float() for r in rows))        # another type than the cache's
    assert not c._store_fused(0, rows[0].clone().requires_grad_(), *rows[1:])
    ref = _cache(2, 2, 64, 70)
    ref.prefill(0, *rows)
    c.prefill(0, *(r.contiguous() for r in rows))
    for x, y in zip(_all(c), _all(ref)):
        assert torch.equal(x, y)
