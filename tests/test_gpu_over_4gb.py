"""Head dim 256 and fp32 on both sides of the size at which their kernels change:
with q below 4 GB they run on kernels that address its rows by 32 bits
(logo_amd/csrc/wide_attn.hip, f32_attn.hip), from there on on the generic ones
(gen_attn.hip).  Packed segments of every tile remainder at both ends of the
tensors, GQA, one selection or one per head (one head without rows, one with a
single one), dense rows; the first and the last
segments against the float64 oracle, with the bounds of the kernels' own tests,
and every unselected row zero."""

import numpy as np
import pytest
import torch

from oracle import attn
from tests.helpers import assert_within

pytestmark = pytest.mark.gpu

HQ, H = 32, 4
EDGES = [1, 15, 16, 17, 0, 33, 63, 64, 65, 127, 130, 200]  # a few tokens around every tile size


@pytest.mark.parametrize("side", ["below", "from"])
@pytest.mark.parametrize("dtype,d,rows,per_head", [
    (torch.float32, 64, 0.4, False),
    (torch.float32, 128, 0.4, True),
    (torch.float32, 256, 0.4, False),
    (torch.bfloat16, 256, 0.4, False),
    (torch.bfloat16, 256, None, False),
    (torch.float16, 256, 0.4, True),
])
def test_first_and_last_segments(gpu, side, dtype, d, rows, per_head):
    from logo_amd.ops import dense_causal_attn, sq_full_attn

    limit = 2 ** 32 // (HQ * d * dtype.itemsize)  # tokens at which q is 4 GB
    n = limit - 1 if side == "below" else limit + 37
    left = n - 2 * sum(EDGES)
    lens = EDGES + [250] * (left // 250) + [left % 250] + EDGES[::-1]
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32, device=gpu)
    assert int(cu[-1]) == n and (n * HQ * d * dtype.itemsize < 2 ** 32) == (side == "below")
    g = torch.Generator(device=gpu).manual_seed(d)
    q, k, v, do = (torch.empty(n, x, d, dtype=dtype, device=gpu).normal_(generator=g) for x in (HQ, H, H, HQ))
    sel = None if rows is None else torch.rand((n, HQ) if per_head else (n,), generator=g, device=gpu) < rows
    if per_head:
        sel[:, 1:3] = False
        sel[n - 5, 2] = True
    for x in (q, k, v):
        x.requires_grad_()
    print(f"{side} 4 GB: {dtype} d={d} n={n}", flush=True)
    if sel is None:
        o = dense_causal_attn(q[None], k[None], v[None], cu)[0]
    else:
        o = sq_full_attn(q[None], k[None], v[None], sel[None], cu_seqlens=cu)[0]
    dq, dk, dv = torch.autograd.grad(o, (q, k, v), do)
    span = sum(EDGES)
    for lo, ls in ((0, EDGES), (n - span, EDGES[::-1])):
        part = slice(lo, lo + span)
        qn, kn, vn, dn = (x[part].detach().double().cpu().numpy() for x in (q, k, v, do))
        s = None if sel is None else sel[part].cpu().numpy()
        c = np.concatenate([[0], np.cumsum(ls)]).astype(np.int32)
        ro, _ = attn.sq_attn_fwd(qn, kn, vn, s, c)
        ref = (ro, *attn.sq_attn_bwd(qn, kn, vn, ro, dn, s, c))
        for name, x, r in zip(("o", "dq", "dk", "dv"), (o, dq, dk, dv), ref):
            got, top = x[part].detach(), float(np.abs(r).max())
            if dtype == torch.float32:
                err = np.abs(got.double().cpu().numpy() - r).max()
                assert err <= 1e-5 * max(1.0, top), f"{name} at {lo}: {err:.3e} at scale {top:.2f}"
            else:
                assert_within(f"{name} at {lo}", got, r, max_abs=2e-2 * max(1.0, top / 2))
    if sel is not None:
        for x in (o, dq):
            for t in range(0, n, 65536):  # (in pieces: no mask of the tensor's size)
                assert int(x[t:t + 65536][~sel[t:t + 65536]].count_nonzero()) == 0
    del q, k, v, do, o, dq, dk, dv, x
    torch.cuda.empty_cache()
