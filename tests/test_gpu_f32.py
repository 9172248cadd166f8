"""fp32 attention (logo_amd/csrc/f32_attn.hip) at the edges of its tiles and in
every split of a workgroup's eight waves: 16-key tiles and 16-row steps, rows
and keys that end inside a tile, key and row groups without work, GQA, per-head
rows, packed and empty segments; and the sizes at which the number of row waves
(keys: wave pairs) changes.  Against the float64 oracle fed the same fp32
values; the products and sums are fp32, so an output of magnitude m over sums of
up to n terms is off by a few n^0.5 2^-24 m (1e-5 relative covers n = 4096 with
room; the tile edges see smaller sums).
"""

import numpy as np
import pytest
import torch

from oracle import attn
from tests.helpers import gen

pytestmark = pytest.mark.gpu


def _check(gpu, lens, hq, h, d, rows, per_head=False):
    from logo_amd.ops import sq_full_attn

    n = sum(lens)
    g = gen(1500 + n + hq + d)
    q, k, v, do = (torch.randn(n, x, d, generator=g) for x in (hq, h, h, hq))
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32)
    sel = torch.rand((n, hq) if per_head else (n,), generator=g) < rows
    qg, kg, vg = (x.to(gpu)[None].requires_grad_() for x in (q, k, v))
    o = sq_full_attn(qg, kg, vg, sel.to(gpu)[None], cu_seqlens=cu.to(gpu))
    o.backward(do.to(gpu)[None])
    qn, kn, vn, dn = (x.double().numpy() for x in (q, k, v, do))
    ro, _ = attn.sq_attn_fwd(qn, kn, vn, sel.numpy(), cu.numpy())
    rdq, rdk, rdv = attn.sq_attn_bwd(qn, kn, vn, ro, dn, sel.numpy(), cu.numpy())
    for name, x, r in (("o", o, ro), ("dq", qg.grad, rdq), ("dk", kg.grad, rdk), ("dv", vg.grad, rdv)):
        got = x[0].detach().double().cpu().numpy()
        scale = max(1.0, float(np.abs(r).max()))
        assert np.abs(got - r).max() <= 1e-5 * scale, f"{name}: {np.abs(got - r).max():.3e} at scale {scale:.2f}"
    if not per_head:
        assert torch.all(o[0][~sel.to(gpu)] == 0) and torch.all(qg.grad[0][~sel.to(gpu)] == 0)


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("lens", [[1], [15], [16], [17, 0, 33], [127], [129, 16], [300]])
def test_tile_edges_every_row_selected(gpu, lens, d):
    _check(gpu, lens, 2, 1, d, 1.1)


@pytest.mark.parametrize("lens,hq,h,d,rows,per_head", [
    ([900], 4, 2, 64, 0.3, True),
    ([700, 1, 350], 2, 2, 128, 0.1, False),
    ([600], 4, 1, 256, 0.5, False),
    ([2100], 16, 16, 64, 0.02, False),    # 2 row waves, 2 pairs
    ([3300], 16, 16, 64, 0.02, False),    # 4 row waves, 4 pairs
    ([4200], 16, 16, 128, 0.01, False),   # 4 pairs
    ([6200], 16, 4, 128, 0.01, False),    # 4 row waves
])
def test_waves_of_a_workgroup(gpu, lens, hq, h, d, rows, per_head):
    _check(gpu, lens, hq, h, d, rows, per_head)


@pytest.mark.parametrize("d", [64, 128, 256])
def test_probabilities_below_the_normal_range_count(gpu, d):
    """Key 0 has probability 2^-131 to 2^-135 in every later row, a subnormal fp32
    number, and dO v_0 = 2^60: its share of dq and all of dk_0 come from their
    product, which fp32 holds.  A subnormal of 15 bits or more and scores of 135
    with a few 2^-24 of relative error leave 1e-4."""
    from logo_amd.ops import sq_full_attn

    n = 40
    q, k, v, do = (torch.zeros(n, 2, d) for _ in range(4))
    q[:, :, 0] = 8.0
    k[0, :, 0] = -130.0 / 8.0
    v[0, :, 1] = 2.0 ** 30
    do[1:, :, 1] = 2.0 ** 30
    do[:, :, 2] = torch.randn(n, 2, generator=gen(5))
    v[1:, :, 2] = torch.randn(n - 1, 2, generator=gen(6))
    scale = float(np.log(2.0))  # scores in the log2 domain: 8 times k_0
    sel = torch.ones(n, dtype=torch.bool)
    cu = torch.tensor([0, n], dtype=torch.int32)
    qg, kg, vg = (x.to(gpu)[None].requires_grad_() for x in (q, k, v))
    o = sq_full_attn(qg, kg, vg, sel.to(gpu)[None], cu_seqlens=cu.to(gpu), scale=scale)
    _, dk, dv = torch.autograd.grad(o, (qg, kg, vg), do.to(gpu)[None])
    qn, kn, vn, dn = (x.double().numpy() for x in (q, k, v, do))
    ro, _ = attn.sq_attn_fwd(qn, kn, vn, sel.numpy(), cu.numpy(), scale=scale)
    _, rdk, rdv = attn.sq_attn_bwd(qn, kn, vn, ro, dn, sel.numpy(), cu.numpy(), scale=scale)
    want = rdk[0, :, 0]
    assert 0 < np.abs(want).max() < 2.0 ** -50
    got = dk[0, 0, :, 0].double().cpu().numpy()
    assert np.abs(got - want).max() <= 1e-4 * np.abs(want).max(), (got, want)
