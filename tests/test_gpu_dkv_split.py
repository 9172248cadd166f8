"""Row-range split of the dk/dv kernel: key blocks whose query rows (of all the
group's heads) are cut into pieces give dk and dv of the unsplit call up to the
order of the fp32 sums (one bf16 / fp16 rounding of the result), the same bits on
every call, and the oracle's within the kernels' bound; over piece counts, GQA,
per-head rows, packed segments, dense rows, blocks with fewer steps than pieces
and blocks without rows."""

import numpy as np
import pytest
import torch

from oracle import attn
from tests.helpers import assert_within, gen, randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens,hq,h,d,rows,per_head,dtype", [
    ([2500], 4, 1, 64, 0.5, False, torch.bfloat16),
    ([1300, 1, 1200], 8, 2, 128, 0.4, False, torch.bfloat16),
    ([1800], 4, 2, 128, 0.5, True, torch.bfloat16),
    ([3000], 2, 2, 128, 0.6, False, torch.float16),
    ([1500, 700], 4, 2, 64, None, False, torch.bfloat16),
    ([900], 16, 16, 128, 0.9, False, torch.bfloat16),
    ([1000], 8, 4, 64, 0.001, False, torch.bfloat16),
])
def test_split_matches_unsplit(gpu, monkeypatch, lens, hq, h, d, rows, per_head, dtype):
    from logo_amd.ops import dense_causal_attn, sq_full_attn

    n = sum(lens)
    g = gen(1700 + n + hq)
    q, k, v, do = (randn((n, x, d), g, dtype=dtype) for x in (hq, h, h, hq))
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32)
    sel = None if rows is None else torch.rand((n, hq) if per_head else (n,), generator=g) < rows
    got = {}
    for name, env in (("split", "1"), ("again", "1"), ("whole", "0")):
        monkeypatch.setenv("LOGO_SQ_SPLIT", env)
        qg, kg, vg = (x.to(gpu)[None].requires_grad_() for x in (q, k, v))
        if sel is None:
            o = dense_causal_attn(qg, kg, vg, cu.to(gpu))
        else:
            o = sq_full_attn(qg, kg, vg, sel.to(gpu)[None], cu_seqlens=cu.to(gpu))
        o.backward(do.to(gpu)[None])
        got[name] = (kg.grad[0], vg.grad[0])
    qn, kn, vn, dn = (x.double().numpy() for x in (q, k, v, do))
    s = None if sel is None else sel.numpy()
    ro, _ = attn.sq_attn_fwd(qn, kn, vn, s, cu.numpy())
    _, rdk, rdv = attn.sq_attn_bwd(qn, kn, vn, ro, dn, s, cu.numpy())
    for i, (name, r) in enumerate((("dk", rdk), ("dv", rdv))):
        a, b, w = (got[x][i] for x in ("split", "again", "whole"))
        assert torch.equal(a, b), f"{name} differs between two calls"
        assert_within(f"{name} {lens} hq={hq} h={h}", a, r, max_abs=2e-2 * max(1.0, float(np.abs(r).max())))
        # the forward and lse of the two calls may differ by their own split: a
        # few 16-bit roundings of P and of the result
        err = (a.double() - w.double()).norm() / max(float(w.double().norm()), 1e-30)
        assert float(err) <= 4e-3, f"{name}: split against whole {float(err):.2e}"
