"""dq and dk/dv of one call beside each other on one split workspace: what they
write of it (arrival counters, fp32 partials) lies apart, and on two streams they
give the bits of the two calls in a row.  Shapes: both split, grouped heads, a
short sequence with one kv head, and one whose key blocks are too many to be cut."""

import pytest
import torch

from logo_amd import _lib
from logo_amd.ops.common import compact_selection
from tests.helpers import gen, randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,hq,h,d,cu,dkv_splits", [
    (6001, 16, 4, 64, [0, 6001], True),
    (4000, 8, 2, 128, [0, 1300, 1301, 4000], True),
    (2000, 8, 1, 128, [0, 2000], True),
    (9000, 16, 16, 128, [0, 9000], False),
])
def test_dq_and_dkv_share_a_workspace(gpu, n, hq, h, d, cu, dkv_splits):
    lib = _lib.lib()
    g = gen(1900 + n)
    q, k, v, do = (randn((n, x, d), g).to(gpu) for x in (hq, h, h, hq))
    cu = torch.tensor(cu, dtype=torch.int32, device=gpu)
    ds = compact_selection((torch.rand(n, generator=g) < 0.6).to(gpu), cu)
    nseq, scale = cu.numel() - 1, d ** -0.5
    nbytes, cnt = lib.logo_sq_workspace_bytes(n, nseq, hq, d), lib.logo_sq_workspace_counter_bytes()
    assert lib.logo_sq_kv_workspace_bytes(n, nseq, hq, h, d) <= nbytes
    ws = torch.zeros(nbytes, dtype=torch.uint8, device=gpu)
    o, dq = torch.empty_like(q), torch.empty_like(q)
    dk, dv = torch.empty_like(k), torch.empty_like(v)
    lse, delta = (torch.empty(hq, n, device=gpu) for _ in range(2))
    q_sel, do_sel = (torch.empty(hq, n, d, dtype=q.dtype, device=gpu) for _ in range(2))
    tail = [_lib.ptr(x) for x in (ds.q_idx, ds.pos, ds.meta, cu)] + [n, nseq, hq, h, d, d, 1, scale, -1,
                                                                    _lib.DTYPE_BF16, _lib.ptr(ws), nbytes]
    args = [_lib.ptr(x) for x in (q, k, v, o, do, lse, delta, q_sel, do_sel, dq, dk, dv)] + tail
    main = _lib.stream_of(q)
    assert lib.logo_sq_fwd(*[_lib.ptr(x) for x in (q, k, v, o, lse)], *tail, main) == 0
    assert lib.logo_sq_bwd_delta(*args, main) == 0

    def written(fn):
        """The bytes of the workspace's partials that a call changes."""
        touched = torch.zeros(nbytes, dtype=torch.bool, device=gpu)
        for fill in (0xA5, 0x5A):
            ws[cnt:] = fill
            assert fn(*args, main) == 0
            touched |= ws != fill
        assert int(ws[:cnt].count_nonzero()) == 0
        return touched[cnt:]

    by_dq, by_dkv = written(lib.logo_sq_bwd_dq), written(lib.logo_sq_bwd_dkv)
    assert bool(by_dkv.any()) == dkv_splits
    assert not bool((by_dq & by_dkv).any()), "dq and dk/dv write the same partials"

    want = [x.clone() for x in (dq, dk, dv)]
    side = torch.cuda.Stream()
    for _ in range(3):
        for x in (dq, dk, dv):
            x.fill_(7.0)
        side.wait_stream(torch.cuda.current_stream())
        assert lib.logo_sq_bwd_dkv(*args, _lib.ctypes.c_void_p(side.cuda_stream)) == 0
        assert lib.logo_sq_bwd_dq(*args, main) == 0
        torch.cuda.current_stream().wait_stream(side)
        assert all(torch.equal(a, b) for a, b in zip((dq, dk, dv), want))
    assert int(ws[:cnt].count_nonzero()) == 0


@pytest.mark.parametrize("n,hq,h,d,rows,per_head,splits", [
    # fewer key blocks than half the CUs: from 6 steps of 128 rows on
    (4000, 4, 2, 64, 0.05, False, False),
    (2000, 16, 4, 128, 0.25, False, True),
    (2000, 16, 4, 64, 0.25, True, True),
    # up to one a CU: from 20 steps on
    (4000, 16, 8, 64, 0.2, False, False),
    (4000, 16, 8, 64, 0.4, False, True),
    (6000, 16, 4, 128, 0.05, True, False),
    # more: from 32, then 144 steps on
    (9000, 16, 4, 64, 0.08, False, False),
    (9000, 16, 4, 64, 0.4, False, True),
    (6000, 32, 8, 64, 0.4, False, False),
    (6000, 32, 8, 64, 0.9, False, True),
    # no choice of rows gives the steps
    (1000, 4, 4, 64, 0.6, False, False),
    (1100, 16, 16, 64, 1.1, False, False),
])
def test_key_blocks_of_few_steps_stay_whole(gpu, n, hq, h, d, rows, per_head, splits):
    """dk/dv cuts a key block (and writes partials) only where its steps pay for
    the pieces; cut or whole, the same gradients to a few roundings."""
    lib = _lib.lib()
    g = gen(2000 + n + hq)
    q, k, v, do = (randn((n, x, d), g).to(gpu) for x in (hq, h, h, hq))
    cu = torch.tensor([0, n], dtype=torch.int32, device=gpu)
    ds = compact_selection((torch.rand((n, hq) if per_head else (n,), generator=g) < rows).to(gpu), cu)
    scale, cnt = d ** -0.5, lib.logo_sq_workspace_counter_bytes()
    nbytes = lib.logo_sq_kv_workspace_bytes(n, 1, hq, h, d)
    ws = torch.zeros(nbytes, dtype=torch.uint8, device=gpu)
    o, dq = torch.empty_like(q), torch.empty_like(q)
    lse, delta = (torch.empty(hq, n, device=gpu) for _ in range(2))
    q_sel, do_sel = (torch.empty(hq, n, d, dtype=q.dtype, device=gpu) for _ in range(2))
    out = []
    for size in (0, nbytes):
        tail = [_lib.ptr(x) for x in (ds.q_idx, ds.pos, ds.meta, cu)] + [
            n, 1, hq, h, d, d, ds.lanes, scale, -1, _lib.DTYPE_BF16, _lib.ptr(ws) if size else None, size,
            _lib.stream_of(q)]
        dk, dv = torch.full_like(k, 7.0), torch.full_like(v, 7.0)
        if not out:
            assert lib.logo_sq_fwd(*[_lib.ptr(x) for x in (q, k, v, o, lse)], *tail) == 0
        args = [_lib.ptr(x) for x in (q, k, v, o, do, lse, delta, q_sel, do_sel, dq, dk, dv)] + tail
        assert lib.logo_sq_bwd_delta(*args) == 0
        ws[cnt:] = 0xA5
        assert lib.logo_sq_bwd_dkv(*args) == 0
        out.append((dk, dv))
    assert bool((ws[cnt:] != 0xA5).any()) == splits
    assert int(ws[:cnt].count_nonzero()) == 0
    for a, b in zip(*out):
        # the order of the fp32 sums, then one bf16 rounding
        assert float((a.double() - b.double()).norm()) <= 2.0 ** -8 * float(b.double().norm())
        assert splits or torch.equal(a, b)
