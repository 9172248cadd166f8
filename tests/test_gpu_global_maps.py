"""The fused global maps + RoPE launches against the kernels they stand for, at
the edges of their token passes (128), partial weight gradients (1024) and runs."""

import pytest
import torch

from logo_amd.layers import rope_cos_sin
from logo_amd.ops.glue import (_aligned16, _global_maps_launch, _head_linear_dw, _head_linear_launch, _rope_launch,
                               attn_inputs, global_maps_, global_maps_ok, head_linear_grad_acc)

pytestmark = pytest.mark.gpu


def _inputs(n, H, HK, D, seed):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g).bfloat16().cuda()  # noqa: E731
    xs = [r(1, n, h, D) for h in (H, HK, HK)]
    ws = [(torch.eye(D).cuda() + 0.05 * r(h, D, D)).bfloat16() for h in (H, HK, HK)]
    cos, sin = rope_cos_sin(torch.randint(0, 9000, (1, n), generator=g).cuda(), D, 10000.0, torch.bfloat16)
    return xs, ws, cos, sin, r


# fewer tokens than a pass, whole passes, one more, several runs with a ragged last one
@pytest.mark.parametrize("n,H,HK,D", [(1, 2, 1, 128), (127, 4, 4, 128), (128, 3, 1, 64), (129, 16, 4, 128),
                                      (1025, 8, 2, 64), (6001, 16, 16, 128)])
def test_forward_is_the_chain(gpu, n, H, HK, D):
    xs, ws, cos, sin, _ = _inputs(n, H, HK, D, n)
    gs = [_head_linear_launch(x, w, False) for x, w in zip(xs, ws)]
    ref = _rope_launch([xs[0], xs[1], gs[0], gs[1]], cos, sin, n, D, inverse=False)
    ref = (ref[0], ref[1], xs[2], ref[2], ref[3], gs[2])
    out = _global_maps_launch(xs, ws, cos, sin, inplace=False)
    for a, b in zip(out, ref):
        assert torch.equal(a, b)
    out = global_maps_(xs[0].clone(), xs[1].clone(), xs[2], ws, cos, sin)
    for a, b in zip(out, ref):
        assert torch.equal(a, b)


@pytest.mark.parametrize("n,H,HK", [(65, 2, 1), (128, 3, 3), (1024, 4, 2), (1153, 16, 4), (9217, 8, 8), (33000, 16, 16)])
def test_backward_is_the_chain(gpu, n, H, HK):
    """attn_inputs' gradients of the maps and, through an identity projection,
    of q, k and v: bit-identical to the separate kernels."""
    D = 128
    xs, ws, cos, sin, r = _inputs(n, H, HK, D, n)
    xs = [x * 0.5 for x in xs]
    grads = [r(1, n, h, D) for h in (H, HK, HK, H, HK, HK)]
    # the node's own launch, with its dx in the columns of one wider buffer
    from logo_amd import _lib
    lib = _lib.lib()
    cols = (H * D, HK * D, HK * D, 8)
    dy = torch.full((n, sum(cols)), 7.0, dtype=torch.bfloat16, device="cuda")
    outs = dy.split(cols, dim=1)
    wsp = torch.empty(lib.logo_head_linear_dw_workspace_bytes(n, H + 2 * HK, D) // 4, device="cuda")
    dws = [torch.empty_like(w) for w in ws]
    for with_dw in ((True, True, True), (True, False, True)):
        args = []
        for i in range(3):
            args += [_lib.ptr(xs[i]), _lib.ptr(ws[i]), _lib.ptr(grads[i]), _lib.ptr(grads[3 + i]), _lib.ptr(outs[i]),
                     _lib.ptr(dws[i]) if with_dw[i] else None, (H, HK, HK)[i], int(i < 2)]
        rc = lib.logo_global_maps_bwd(*args, _lib.ptr(cos), _lib.ptr(sin), dy.stride(0), _lib.ptr(wsp), n, D,
                                      _lib.DTYPE_BF16, _lib.stream_of(dy))
        assert rc == 0
        dqa, dka, dgq, dgk = _rope_launch([grads[0], grads[1], grads[3], grads[4]], cos, sin, n, D, inverse=True)
        for i, (a, g) in enumerate(((dqa, dgq), (dka, dgk), (grads[2], grads[5]))):
            nh = a.shape[-2]
            ref = torch.empty(n, nh, D, dtype=torch.bfloat16, device="cuda")
            head_linear_grad_acc(g.view(n, nh, D), ws[i], a.view(n, nh, D), ref)
            assert torch.equal(outs[i], ref.view(n, -1))
            if with_dw[i]:
                assert torch.equal(dws[i], _head_linear_dw(xs[i], g))
        assert (outs[3] == 7.0).all()


def test_layouts_that_are_not_the_kernels(gpu):
    """Misaligned or strided operands are refused by the rule (the layer then
    takes its separate steps); attn_inputs copies them."""
    xs, ws, cos, sin, _ = _inputs(130, 2, 2, 128, 3)
    assert global_maps_ok(*xs, ws, cos, sin)
    buf = torch.empty(xs[0].numel() + 4, dtype=torch.bfloat16, device="cuda")
    off = buf[4:].view(xs[0].shape)
    off.copy_(xs[0])
    assert not global_maps_ok(off, xs[1], xs[2], ws, cos, sin)
    assert not global_maps_ok(xs[0].transpose(0, 1), xs[1], xs[2], ws, cos, sin)
    assert not global_maps_ok(*xs, ws, cos[:, :64], sin)
    with pytest.raises(ValueError):
        global_maps_(off, xs[1], xs[2], ws, cos, sin)
    lin = [torch.nn.Linear(256, k, bias=False).cuda().bfloat16() for k in (256, 256, 256, 1)]
    h = torch.randn(1, 130, 256, device="cuda").bfloat16()
    ref = attn_inputs(h, *lin, ws, cos, sin, 2, 2)
    shifted = [torch.cat([t.new_zeros(4), t.flatten()])[4:].view(t.shape) for t in (cos, sin)]
    assert shifted[0].data_ptr() % 16 and _aligned16(shifted[0]).data_ptr() % 16 == 0
    for a, b in zip(attn_inputs(h, *lin, ws, *shifted, 2, 2), ref):
        assert torch.equal(a, b)


def test_no_tokens_are_refused(gpu):
    """An empty batch is an error, not uninitialised weight gradients."""
    _, ws, _, _, _ = _inputs(1, 2, 2, 128, 4)
    lin = [torch.nn.Linear(256, k, bias=False).cuda().bfloat16() for k in (256, 256, 256, 1)]
    h = torch.empty(1, 0, 256, dtype=torch.bfloat16, device="cuda")
    cos = torch.empty(1, 0, 128, dtype=torch.bfloat16, device="cuda")
    with pytest.raises(RuntimeError, match="n_tokens"):
        attn_inputs(h, *lin, [w.requires_grad_() for w in ws], cos, cos.clone(), 2, 2)
