"""The decode step's linear layers (``dec_linear``) against float64 products.

Sizes at the edges of the kernel: one k step and uneven k ranges of its waves,
one and several batches of steps, output columns that end inside a tile, one
to sixteen rows, a strided input.  Every output is a few bf16 roundings away
from the float64 result: of the product, of the normalised input (each input
off by 2^-8 at most, in independent directions) and of the last operation.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _norm(x, w, eps):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w


SIZES = [(8, 32), (40, 288), (24, 1024), (6152, 1056), (16, 2048), (48, 2080), (32, 5632), (200, 4128)]


# (the norm's launch of its own takes at most 4096 columns)
@pytest.mark.parametrize("m", [1, 5, 16])
@pytest.mark.parametrize("mode,n,k", [(mode, n, k) for mode in ("plain", "norm", "resid", "glu", "norm_glu")
                                      for n, k in SIZES if k <= 4096 or not mode.startswith("norm")])
def test_dec_linear(gpu, m, mode, n, k):
    from logo_amd.ops.glue import dec_linear

    g = torch.Generator().manual_seed(m * n + k)
    glu = mode.endswith("glu")
    x = torch.randn(m, k + 8, generator=g).bfloat16().to(gpu)[:, :k]  # rows apart by more than k
    w = (torch.randn(2 * n if glu else n, k, generator=g) / k ** 0.5).bfloat16().to(gpu)
    nw = (1 + 0.1 * torch.randn(k, generator=g)).bfloat16().to(gpu) if mode.startswith("norm") else None
    res = torch.randn(m, n, generator=g).bfloat16().to(gpu) if mode == "resid" else None
    got = dec_linear(x, w, norm_w=nw, eps=1e-5, resid=res, glu=glu).double()
    xd = x.double() if nw is None else _norm(x.double(), nw.double(), 1e-5)
    y = xd @ w.double().T
    # rounding of one product: its own, and that of its normalised inputs
    u = 2.0 ** -8
    tol = u * y.abs() + 1e-5
    if nw is not None:
        tol = tol + 6 * 2 * u * (xd.pow(2) @ w.double().T.pow(2)).sqrt()
    if glu:
        ya, yb = y.split(n, dim=1)
        ta, tb = tol.split(n, dim=1)
        s = torch.nn.functional.silu(ya)
        ref = s * yb
        # |silu'| <= 1.1
        tol = (1.1 * ta + u * s.abs()) * (yb.abs() + tb) + (s.abs() + 1.1 * ta) * tb + u * ref.abs() + 1e-5
    else:
        ref = y if res is None else y + res.double()
        tol = tol + u * ref.abs()
    assert got.shape == ref.shape
    assert bool(((got - ref).abs() <= tol).all()), f"max excess {float(((got - ref).abs() - tol).max()):.3e}"


@pytest.mark.parametrize("m,n,k", [(3, 64, 256), (16, 8193, 2048), (12, 8193, 2048), (4, 4097, 2080), (5, 4097, 2080), (1, 40, 4128)])
def test_single_products_on_both_sides_of_the_rule(gpu, m, n, k):
    """On the kernel or the library's product: a bf16 rounding from float64."""
    from logo_amd.layers import linear_rows

    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, 1, k, generator=g).bfloat16().to(gpu)
    lin = torch.nn.Linear(k, n, bias=False).to(device=gpu, dtype=torch.bfloat16)
    with torch.no_grad():
        got = linear_rows(lin, x).double()
    ref = x.double() @ lin.weight.detach().double().T
    assert got.shape == ref.shape
    assert bool(((got - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-5).all())


def test_hooks_and_other_modules_keep_their_calls(gpu):
    """A decode step calls a module that carries a forward hook (or is no plain
    linear layer) as before, with the same logits within bf16 rounding."""
    from logo_amd.layers import LoGoConfig
    from logo_amd.model import LoGoForCausalLM

    cfg = LoGoConfig(vocab_size=256, hidden_size=256, intermediate_size=512, num_hidden_layers=2,
                     num_attention_heads=4, gate_thres_init=-1.0)
    model = LoGoForCausalLM(cfg)
    model.init_weights(torch.Generator().manual_seed(0))
    model = model.to(device=gpu, dtype=torch.bfloat16).eval()
    ids = torch.randint(0, 256, (3, 40), generator=torch.Generator().manual_seed(1)).to(gpu)
    tok = ids[:, 0].clone()
    logits, calls = [], []
    for hooked in (False, True):
        cache = model.new_cache(3, 60, device=gpu)
        model.prefill(ids, cache)
        if hooked:
            for mod in (model.model.layers[0].mlp, model.model.layers[1].self_attn.o_proj, model.lm_head):
                mod.register_forward_hook(lambda *a: calls.append(1))
        logits.append(model.decode_step(tok, cache).double())
    assert len(calls) == 3
    assert float((logits[0] - logits[1]).norm() / logits[1].norm()) <= 2e-2


def _model(gpu, **kw):
    from logo_amd.layers import LoGoConfig
    from logo_amd.model import LoGoForCausalLM

    cfg = LoGoConfig(**{"vocab_size": 256, "hidden_size": 256, "intermediate_size": 512, "num_hidden_layers": 2,
                        "num_attention_heads": 4, "gate_thres_init": -1.0, **kw})
    model = LoGoForCausalLM(cfg)
    model.init_weights(torch.Generator().manual_seed(0))
    return model.to(device=gpu, dtype=torch.bfloat16).eval()


def _step(model, gpu, rows=3):
    ids = torch.randint(0, 256, (rows, 40), generator=torch.Generator().manual_seed(1)).to(gpu)
    cache = model.new_cache(rows, 60, device=gpu)
    model.prefill(ids, cache)
    return model.decode_step(ids[:, 0].clone(), cache)


@pytest.mark.parametrize("where", ["mlp", "self_attn", "o_proj", "down_proj", "lm_head"])
def test_a_forward_set_on_an_instance_is_called(gpu, where):
    """A decode step runs the replacement that a wrapping tool puts on a module,
    as the prefill before it does: here one that doubles the module's output."""
    model = _model(gpu)
    layer = model.model.layers[1]
    mod = {"mlp": layer.mlp, "self_attn": layer.self_attn, "o_proj": layer.self_attn.o_proj,
           "down_proj": layer.mlp.down_proj, "lm_head": model.lm_head}[where]
    want = _step(model, gpu)
    calls, own = [], mod.forward

    def wrapped(*args, **kw):
        calls.append(args[0].shape[1] if args[0].dim() == 3 else 1)
        out = own(*args, **kw)
        return (2 * out[0], *out[1:]) if isinstance(out, tuple) else 2 * out

    mod.forward = wrapped
    got = _step(model, gpu)
    assert 1 in calls, f"{where}: the decode step skipped the replacement"
    if where == "lm_head":
        assert torch.equal(got, 2 * want)
    else:
        assert float((got.double() - want.double()).norm() / want.double().norm()) > 2e-2


class _Scaled(torch.Tensor):
    """A weight whose layer computes something else: linear() doubles its result."""

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        out = super().__torch_function__(func, types, args, kwargs or {})
        return 2 * out.as_subclass(torch.Tensor) if func is torch.nn.functional.linear else out


def test_weights_of_a_tensor_subclass_keep_their_arithmetic(gpu):
    from logo_amd.layers import linear_rows

    lin = torch.nn.Linear(256, 64, bias=False).to(device=gpu, dtype=torch.bfloat16)
    x = torch.randn(2, 256, device=gpu).bfloat16()
    with torch.no_grad():
        want = 2 * torch.nn.functional.linear(x, lin.weight)
        lin.weight = torch.nn.Parameter(lin.weight.detach().as_subclass(_Scaled), requires_grad=False)
        assert torch.equal(linear_rows(lin, x), want)


def test_a_stacked_weight_past_the_kernels_size(gpu):
    """gate and up of 2^29 elements each, which stacked are one more than the
    kernel takes: the step takes the library's product there."""
    from logo_amd.layers import LoGoConfig, rope_cos_sin
    from logo_amd.model import LoGoDecoderLayer
    from logo_amd.ops.decode import LogoKVCache

    cfg = LoGoConfig(hidden_size=4096, num_attention_heads=32, num_key_value_heads=4, num_hidden_layers=1,
                     intermediate_size=131072, gate_thres_init=-1.0)
    with torch.device(gpu):
        torch.manual_seed(0)
        layer = LoGoDecoderLayer(cfg, 0).to(torch.bfloat16).eval()
    cache = LogoKVCache(1, 2, 4, 128, 32, window=128, device=gpu)
    cache.set_length(5)
    h = torch.randn(2, 1, 4096, device=gpu).bfloat16()
    pe = rope_cos_sin(cache.positions(1), 128, cfg.rope_theta, torch.bfloat16)
    with torch.no_grad():
        assert layer._decode_ok(h, cache)
        got = layer._decode_step(h, cache, pe, None).double()
        want = layer(h, past_key_value=cache, position_embeddings=pe).double()
    assert float((got - want).norm() / want.norm()) <= 2e-2
    del layer, cache
    torch.cuda.empty_cache()
