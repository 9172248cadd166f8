"""Which modules a decode step does the arithmetic of without calling them (only
those on which nobody has put anything, ``logo_amd.layers._plain``), and which
single products it takes from the library."""

import pytest
import torch.nn as nn

from logo_amd.layers import LoGoAttention, LoGoConfig, RMSNorm, _plain
from logo_amd.model import LoGoDecoderLayer, LoGoMLP
from logo_amd.ops.glue import dec_linear_faster

CFG = LoGoConfig(hidden_size=128, num_attention_heads=2, num_hidden_layers=1, intermediate_size=64)
MAKE = [lambda: nn.Linear(8, 8), lambda: RMSNorm(8), lambda: LoGoMLP(CFG), lambda: LoGoAttention(CFG),
        lambda: LoGoDecoderLayer(CFG, 0)]


@pytest.mark.parametrize("make", MAKE)
def test_what_a_call_would_run_is_not_skipped(make, monkeypatch):
    assert _plain(make(), make())
    m = make()
    m.forward = lambda *a, **kw: None
    assert not _plain(m) and not _plain(make(), m)
    for register in ("register_forward_hook", "register_forward_pre_hook"):
        m = make()
        handle = getattr(m, register)(lambda *a: None)
        assert not _plain(m)
        handle.remove()
        assert _plain(m)
    m = make()
    m.__class__ = type("Other", (type(m),), {"forward": lambda self, *a: None})
    assert not _plain(m)
    m = make()
    monkeypatch.setattr(type(m), "forward", lambda self, *a: None)
    assert not _plain(m)


def test_a_hook_on_every_module():
    handle = nn.modules.module.register_module_forward_hook(lambda *a: None)
    try:
        assert not _plain(nn.Linear(8, 8))
    finally:
        handle.remove()
    assert _plain(nn.Linear(8, 8))


@pytest.mark.parametrize("n,k,most_rows", [
    (6152, 2048, 16), (2048, 2048, 16), (32000, 2048, 12), (32000, 1024, 16), (32000, 1536, 16),  # by themselves
    (8192, 2048, 16), (8193, 2048, 12), (65537, 1024, 10), (128256, 512, 10),
    (4096, 2080, 16), (4097, 2080, 4), (4096, 4096, 16), (128256, 4096, 4), (4096, 4128, 0), (32000, 5120, 0),
])
def test_the_single_products_that_dec_linear_takes(n, k, most_rows):
    """The lines of the measured rule: up to ``most_rows`` rows, and no more."""
    assert [m for m in range(1, 17) if dec_linear_faster(m, n, k)] == list(range(1, most_rows + 1))
