"""Which modules a decode step does the arithmetic of without calling them: only
those on which nobody has put anything (``logo_amd.layers._plain``)."""

import pytest
import torch.nn as nn

from logo_amd.layers import LoGoAttention, LoGoConfig, RMSNorm, _plain
from logo_amd.model import LoGoDecoderLayer, LoGoMLP

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
