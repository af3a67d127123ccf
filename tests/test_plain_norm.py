"""Which norms the decode runner may replace by its fused kernel (`decode_step.plain_norm`)."""

from __future__ import annotations

import pytest
import torch
from torch import nn
from transformers.models.llama.modeling_llama import LlamaRMSNorm


def _norm(cls=LlamaRMSNorm):
    return cls(32).to(torch.bfloat16)


@pytest.fixture
def plain(pkg):
    from llm_serving_engine_amd.decode_step import plain_norm

    return plain_norm


def test_a_plain_norm(plain):
    assert plain(_norm())


def test_namesakes_and_subclasses(plain):
    sub = type("LlamaRMSNorm", (LlamaRMSNorm,), {"forward": lambda self, x: x})
    assert not plain(_norm(sub))
    assert not plain(_norm(type("Norm", (LlamaRMSNorm,), {})))
    assert not plain(nn.LayerNorm(32, dtype=torch.bfloat16))


def test_replaced_forwards(plain, monkeypatch):
    norm = _norm()
    norm.forward = lambda x: x
    assert not plain(norm)
    norm = _norm()
    monkeypatch.setattr(LlamaRMSNorm, "forward", lambda self, x: x)
    assert not plain(norm)


def test_hooks(plain):
    for register in ("register_forward_hook", "register_forward_pre_hook"):
        norm = _norm()
        handle = getattr(norm, register)(lambda *a: None)
        assert not plain(norm)
        handle.remove()
        assert plain(norm)
    for register in ("register_module_forward_hook", "register_module_forward_pre_hook"):
        handle = getattr(nn.modules.module, register)(lambda *a: None)
        try:
            assert not plain(_norm())
        finally:
            handle.remove()
    assert plain(_norm())


def test_weights_and_eps(plain):
    assert not plain(LlamaRMSNorm(32))  # fp32
    assert not plain(LlamaRMSNorm(32, eps=-1e-5).to(torch.bfloat16))
    swapped = nn.utils.parametrizations.weight_norm(_norm(), "weight", dim=None)
    assert not plain(swapped)
