"""Which decoders run as one native call over all layers (_native_layers_for),
decided on the host. The plans are built from CPU weights here: the one check
that asks for GPU weights is stubbed."""

from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch
from transformers import LlamaConfig, LlamaForCausalLM, Qwen3Config, Qwen3ForCausalLM

from kv_cache_repair_amd.kernels import packed_cache as pc


@pytest.fixture
def base(monkeypatch, request):
    monkeypatch.setattr(pc._projection, "supported_weight", lambda weight: weight.ndim == 2)
    family = getattr(request, "param", "llama")
    kw = dict(vocab_size=32, hidden_size=64, intermediate_size=128, num_hidden_layers=3, num_attention_heads=4,
              num_key_value_heads=2, head_dim=16)
    config, ctor = (LlamaConfig, LlamaForCausalLM) if family == "llama" else (Qwen3Config, Qwen3ForCausalLM)
    torch.manual_seed(0)
    return ctor(config(**kw)).to(torch.bfloat16).eval().model


def resize(layer, name, rows, cols):
    parent = layer.mlp if name in ("gate_proj", "up_proj", "down_proj") else layer.self_attn
    setattr(parent, name, torch.nn.Linear(cols, rows, bias=False, dtype=torch.bfloat16).eval())


def native(base, heads=(4, 2, 16)):
    launcher = SimpleNamespace(q_heads=heads[0], kv_heads=heads[1], head_dim=heads[2])
    return pc._native_layers_for(None, base, pc._model_plans(base), True, True, launcher)


@pytest.mark.parametrize("base", ["llama", "qwen3"], indirect=True)
def test_layers_of_one_geometry_run_natively(base):
    assert native(base)
    assert not native(base, heads=(2, 2, 16)) and not native(base, heads=(4, 1, 16)) and not native(base, heads=(8, 4, 8))


@pytest.mark.parametrize("narrow", [0, 1, 2])
def test_layers_of_several_widths_run_as_modules(base, narrow):
    """One refresh descriptor holds the shapes of all layers: a narrower MLP would be
    read past its weights."""
    for name, rows, cols in (("gate_proj", 96, 64), ("up_proj", 96, 64), ("down_proj", 64, 96)):
        resize(base.layers[narrow], name, rows, cols)
    assert not native(base)
    for layer in base.layers:
        for name, rows, cols in (("gate_proj", 96, 64), ("up_proj", 96, 64), ("down_proj", 64, 96)):
            resize(layer, name, rows, cols)
    assert native(base)


@pytest.mark.parametrize("change", [("q_proj", 48, 64), ("o_proj", 64, 48), ("k_proj", 16, 64), ("v_proj", 16, 64),
                                    ("o_proj", 56, 64), ("down_proj", 56, 128), ("down_proj", 64, 120)])
def test_weights_that_do_not_chain_run_as_modules(base, change):
    resize(base.layers[1], *change)
    assert not native(base)
