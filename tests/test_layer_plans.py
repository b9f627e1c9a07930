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


def constants(layers):
    out = []
    for layer in layers:
        attn, mlp = layer.self_attn, layer.mlp
        out += [getattr(getattr(m, name, None), "variance_epsilon", None)
                for m, name in ((layer, "input_layernorm"), (layer, "post_attention_layernorm"), (attn, "q_norm"),
                                (attn, "k_norm"))]
        act = getattr(mlp, "act_fn", None)
        out += [getattr(attn, "head_dim", None), None if act is None else type(act)]
    return tuple(out)


@pytest.mark.parametrize("base", ["llama", "qwen3"], indirect=True)
def test_layer_constants_match_the_attribute_reads(base):
    walk = pc._module_walk()
    assert walk.layer_constants(base.layers) == constants(base.layers)
    base.layers[1].mlp.act_fn = torch.nn.GELU()
    base.layers[2].input_layernorm.variance_epsilon = 0.25
    base.layers[0].self_attn.head_dim = 3
    assert walk.layer_constants(list(base.layers)) == constants(base.layers)
    base.layers[0].mlp = torch.nn.Identity()
    del base.layers[1].input_layernorm.variance_epsilon
    assert walk.layer_constants(base.layers) == constants(base.layers)
    assert walk.layer_constants([]) == ()
    with pytest.raises(TypeError):
        walk.layer_constants(3)
    with pytest.raises(AttributeError):
        walk.layer_constants([object()])


def test_layout_key_tells_every_view_of_a_storage_apart():
    from kv_cache_repair_amd.kernels.executor import tensor_layout

    key = tensor_layout().layout_key
    w = torch.randn(6, 6)
    views = [w, w[:4], w[:, :4], w.t(), w[:4, :4], w.view(36), w.view(2, 3, 2, 3, 1), w.view(torch.int32), w[1:],
             w[:, 1:], torch.randn(6, 6)]
    assert len({key(v) for v in views}) == len(views)
    assert key(w.view(6, 6)) == key(w) == key(torch.nn.Parameter(w, requires_grad=False))
    with pytest.raises(TypeError, match="expected a tensor"):
        key(None)


@pytest.mark.parametrize("change", ["epsilon", "activation", "rows", "stride"])
def test_plans_follow_what_changes_on_the_same_modules(base, change):
    """The modules, parameters and addresses stay: only a constant, the activation or
    a weight's view is set anew."""
    layer = base.layers[1]
    first = pc._layer_plans(layer)
    assert pc._layer_plans(layer) is first
    mlp = layer.mlp
    if change == "epsilon":
        layer.post_attention_layernorm.variance_epsilon = 0.5
        assert pc._layer_plans(layer).desc.eps_post == 0.5
    elif change == "activation":
        mlp.act_fn = torch.nn.GELU()
        assert pc._layer_plans(layer) is None
    elif change == "rows":
        for proj in (mlp.gate_proj, mlp.up_proj):
            proj.weight.data = proj.weight.data[:64]
        mlp.down_proj.weight.data = mlp.down_proj.weight.data[:, :64]
        plans = pc._layer_plans(layer)
        assert plans.gate_up.n_out == plans.down.k == 64 and plans.desc.ld_down == 128
        assert not native(base)
    else:
        proj = layer.self_attn.q_proj
        proj.weight.data = proj.weight.data.as_strided((64, 64), (32, 1))
        assert pc._layer_plans(layer).desc.ld_q == 32


@pytest.mark.parametrize("hidden,rows,tiled", [(64, 4096, True), (64, 64, False), (64, 65, True), (8192, 4095, True),
                                               (8192, 4096, False), (8192, 65, True), (8192, 15104, False),
                                               (8128, 15104, True), (64, 1 << 20, True), (64, (1 << 20) + 1, False)])
def test_rows_and_widths_that_run_tiled(monkeypatch, hidden, rows, tiled):
    monkeypatch.setattr(pc._projection, "supported_weight", lambda weight: weight.ndim == 2)
    base = LlamaForCausalLM(LlamaConfig(vocab_size=32, hidden_size=hidden, intermediate_size=128, num_hidden_layers=2,
                                        num_attention_heads=4, num_key_value_heads=2, head_dim=16)).to(torch.bfloat16)
    launcher = SimpleNamespace(q_heads=4, kv_heads=2, head_dim=16, n_sel=rows, dtype_code=2)
    found = pc._tiled_plans_for(base.model, launcher, None, None, True, True)
    assert (found is not None) == tiled


class TwoMatrixMlp(torch.nn.Module):
    """A decoder MLP of another form: the packed layer runs it as it is."""

    def __init__(self, hidden, inner, dtype, device=None):
        super().__init__()
        self.fc1 = torch.nn.Linear(hidden, inner, dtype=dtype, device=device)
        self.fc2 = torch.nn.Linear(inner, hidden, dtype=dtype, device=device)
        self.act_fn = torch.nn.GELU()

    def forward(self, x):
        return self.fc2(self.act_fn(self.fc1(x)))


def test_an_mlp_without_the_three_projections_has_no_plans(base):
    base.layers[1].mlp = TwoMatrixMlp(64, 96, torch.bfloat16).eval()
    assert [plans is None for plans in pc._model_plans(base)] == [False, True, False]
    assert not native(base)
    base.layers[2].mlp._modules["up_proj"] = None
    assert pc._layer_plans(base.layers[2]) is None


@pytest.mark.gpu
@pytest.mark.parametrize("end", [60, 136])
def test_refresh_runs_an_mlp_of_another_form(gpu_device, end):
    from test_gpu_packed import make_model, make_request

    model = make_model(gpu_device, "llama", kv_heads=2, head_dim=64, dtype=torch.bfloat16, layers=2)
    model.model.layers[1].mlp = TwoMatrixMlp(256, 384, torch.bfloat16, gpu_device).eval()
    shim, ids, base = make_request(model, length=200)
    ours, _ = pc.packed_interval_repair(shim, base, ids, [(20, end)])
    modules, _ = pc.packed_interval_repair(shim, base, ids, [(20, end)], fused_projections=False)
    for a, b in zip(ours.layers, modules.layers):
        for x, y in ((a.keys, b.keys), (a.values, b.values)):
            # one layer of the default path up to 64 rows: the streaming projections' summation order
            assert (x.double() - y.double()).norm() <= 2 * torch.finfo(torch.bfloat16).eps * y.double().norm()
