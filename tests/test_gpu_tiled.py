"""Projections and refreshes of more than 64 packed rows (kvr_tiled_linear_multi,
kvr_decoder_tiled_forward): against fp64 products, and against the module path
whose library GEMMs they replace. The rows cross the tiles' edges (64 + 1, 80,
96, 128, 144, ... 288 rows a tile, then several tiles), k has fewer 64-wide
stages than LDS buffers, ragged splits and the full sizes of an 8B layer."""

from __future__ import annotations

import ctypes
import re
from pathlib import Path

import pytest
import torch

from test_gpu_operators import assert_linear_close, exact_linear, ulp_distance
from test_gpu_packed import make_model, make_request

CONCAT, SILU_GATE, RESIDUAL = 0, 1, 2


def tiled(x, weights, epilogue=CONCAT, residual=None):
    from kv_cache_repair_amd import _native

    lib = _native.lib()
    m, k = x.shape
    rows = [int(w.shape[0]) for w in weights]
    n_out = rows[0] if epilogue == SILU_GATE else sum(rows)
    y = torch.full((m, n_out), float("nan"), dtype=x.dtype, device=x.device)
    need = int(lib.kvr_tiled_linear_workspace_bytes(m, sum(rows), k))
    assert need >= 0
    ws = torch.empty(max(need, 1), dtype=torch.uint8, device=x.device)
    status = lib.kvr_tiled_linear_multi(
        x.data_ptr(), len(weights), (ctypes.c_void_p * len(weights))(*(w.data_ptr() for w in weights)),
        (ctypes.c_int32 * len(weights))(*rows), _native.i64_array([int(w.stride(0)) for w in weights]), y.data_ptr(), m,
        k, int(x.stride(0)), n_out, epilogue, residual.data_ptr() if residual is not None else None,
        n_out if residual is not None else 0, ws.data_ptr() if need else None, need, _native.DTYPE_CODES[x.dtype],
        _native.stream_handle(x.device))
    _native.check(status, "kvr_tiled_linear_multi")
    return y


def assert_gate_close(y, x, gate, up):
    """Every element of silu(x gate^T) * (x up^T) within what the roundings of the
    two products (assert_linear_close's bound), of the activation and of the
    result allow; |silu'| <= 1.1."""
    eps, tiny = torch.finfo(y.dtype).eps, torch.finfo(y.dtype).tiny
    size = x.double().abs()
    g, u = (x.double() @ w.double().T for w in (gate, up))
    g_off, u_off = (eps * p.abs() + 2.0 ** -20 * (size @ w.double().abs().T) for p, w in ((g, gate), (u, up)))
    act = g * torch.sigmoid(g)
    act_off = 1.1 * g_off + eps * act.abs() + tiny
    bound = act_off * (u.abs() + u_off) + act.abs() * u_off
    bound += eps * (act * u).abs() + eps * bound + tiny
    assert ((y.double() - act * u).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows", [(4096, 1024, 1024), (4096,), (264, 72, 40), (8,)])
@pytest.mark.parametrize("k", [64, 192, 1088, 4096])
@pytest.mark.parametrize("m", [1, 65, 81, 113, 129, 145, 209, 282, 289, 513, 1383])
def test_tiled_projection_matches_the_exact_product(gpu_device, dtype, rows, k, m):
    torch.manual_seed(m + k + rows[0])
    x = torch.randn(m, k + 8, device=gpu_device).to(dtype)[:, :k]
    weights = [(torch.randn(n, k + 16, device=gpu_device) * 0.03).to(dtype)[:, 8:8 + k] for n in rows]
    y = tiled(x, weights)
    assert_linear_close(y, x, torch.cat(weights))
    residual = torch.randn(m, sum(rows), device=gpu_device).to(dtype)
    assert torch.equal(tiled(x, weights, RESIDUAL, residual), y + residual)
    assert torch.equal(tiled(x, weights), y)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(4096, 14336), (4096, 12288)])
@pytest.mark.parametrize("m", [65, 97, 160, 240, 400, 841, 2049, 4099])
def test_tiled_projection_with_long_rows_and_many_tiles(gpu_device, shape, m):
    n, k = shape
    torch.manual_seed(m)
    x = torch.randn(m, k, device=gpu_device).to(torch.bfloat16)
    w = (torch.randn(n, k, device=gpu_device) * 0.03).to(torch.bfloat16)
    assert_linear_close(tiled(x, [w]), x, w)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,k", [(14336, 4096), (12288, 4096), (136, 192), (8, 64)])
@pytest.mark.parametrize("m", [65, 79, 96, 113, 200, 282, 400, 641, 1383])
def test_tiled_gate_matches_the_eager_chain(gpu_device, dtype, n, k, m):
    """The gated epilogue rounds as act_fn(gate_proj(x)) * up_proj(x): at most one
    unit from each of the two projections' roundings."""
    torch.manual_seed(m + n)
    x = torch.randn(m, k, device=gpu_device).to(dtype)
    gate, up = ((torch.randn(n, k, device=gpu_device) * 0.05).to(dtype) for _ in range(2))
    y = tiled(x, [gate, up], SILU_GATE)
    eager = torch.nn.functional.silu(exact_linear(x, gate)) * exact_linear(x, up)
    assert_gate_close(y, x, gate, up)
    assert (ulp_distance(y, eager) <= 2).float().mean().item() >= 0.99


def wide_model(device, family, dtype):
    """Hidden size 1024, heads of 128: q/k/v and o split K up to some hundred rows."""
    from transformers import LlamaConfig, LlamaForCausalLM, Qwen3Config, Qwen3ForCausalLM

    kw = dict(vocab_size=97, hidden_size=1024, intermediate_size=2048, num_hidden_layers=3, num_attention_heads=8,
              num_key_value_heads=4, head_dim=128, max_position_embeddings=512)
    config, ctor = (LlamaConfig, LlamaForCausalLM) if family == "llama" else (Qwen3Config, Qwen3ForCausalLM)
    torch.manual_seed(3)
    model = ctor(config(**kw)).to(device=device, dtype=dtype).eval()
    for name, p in model.named_parameters():  # per-head norms of their own
        if "norm" in name:
            p.data.copy_(1 + 0.2 * torch.randn(p.shape, device=device))
    return model


@pytest.mark.gpu
@pytest.mark.parametrize("family", ["llama", "qwen3"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("count", [65, 141, 282])
def test_tiled_refresh_from_split_partials_matches_the_module_path(gpu_device, family, dtype, count):
    """q/k/v, o and down leave split-K partials of `count` rows a split to the
    fresh-row epilogue (per-head norms folded in or not) and the norms. (fp16 layers
    with per-head norms project q, k and v apart and reduce them.)"""
    from kv_cache_repair_amd import _native
    from kv_cache_repair_amd.kernels import packed_cache as pc

    lib = _native.lib()
    assert all(lib.kvr_tiled_linear_workspace_bytes(count, n, k) > 0 for n, k in ((2048, 1024), (1024, 1024), (1024, 2048)))
    model = wide_model(gpu_device, family, dtype)
    shim, ids, base = make_request(model, length=400)
    edited = ids.clone()
    edited[0, 70:] = (edited[0, 70:] + 7) % 97
    intervals = [(0, 3), (20, 10 + count), (380, 387)]
    ours, _ = pc.packed_interval_repair(shim, base, edited, intervals)
    modules, _ = pc.packed_interval_repair(shim, base, edited, intervals, fused_projections=False)
    rows = torch.tensor([p for s, e in intervals for p in range(s, e)], device=gpu_device)
    assert len(rows) == count
    for a, b in zip(ours.layers, modules.layers):
        for x, y in ((a.keys, b.keys), (a.values, b.values)):
            u, v = x[0][:, rows].double(), y[0][:, rows].double()
            # as in test_tiled_refresh_matches_the_module_path, and no row of a head apart
            off = (u - v).norm(dim=-1) / v.norm(dim=-1)
            assert (u - v).norm() <= 2 * torch.finfo(dtype).eps * v.norm() and off.max() <= 8 * torch.finfo(dtype).eps


@pytest.mark.gpu
@pytest.mark.parametrize("family,dtype", [("llama", torch.bfloat16), ("qwen3", torch.bfloat16),
                                          ("llama", torch.float16), ("qwen3", torch.float16)])
@pytest.mark.parametrize("count", [65, 96, 133])
def test_tiled_refresh_matches_the_module_path(gpu_device, family, dtype, count):
    """More than 64 rows run as one kvr_decoder_tiled_forward call; the module path
    (library GEMMs) gives the same caches up to fp32 summation order."""
    from kv_cache_repair_amd.kernels import packed_cache as pc

    model = make_model(gpu_device, family, kv_heads=2, head_dim=64, dtype=dtype, layers=3)
    shim, ids, base = make_request(model, length=300)
    edited = ids.clone()
    edited[0, 70:] = (edited[0, 70:] + 7) % 97
    intervals = [(0, 3), (20, 20 + count - 10), (280, 287)]
    calls = []
    native = pc._native_refresh
    pc._native_refresh = lambda *a, **kw: (calls.append(kw.get("tiled")), native(*a, **kw))[1]
    try:
        ours, _ = pc.packed_interval_repair(shim, base, edited, intervals)
        modules, _ = pc.packed_interval_repair(shim, base, edited, intervals, fused_projections=False)
    finally:
        pc._native_refresh = native
    assert calls == [True]
    rows = torch.tensor([p for s, e in intervals for p in range(s, e)], device=gpu_device)
    keep = torch.ones(300, dtype=torch.bool, device=gpu_device)
    keep[rows] = False
    for a, b in zip(ours.layers, modules.layers):
        for x, y in ((a.keys, b.keys), (a.values, b.values)):
            assert torch.equal(x[:, :, keep].view(torch.int16), y[:, :, keep].view(torch.int16))
            u, v = x[0][:, rows], y[0][:, rows]
            # each layer's few 16-bit roundings, made over sums in another order, are half an eps of a row each
            assert (u.double() - v.double()).norm() <= 2 * torch.finfo(dtype).eps * v.double().norm()
            cosine = torch.nn.functional.cosine_similarity(u.float(), v.float(), dim=-1)
            assert cosine.min().item() >= 0.9999


@pytest.mark.gpu
@pytest.mark.parametrize("refused", ["expanded weight", "kv rows", "row limit"])
def test_weights_the_tiled_kernel_refuses_keep_the_module_path(gpu_device, refused, monkeypatch):
    """What the modules served before stays served: overlapping weight rows, K/V
    rows that are no multiple of 8, more rows than a call takes."""
    from kv_cache_repair_amd.kernels import packed_cache as pc

    if refused == "kv rows":  # one KV head of 12
        from transformers import LlamaConfig, LlamaForCausalLM

        torch.manual_seed(7)
        model = LlamaForCausalLM(LlamaConfig(vocab_size=97, hidden_size=192, intermediate_size=256, num_hidden_layers=2,
                                             num_attention_heads=16, num_key_value_heads=1, head_dim=12))
        model = model.to(device=gpu_device, dtype=torch.bfloat16).eval()
        assert not pc._tiled_weights(pc._model_plans(model.model))
    else:
        model = make_model(gpu_device, "llama", kv_heads=2, head_dim=64, dtype=torch.bfloat16, layers=2)
        assert pc._tiled_weights(pc._model_plans(model.model))
    if refused == "expanded weight":
        projection = model.model.layers[1].self_attn.v_proj
        row = projection.weight.detach()[:1].clone()
        projection.weight = torch.nn.Parameter(row.expand(projection.weight.shape), requires_grad=False)
    elif refused == "row limit":
        monkeypatch.setattr(pc, "_TILED_MAX_ROWS", 95)
    shim, ids, base = make_request(model, length=200)
    monkeypatch.setattr(pc, "_native_refresh", lambda *a, **kw: pytest.fail("native forward taken"))
    ours, _ = pc.packed_interval_repair(shim, base, ids, [(20, 80), (100, 136)])
    modules, _ = pc.packed_interval_repair(shim, base, ids, [(20, 80), (100, 136)], fused_projections=False)
    for a, b in zip(ours.layers, modules.layers):
        assert torch.equal(a.keys, b.keys) and torch.equal(a.values, b.values)


@pytest.mark.gpu
@pytest.mark.parametrize("end", [60, 136])
def test_layers_of_several_widths_keep_the_module_path(gpu_device, end, monkeypatch):
    from kv_cache_repair_amd.kernels import packed_cache as pc

    model = make_model(gpu_device, "llama", kv_heads=2, head_dim=64, dtype=torch.bfloat16, layers=2)
    mlp = model.model.layers[1].mlp
    for name, size in (("gate_proj", (384, 256)), ("up_proj", (384, 256)), ("down_proj", (256, 384))):
        weight = torch.randn(size, device=gpu_device) * 0.03
        getattr(mlp, name).weight = torch.nn.Parameter(weight.to(torch.bfloat16), requires_grad=False)
    shim, ids, base = make_request(model, length=200)
    monkeypatch.setattr(pc, "_native_refresh", lambda *a, **kw: pytest.fail("native forward taken"))
    ours, _ = pc.packed_interval_repair(shim, base, ids, [(20, end)])
    modules, _ = pc.packed_interval_repair(shim, base, ids, [(20, end)], fused_projections=False)
    for a, b in zip(ours.layers, modules.layers):
        for x, y in ((a.keys, b.keys), (a.values, b.values)):
            if end > 84:
                assert torch.equal(x, y)
            # up to 64 rows each layer still runs the streaming projections: two layers' 16-bit roundings
            assert (x.double() - y.double()).norm() <= 2 * torch.finfo(torch.bfloat16).eps * y.double().norm()


@pytest.mark.gpu
@pytest.mark.parametrize("end", [60, 136])
@pytest.mark.parametrize("change", ["epsilon", "activation", "rows"])
def test_refreshes_follow_what_changes_on_the_same_modules(gpu_device, change, end):
    """Set on modules and parameters that stay the same objects at the same
    addresses, between two refreshes: seen as the modules see it."""
    from kv_cache_repair_amd.kernels import packed_cache as pc

    model = make_model(gpu_device, "llama", kv_heads=2, head_dim=64, dtype=torch.bfloat16, layers=2)
    shim, ids, base = make_request(model, length=200)
    intervals = [(20, end)]
    before, _ = pc.packed_interval_repair(shim, base, ids, intervals)
    layer = model.model.layers[0]
    if change == "epsilon":
        layer.post_attention_layernorm.variance_epsilon = 0.5
    elif change == "activation":
        layer.mlp.act_fn = torch.nn.ReLU().eval()
    else:
        for mlp in (each.mlp for each in model.model.layers):
            mlp.gate_proj.weight.data = mlp.gate_proj.weight.data[:256]
            mlp.up_proj.weight.data = mlp.up_proj.weight.data[:256]
            mlp.down_proj.weight.data = mlp.down_proj.weight.data[:, :256]
    ours, _ = pc.packed_interval_repair(shim, base, ids, intervals)
    modules, _ = pc.packed_interval_repair(shim, base, ids, intervals, fused_projections=False)
    x, y, z = (cache.layers[1].values[0, :, 20:end].double() for cache in (ours, modules, before))
    tight = 2 * torch.finfo(torch.bfloat16).eps * y.norm()  # two layers' 16-bit roundings
    assert (x - y).norm() <= tight < 0.5 * (z - y).norm()


def test_tiled_entry_points_are_exported_and_refuse_before_any_launch():
    from kv_cache_repair_amd import _native

    lib = _native.lib()
    header = Path(__file__).resolve().parents[1] / "include" / "kvrepair_tiled.h"
    text = re.sub(r"/\*.*?\*/", "", header.read_text(), flags=re.S)
    names = set(re.findall(r"\b(kvr_[a-z0-9_]+)\s*\(", text))
    assert len(names) == 5 and all(hasattr(lib, name) for name in names)
    for m, rows, k in ((0, 64, 64), (65, 4100, 4096), (65, 4096, 4100), ((1 << 20) + 1, 64, 64)):
        assert lib.kvr_tiled_linear_workspace_bytes(m, rows, k) == -3
    w, fake = (ctypes.c_void_p * 1)(4096), ctypes.c_void_p(4096)  # never dereferenced: refused on the host

    def call(x=fake, rows=64, ld=128, ldx=128, ldy=64, k=128, dtype=2, epilogue=CONCAT, n=1):
        return lib.kvr_tiled_linear_multi(x, n, w, (ctypes.c_int32 * 1)(rows), _native.i64_array([ld]), fake, 70, k, ldx,
                                          ldy, epilogue, None, 0, None, 0, dtype, None)

    assert call(dtype=0) == -2 and call(n=4) == -1 and call(epilogue=9) == -1
    assert call(rows=60) == -3 and call(k=100) == -3 and call(epilogue=SILU_GATE) == -3
    assert call(ld=120) == -4 and call(ldx=132) == -4 and call(ldy=66) == -4 and call(x=ctypes.c_void_p(4100)) == -4
    assert call(epilogue=RESIDUAL) == -5 and call(x=None) == -5
    assert call(rows=4096, ldy=4096, k=4096, ldx=4096, ld=4096) == -6  # splits K, no workspace
    d = _native.RefreshDesc(rows=65, hidden=4096, q_heads=32, kv_heads=8, head_dim=128, intermediate=14336,
                            n_keys=7680, scale=128 ** -0.5, dtype=2)
    assert lib.kvr_decoder_scratch_bytes(ctypes.byref(d)) == -3  # the streaming forward keeps its limit
    assert lib.kvr_decoder_tiled_scratch_bytes(ctypes.byref(d)) > 0
    assert lib.kvr_decoder_tiled_gemm_workspace_bytes(ctypes.byref(d)) == max(
        lib.kvr_tiled_linear_workspace_bytes(65, r, k)
        for r, k in ((6144, 4096), (4096, 4096), (1024, 4096), (4096, 14336)))
    for field, value in (("rows", 0), ("hidden", 4100), ("intermediate", 14344), ("q_heads", 30)):
        bad = _native.RefreshDesc.from_buffer_copy(d)
        setattr(bad, field, value)
        assert lib.kvr_decoder_tiled_scratch_bytes(ctypes.byref(bad)) == -3, field
