"""Packed selected-row refresh through isolated native decoder module shells.

MI355X counterpart of the reference packed executor
(src/kv_cache_repair/kernels/packed_cache.py:225-298), re-derived for
transformers 5.15. The selected rows run through every layer in ONE
layer-major HF forward; at each layer the fresh K/V are scattered into the
owned output cache (libkvrepair kvr_indexed_scatter_kv) and then attend to
their full absolute causal history (libkvrepair kvr_packed_causal_attention),
with no materialised mask and no GQA head copies.

transformers 5.15 plugin points used (the reference's three, re-derived):
  1. an attention function registered in ALL_ATTENTION_FUNCTIONS under a name
     with no mask interface, so create_causal_mask returns None;
  2. a DynamicLayer subclass whose update() scatters and returns the full K/V
     (5.15 passes no cache_position, so positions come from the context);
  3. a per-call context passed as a forward kwarg — no global request state.
"""

from __future__ import annotations

import copy
import ctypes
import types
import weakref
from dataclasses import dataclass, field
from threading import Lock
from typing import Any, Sequence

import numpy as np
import torch
import transformers
from transformers.cache_utils import Cache, DynamicLayer

from .. import _native
from . import projection as _projection
from .executor import _validate_cache, _validate_intervals, layer_kv, tensor_layout, uniform_layers
from .indexed_attention import IndexedPlan, DeviceIndexedPlan, _require_gfx950

_ATTENTION_NAME = "kvr_hip_packed_absolute_attention_v1"
_REGISTRATION_LOCK = Lock()
_SUPPORTED_TRANSFORMERS = ("5.15.0",)
_BACKENDS = ("hip",)


@dataclass
class _PackedContext:
    """Per-request state shared by the layer shells of one forward."""

    positions: torch.Tensor
    logical_length: int
    backend: str
    device_plan: Any = None
    launcher: Any = None


@dataclass
class _Launcher:
    """Precomputed ctypes arguments for the per-layer scatter and attention calls."""

    device: torch.device
    n_sel: int
    n_keys: int
    q_heads: int
    kv_heads: int
    head_dim: int
    dtype_code: int
    host_schedule: Any
    device_schedule: torch.Tensor
    workspace: torch.Tensor | None
    workspace_bytes: int
    positions_ptr: int
    _strides: dict = field(default_factory=dict)

    def _stride_array(self, tensors):
        key = tuple(t.stride() for t in tensors)
        arr = self._strides.get(key)
        if arr is None:
            arr = _native.i64_array([s for t in tensors for s in _native.strides3(t)])
            self._strides[key] = arr
        return arr

    def scatter(self, keys, values, fresh_k, fresh_v) -> None:
        status = _native.lib().kvr_indexed_scatter_kv(
            keys.data_ptr(), values.data_ptr(), fresh_k.data_ptr(), fresh_v.data_ptr(), self.positions_ptr,
            self.n_sel, self.kv_heads, self.n_keys, self.head_dim,
            self._stride_array((keys, values, fresh_k, fresh_v)), self.dtype_code,
            _native.stream_handle(self.device))
        _native.check(status, "kvr_indexed_scatter_kv")

    def rope_scatter(self, q, q_out, fresh_k, fresh_v, keys, values, cos, sin, norms=None) -> None:
        """The fresh-row epilogue; ``norms`` = (q_norm, k_norm) modules folds
        their per-head RMSNorm in front of RoPE (kvr_rope_scatter_kv_norm)."""
        lib = _native.lib()
        args = (q.data_ptr(), q_out.data_ptr(), fresh_k.data_ptr(), fresh_v.data_ptr(), keys.data_ptr(),
                values.data_ptr(), cos.data_ptr(), sin.data_ptr(), self.positions_ptr, self.n_sel, self.q_heads,
                self.kv_heads, self.n_keys, self.head_dim,
                self._stride_array((q, q_out, fresh_k, fresh_v, keys, values)),
                _native.i64_array([int(cos.stride(-2)), int(cos.stride(-1)), int(sin.stride(-2)),
                                   int(sin.stride(-1))]))
        if norms is None:
            status = lib.kvr_rope_scatter_kv(*args, self.dtype_code, _native.stream_handle(self.device))
            _native.check(status, "kvr_rope_scatter_kv")
            return
        q_norm, k_norm = norms
        status = lib.kvr_rope_scatter_kv_norm(*args, q_norm.weight.data_ptr(), k_norm.weight.data_ptr(),
                                              float(q_norm.variance_epsilon), float(k_norm.variance_epsilon),
                                              self.dtype_code, _native.stream_handle(self.device))
        _native.check(status, "kvr_rope_scatter_kv_norm")

    def attention(self, q, k, v, out_view, scale: float) -> None:
        status = _native.lib().kvr_packed_causal_attention(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), out_view.data_ptr(), self.positions_ptr, self.n_sel,
            self.q_heads, self.kv_heads, self.n_keys, self.head_dim, float(scale),
            self._stride_array((q, k, v, out_view)), self.device_schedule.data_ptr(), len(self.host_schedule),
            self.host_schedule, self.workspace.data_ptr() if self.workspace is not None else None,
            self.workspace_bytes, self.dtype_code, _native.stream_handle(self.device))
        _native.check(status, "kvr_packed_causal_attention")


def _packed_attention(module, query, key, value, attention_mask, *, scaling=None, dropout=0.0,
                      sur_packed_context=None, **kwargs):
    """Registered attention function: packed queries over the full mixed cache."""
    context = sur_packed_context
    if not isinstance(context, _PackedContext):
        raise RuntimeError("packed attention requires explicit per-call request context")
    if attention_mask is not None:
        raise RuntimeError("native dense mask construction must be bypassed for packed attention")
    if dropout:
        raise ValueError("packed attention supports inference without dropout only")
    if query.shape[-2] != context.positions.numel() or key.shape[-2] != context.logical_length:
        raise RuntimeError("packed attention query/cache lengths drifted")
    if context.backend != "hip":
        raise RuntimeError("unknown packed attention backend")
    launcher = context.launcher
    if (query.shape[1], key.shape[1], query.shape[3]) != (launcher.q_heads, launcher.kv_heads, launcher.head_dim):
        raise RuntimeError("packed attention head geometry drifted")
    scale = query.shape[-1] ** -0.5 if scaling is None else float(scaling)
    # Native modules consume [batch, query, query_head, head_dim]; the kernel
    # writes that layout directly through a permuted view.
    out = torch.empty((1, query.shape[2], query.shape[1], query.shape[3]), dtype=query.dtype, device=query.device)
    launcher.attention(query, key, value, out.permute(0, 2, 1, 3), scale)
    return out, None


def _register_attention() -> None:
    from transformers.masking_utils import ALL_MASK_ATTENTION_FUNCTIONS
    from transformers.modeling_utils import ALL_ATTENTION_FUNCTIONS

    with _REGISTRATION_LOCK:
        if _ATTENTION_NAME in ALL_MASK_ATTENTION_FUNCTIONS:
            raise RuntimeError("packed backend name unexpectedly has a native mask interface")
        if _ATTENTION_NAME in ALL_ATTENTION_FUNCTIONS:
            if ALL_ATTENTION_FUNCTIONS[_ATTENTION_NAME] is not _packed_attention:
                raise RuntimeError("packed backend registry name is already owned by another implementation")
        else:
            ALL_ATTENTION_FUNCTIONS.register(_ATTENTION_NAME, _packed_attention)


def _silu_activations() -> tuple[type, ...]:
    from transformers.activations import SiLUActivation

    return (torch.nn.SiLU, SiLUActivation)


_SILU_ACTIVATIONS = _silu_activations()


def _norms_in_epilogue(dtype, head_dim: int, q_weight: torch.Tensor, k_weight: torch.Tensor) -> bool:
    """Whether Qwen3's per-head q/k norms run inside the fresh-row epilogue
    (kvr_rope_scatter_kv_norm). The fold lives in the epilogue's vector kernel
    only, so it needs what that kernel needs (kvr_fresh.hip, rope_norm_fold_ok):
    bf16 / fp32 rows (fp16 rows take the scalar kernel), each half row a
    power-of-two count (at most 64) of 16-byte chunks, 16-byte aligned norm
    weights. Otherwise the q and k rows are normalised by two kvr_rms_norm
    launches first, as kvr_decoder_layer does under the same condition."""
    if dtype not in (torch.bfloat16, torch.float32):
        return False
    half_bytes = (int(head_dim) // 2) * (4 if dtype == torch.float32 else 2)
    chunks = half_bytes // 16
    return (half_bytes > 0 and half_bytes % 16 == 0 and chunks & (chunks - 1) == 0 and chunks <= 64
            and q_weight.data_ptr() % 16 == 0 and k_weight.data_ptr() % 16 == 0)


def _checked_head_norm(module, x: torch.Tensor):
    weight = module.weight
    if weight.dtype != x.dtype or weight.numel() != x.shape[-1] or not weight.is_contiguous() \
            or not isinstance(getattr(module, "variance_epsilon", None), float):
        raise RuntimeError("packed fused per-head RMSNorm geometry/dtype drifted")
    return module


def _rms_norm(module, x: torch.Tensor, residual: torch.Tensor | None = None):
    """One kvr_rms_norm launch with ``module``'s weight and epsilon over the last
    dim of contiguous ``x``; with ``residual`` also returns s = residual + x."""
    weight = module.weight
    if x.dtype != weight.dtype or not x.is_contiguous() or weight.numel() != x.shape[-1] \
            or (residual is not None and (residual.shape != x.shape or residual.dtype != x.dtype
                                          or not residual.is_contiguous())):
        raise RuntimeError("packed fused RMSNorm geometry/dtype drifted")
    hidden = int(x.shape[-1])
    rows = x.numel() // hidden
    out = torch.empty_like(x)
    summed = torch.empty_like(x) if residual is not None else None
    status = _native.lib().kvr_rms_norm(
        x.data_ptr(), residual.data_ptr() if residual is not None else None,
        summed.data_ptr() if summed is not None else None, out.data_ptr(), weight.data_ptr(), rows, hidden,
        _native.i64_array([hidden] * 4), float(module.variance_epsilon), _native.DTYPE_CODES[x.dtype],
        _native.stream_handle(x.device))
    _native.check(status, "kvr_rms_norm")
    return out if residual is None else (out, summed)


def _silu_mul(gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    if gate.shape != up.shape or gate.dtype != up.dtype or not gate.is_contiguous() or not up.is_contiguous():
        raise RuntimeError("packed fused MLP activation geometry/dtype drifted")
    out = torch.empty_like(gate)
    status = _native.lib().kvr_silu_mul(gate.data_ptr(), up.data_ptr(), out.data_ptr(), gate.numel(),
                                        _native.DTYPE_CODES[gate.dtype], _native.stream_handle(gate.device))
    _native.check(status, "kvr_silu_mul")
    return out


@dataclass
class _LayerPlans:
    """kvr_linear_multi plans of one decoder layer's projections: q/k/v in one
    launch (separate launches for fp16 layers that normalise q/k per head), o,
    the SiLU-gated gate/up pair in one launch, down."""

    pointers: tuple
    qkv: Any
    q: Any
    k: Any
    v: Any
    o: Any
    gate_up: Any
    down: Any
    q_cols: int
    k_cols: int
    geometry: tuple | None = None  # _set_geometry
    desc: Any = None  # kvr_layer_desc template (no cache pointers) for kvr_decoder_layer, or None


_TILED_MAX_ROWS = 1 << 20  # rows of one kvr_decoder_tiled_forward call
_TILED_WIDE, _TILED_WIDE_ROWS = 8192, 4096  # hidden size and rows from which the library's GEMMs are at least as fast


class _PlanList(list):
    """The layers' plans of one module tree; carries the descriptor template
    that _native_layer_descs derives from them."""

    descs_template = None
    tiled = None  # _tiled_weights of these plans, once asked
    geometry = None  # _one_geometry of these plans, once asked


_PLAN_CACHE: "weakref.WeakKeyDictionary[Any, _LayerPlans]" = weakref.WeakKeyDictionary()
_PLAN_LOCK = Lock()
# Per decoder (`base`): the fingerprint of the module tree that last passed
# _qualify with its parameters on GPU `index` -> (fingerprint, index), and the
# layer plans built for that fingerprint -> (fingerprint, plans).
_QUALIFIED: "weakref.WeakKeyDictionary[Any, tuple]" = weakref.WeakKeyDictionary()
_MODEL_PLANS: "weakref.WeakKeyDictionary[Any, tuple]" = weakref.WeakKeyDictionary()


def _plain_linear(module) -> bool:
    return (type(module) is torch.nn.Linear and module.bias is None
            and _projection.supported_weight(module.weight))


def _layer_modules(layer):
    """(projection modules, norm modules) of a Llama/Qwen3 decoder layer, read
    through the `_modules` dicts (plain dict lookups: this runs per layer), or
    None when one of the projections is not there (another attention or MLP put
    in the layer, which runs as the module it is)."""
    attention, mlp = layer._modules["self_attn"], layer._modules["mlp"]
    am, mm = attention._modules, mlp._modules
    projections = (*map(am.get, ("q_proj", "k_proj", "v_proj", "o_proj")),
                   *map(mm.get, ("gate_proj", "up_proj", "down_proj")))
    if None in projections:
        return None
    norms = [layer._modules["input_layernorm"], layer._modules["post_attention_layernorm"]]
    if am.get("q_norm") is not None:
        norms += [am["q_norm"], am["k_norm"]]
    return projections, norms


def _plans_key(layer, projections, norms) -> tuple:
    """Identity of everything a layer's plans point at: module objects, weight
    tensors, their storage and layout, the projections' (absent) biases, and the
    constants taken from the modules."""
    layout_key = tensor_layout().layout_key
    key = [_module_walk().layer_constants((layer,))]
    add = key.extend
    for m in (*projections, *norms):
        params = m.__dict__["_parameters"]
        w = params.get("weight")
        add((id(m), id(w), layout_key(w) if w is not None else b"", params.get("bias") is None))
    return tuple(key)


def _layer_plans(layer) -> _LayerPlans | None:
    """Plans for ``layer`` (one of the caller's decoder layers), cached per layer
    and rebuilt when a module, weight, weight layout or constant changes; None when any
    projection is missing, has a bias, is not a plain fp16/bf16 nn.Linear, or the MLP
    activation is not SiLU."""
    found = _layer_modules(layer)
    if found is None:
        return None
    projections, norms = found
    key = _plans_key(layer, projections, norms)
    with _PLAN_LOCK:
        cached = _PLAN_CACHE.get(layer)
    if cached is not None and cached.pointers == key:
        return cached
    mlp = layer._modules["mlp"]
    if not all(_plain_linear(m) for m in projections) or not isinstance(mlp.act_fn, _SILU_ACTIVATIONS):
        return None
    weights = [m.weight for m in projections]
    if len({(w.dtype, w.device) for w in weights}) != 1 or weights[4].shape != weights[5].shape:
        return None
    q, k, v, o, gate, up, down = weights
    plan = _projection.ProjectionPlan
    # q/k/v in one launch, unless per-head norms must run as separate launches
    # on contiguous q and k (where the epilogue cannot fold them in)
    separate = len(norms) > 2 and not _norms_in_epilogue(
        q.dtype, getattr(layer._modules["self_attn"], "head_dim", 0), norms[2].weight, norms[3].weight)
    plans = _LayerPlans(
        pointers=key, qkv=None if separate else plan([q, k, v]), q=plan([q]) if separate else None,
        k=plan([k]) if separate else None, v=plan([v]) if separate else None, o=plan([o]),
        gate_up=plan([gate, up], _projection.SILU_GATE), down=plan([down]), q_cols=int(q.shape[0]),
        k_cols=int(k.shape[0]), desc=_layer_desc(layer, weights, norms))
    _set_geometry(plans, int(getattr(layer._modules["self_attn"], "head_dim", 0)))
    with _PLAN_LOCK:
        _PLAN_CACHE[layer] = plans
    return plans


def _set_geometry(plans: _LayerPlans, head_dim: int) -> None:
    """plans.geometry = (query columns, K columns, head dim, hidden, intermediate)
    when the layer's weights chain as the native layer call runs them."""
    first = plans.q or plans.qkv
    k_rows, v_rows = (plans.k.rows, plans.v.rows) if plans.qkv is None else (plans.qkv._rows[1], plans.qkv._rows[2])
    o, gate_up, down = plans.o, plans.gate_up, plans.down
    if (first.k, gate_up.k, down.rows, o.k, down.k, v_rows) == (o.rows, o.rows, o.rows, plans.q_cols, gate_up.n_out,
                                                                k_rows):
        plans.geometry = (plans.q_cols, k_rows, head_dim, o.rows, down.k)


def _layer_desc(layer, weights, norms):
    """kvr_layer_desc of ``layer`` without cache pointers, or None when a norm is
    not a plain weight-times-normalised RMSNorm of the projections' dtype."""
    dtype, device = weights[0].dtype, weights[0].device
    hidden = int(weights[3].shape[0])
    head_dim = int(getattr(layer.self_attn, "head_dim", 0))
    for i, norm in enumerate(norms):
        w = getattr(norm, "weight", None)
        size = hidden if i < 2 else head_dim
        if not isinstance(w, torch.Tensor) or w.dtype != dtype or w.device != device or tuple(w.shape) != (size,) \
                or not w.is_contiguous() or not isinstance(getattr(norm, "variance_epsilon", None), float):
            return None
    q, k, v, o, gate, up, down = weights
    desc = _native.LayerDesc()
    desc.input_norm, desc.post_norm = norms[0].weight.data_ptr(), norms[1].weight.data_ptr()
    desc.q_norm = norms[2].weight.data_ptr() if len(norms) > 2 else None
    desc.k_norm = norms[3].weight.data_ptr() if len(norms) > 2 else None
    desc.w_q, desc.w_k, desc.w_v, desc.w_o = q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr()
    desc.w_gate, desc.w_up, desc.w_down = gate.data_ptr(), up.data_ptr(), down.data_ptr()
    desc.ld_q, desc.ld_k, desc.ld_v, desc.ld_o = q.stride(0), k.stride(0), v.stride(0), o.stride(0)
    desc.ld_gate, desc.ld_up, desc.ld_down = gate.stride(0), up.stride(0), down.stride(0)
    desc.eps_input, desc.eps_post = norms[0].variance_epsilon, norms[1].variance_epsilon
    if len(norms) > 2:
        desc.eps_q, desc.eps_k = norms[2].variance_epsilon, norms[3].variance_epsilon
    return desc


def _fused_layer_forward(self, hidden_states, attention_mask=None, position_ids=None, past_key_values=None,
                         use_cache=False, position_embeddings=None, **kwargs):
    """Decoder layer of a packed shell with its elementwise work fused.

    The native Llama/Qwen3 decoder layer (transformers 5.15.0
    modeling_llama.py:301-330, modeling_qwen3.py:287-316): input RMSNorm,
    attention, residual add, post-attention RMSNorm, SiLU-gated MLP, residual
    add. Each RMSNorm is one kvr_rms_norm launch (the first residual add fused
    into the second norm); the MLP is kvr_linear_multi's SiLU-gated gate/up
    launch plus the down projection with the second residual add in its
    epilogue when the shell carries projection plans, else the module's linear
    layers around one kvr_silu_mul launch.
    """
    normed = _rms_norm(self.input_layernorm, hidden_states)
    attended, _ = self.self_attn(hidden_states=normed, attention_mask=attention_mask, position_ids=position_ids,
                                 past_key_values=past_key_values, use_cache=use_cache,
                                 position_embeddings=position_embeddings, **kwargs)
    normed, residual = _rms_norm(self.post_attention_layernorm, attended, residual=hidden_states)
    mlp = self.mlp
    plans = getattr(self, "_kvr_plans", None)
    if plans is not None:  # gate/up with the SiLU gate, then down with the residual add
        return plans.down(plans.gate_up(normed), residual=residual)
    if isinstance(mlp.act_fn, _SILU_ACTIVATIONS):
        out = mlp.down_proj(_silu_mul(mlp.gate_proj(normed), mlp.up_proj(normed)))
    else:
        out = mlp(normed)
    return residual + out


class _NativeForward:
    """kvr_refresh_desc of one refresh and the device buffers it points into
    (scratch slab for the layer intermediates, projection workspace)."""

    def __init__(self, launcher: _Launcher, hidden: int, intermediate: int, scale: float, tiled: bool = False):
        d = _native.RefreshDesc()
        d.rows, d.hidden, d.intermediate = launcher.n_sel, hidden, intermediate
        d.q_heads, d.kv_heads, d.head_dim = launcher.q_heads, launcher.kv_heads, launcher.head_dim
        d.n_keys, d.scale, d.dtype = launcher.n_keys, scale, launcher.dtype_code
        d.positions = launcher.positions_ptr
        d.schedule = launcher.device_schedule.data_ptr()
        d.schedule_len = len(launcher.host_schedule)
        d.host_schedule = ctypes.cast(launcher.host_schedule, ctypes.c_void_p)
        if launcher.workspace is not None:
            d.attn_workspace, d.attn_workspace_bytes = launcher.workspace.data_ptr(), launcher.workspace_bytes
        lib = _native.lib()
        names = [f"kvr_decoder_{'tiled_' if tiled else ''}{size}_bytes" for size in ("scratch", "gemm_workspace")]
        scratch, gemm = (int(getattr(lib, name)(ctypes.byref(d))) for name in names)
        _native.check(scratch, names[0])
        _native.check(gemm, names[1])
        self.scratch = torch.empty(scratch, dtype=torch.uint8, device=launcher.device)
        self.gemm = torch.empty(gemm, dtype=torch.uint8, device=launcher.device) if gemm else None
        d.scratch, d.scratch_bytes = self.scratch.data_ptr(), scratch
        if self.gemm is not None:
            d.gemm_workspace, d.gemm_workspace_bytes = self.gemm.data_ptr(), gemm
        self.desc = d
        self.tables = None
        self.stream = ctypes.c_void_p(torch.cuda.current_stream(launcher.device).cuda_stream)

    def bind_tables(self, position_embeddings) -> None:
        """Point the descriptor at the forward's rotary tables (shared by all layers)."""
        if position_embeddings is None:
            raise RuntimeError("native packed layer requires the model's rotary embeddings")
        cos, sin = position_embeddings
        if self.tables is not None and self.tables[0] is cos and self.tables[1] is sin:
            return
        d = self.desc
        for table in (cos, sin):
            if table.shape[-2:] != (d.rows, d.head_dim) or table.numel() != d.rows * d.head_dim \
                    or _native.DTYPE_CODES.get(table.dtype) != d.dtype:
                raise RuntimeError("packed native rotary embedding geometry/dtype drifted")
        d.cos, d.sin = cos.data_ptr(), sin.data_ptr()
        d.cs_strides[:] = (cos.stride(-2), cos.stride(-1), sin.stride(-2), sin.stride(-1))
        self.tables = (cos, sin)


def _fused_norm_forward(self, hidden_states):
    return _rms_norm(self, hidden_states)


def _fused_attention_forward(self, hidden_states, position_embeddings=None, attention_mask=None,
                             past_key_values=None, sur_packed_context=None, **kwargs):
    """Attention block of a packed layer shell with the fresh-row epilogue fused.

    The same computation as the native Llama/Qwen3 attention forward
    (transformers 5.15.0 modeling_llama.py:243-293, modeling_qwen3.py:231-276)
    routed through the packed plugin points: projections run as kvr_linear_multi
    launches when the shell carries projection plans (q/k/v in one), else as
    the module's own layers, Qwen3's per-head q/k RMSNorm as kvr_rms_norm; RoPE of the fresh queries and
    keys at their absolute positions, the key/value scatter into the cache and
    the cache-update bookkeeping are ONE libkvrepair launch
    (kvr_rope_scatter_kv, bit-identical to apply_rotary_pos_emb + the packed
    layer's scatter); then the packed attention and o_proj. Bound only to the
    executor's private module shells, never to the caller's modules.
    """
    context = sur_packed_context
    if not isinstance(context, _PackedContext):
        raise RuntimeError("packed attention requires explicit per-call request context")
    if attention_mask is not None:
        raise RuntimeError("native dense mask construction must be bypassed for packed attention")
    if position_embeddings is None:
        raise RuntimeError("packed fused epilogue requires the model's rotary embeddings")
    if not isinstance(past_key_values, Cache) or not isinstance(past_key_values.layers[self.layer_idx], _PackedLayer):
        raise RuntimeError("packed fused epilogue requires the packed cache layers")
    input_shape = hidden_states.shape[:-1]
    hidden_shape = (*input_shape, -1, self.head_dim)
    plans = getattr(self, "_kvr_plans", None)
    if plans is None:
        query = self.q_proj(hidden_states).view(hidden_shape)
        key = self.k_proj(hidden_states).view(hidden_shape)
        value = self.v_proj(hidden_states).view(hidden_shape)
    elif plans.qkv is not None:  # one launch, three column blocks of one output
        qkv = plans.qkv(hidden_states)
        split = plans.q_cols + plans.k_cols
        query = qkv[..., :plans.q_cols].view(hidden_shape)
        key = qkv[..., plans.q_cols:split].view(hidden_shape)
        value = qkv[..., split:].view(hidden_shape)
    else:
        query = plans.q(hidden_states).view(hidden_shape)
        key = plans.k(hidden_states).view(hidden_shape)
        value = plans.v(hidden_states).view(hidden_shape)
    q_norm = getattr(self, "q_norm", None)
    norms = None
    if q_norm is not None:  # Qwen3: per-head RMSNorm before RoPE
        fused_norms = getattr(self, "_kvr_fused_norms", False)
        if fused_norms and _norms_in_epilogue(query.dtype, self.head_dim, q_norm.weight, self.k_norm.weight):
            norms = (_checked_head_norm(q_norm, query), _checked_head_norm(self.k_norm, key))
        elif fused_norms:  # kvr_rms_norm reads contiguous rows
            query = _rms_norm(q_norm, query.contiguous())
            key = _rms_norm(self.k_norm, key.contiguous())
        else:
            query = q_norm(query)
            key = self.k_norm(key)
    cos, sin = position_embeddings
    layer = past_key_values.layers[self.layer_idx]
    rotated = torch.empty(query.shape, dtype=query.dtype, device=query.device)
    layer.fused_update(query.transpose(1, 2), rotated.transpose(1, 2), key.transpose(1, 2), value.transpose(1, 2),
                       cos, sin, norms)
    launcher = context.launcher
    out = torch.empty(query.shape, dtype=query.dtype, device=query.device)  # [1, B, Hq, D]
    launcher.attention(rotated.transpose(1, 2), layer.keys, layer.values, out.transpose(1, 2), float(self.scaling))
    attended = out.reshape(*input_shape, -1)
    return (plans.o(attended) if plans is not None else self.o_proj(attended)), None


def _make_native_view(base, fused_epilogue: bool = True, fused_layers: bool = True, plans=None):
    """Shallow module shells sharing parameters, with a private config naming the
    packed attention; the caller's modules and config are never modified. With
    ``fused_epilogue`` the attention shells run _fused_attention_forward; with
    ``fused_layers`` the layer and final-norm shells run their fused forwards.
    ``plans`` (one _LayerPlans or None per layer) routes the shells'
    projections through kvr_linear_multi."""
    _register_attention()
    config = copy.deepcopy(base.config)
    config._attn_implementation = _ATTENTION_NAME
    view = copy.copy(base)
    view._modules = base._modules.copy()
    view.config = config
    layers = []
    for original in base.layers:
        layer = copy.copy(original)
        layer._modules = original._modules.copy()
        if hasattr(layer, "config"):
            layer.config = config
        attention = copy.copy(original.self_attn)
        attention._modules = original.self_attn._modules.copy()
        attention.config = config
        layer_plans = plans[len(layers)] if plans is not None else None
        if fused_epilogue:
            attention.forward = types.MethodType(_fused_attention_forward, attention)
            attention._kvr_fused_norms = fused_layers
            attention._kvr_plans = layer_plans
        if fused_layers:
            layer.forward = types.MethodType(_fused_layer_forward, layer)
            layer._kvr_plans = layer_plans
        layer._modules["self_attn"] = attention
        layers.append(layer)
    view._modules["layers"] = torch.nn.ModuleList(layers)
    view.layers.training = False
    if fused_layers:
        norm = copy.copy(base.norm)
        norm.forward = types.MethodType(_fused_norm_forward, norm)
        view._modules["norm"] = norm
    return view


def _module_walk():
    """The _kvr_walk extension (built in-tree with libkvrepair.so): one C pass
    over the module tree for the qualification below. No Python fallback: a
    missing build raises here."""
    try:
        from .. import _kvr_walk
    except ImportError as error:
        raise ImportError("kv_cache_repair_amd._kvr_walk is not built: run build_lib.py (or "
                          "__graft_entry__.build())") from error
    return _kvr_walk


def _qualify(shim, edited_ids, base_cache, attention_backend, writeback_backend):
    """Fail closed outside the inspected contract, before any device work.
    Returns (the module tree's fingerprint (see below) for _projection_plans_for,
    whether any decoder module or the process carries forward hooks)."""
    if transformers.__version__ not in _SUPPORTED_TRANSFORMERS:
        raise ValueError(f"packed HIP executor requires transformers in {_SUPPORTED_TRANSFORMERS}")
    from transformers.models.llama.modeling_llama import LlamaForCausalLM, LlamaModel
    from transformers.models.qwen3.modeling_qwen3 import Qwen3ForCausalLM, Qwen3Model

    model = shim.generator
    base = shim._base_transformer(model)
    if (type(model), type(base)) not in {(LlamaForCausalLM, LlamaModel), (Qwen3ForCausalLM, Qwen3Model)}:
        raise ValueError("packed executor requires exact native dense Llama or Qwen3 classes")
    device = edited_ids.device
    # Module-tree conditions, gathered from the modules' __dict__s in one C pass
    # (_kvr_walk.qualify_walk) through the `_modules` dicts: over the decoder
    # (`base`) subtree, whose modules must all be in eval mode with no
    # per-instance forward and whose forward hooks send the refresh down the
    # module path, and over the rest of the model; no module anywhere may carry
    # a dispatch hook (accelerate's lives in the module's __dict__ as `_hf_hook`)
    # or a parameter off the request device (compared by index: get_device() is
    # -1 off the GPUs, and the request device is a GPU when it matters below).
    index = device.index if device.type == "cuda" else -2
    training, overridden, hooked, forward_hooked, params, dict_ids, param_ids, ptrs = \
        _module_walk().qualify_walk(model, base, tensor_layout().layout_key)
    from torch.nn.modules import module as _module

    forward_hooked = (forward_hooked or bool(_module._global_forward_hooks)
                      or bool(_module._global_forward_pre_hooks))
    # Fingerprint of the tree: every module (its __dict__'s identity) and every
    # parameter slot (the tensor's identity, storage address and layout; an empty
    # slot counts), and the layers' constants by value. A tree with the
    # fingerprint that last qualified on this GPU has the same parameter tensors
    # at the same addresses, so their device check holds as it did; the layer
    # plans are reused under the same condition.
    fingerprint = (dict_ids, param_ids, ptrs, _module_walk().layer_constants(list(base.layers)))
    with _PLAN_LOCK:
        previous = _QUALIFIED.get(base)
    if previous is not None and previous[1] == index and previous[0] == fingerprint:
        fingerprint, off_device = previous[0], False
    else:
        off_device = True in [p is not None and p.get_device() != index for p in params]
    if model.training or base.training or training:
        raise ValueError("packed executor requires eval mode on all decoder modules")
    config = model.config
    if config.num_hidden_layers != len(base_cache.layers) or len(base.layers) != len(base_cache.layers):
        raise ValueError("model and cache layer counts must agree")
    rope = getattr(config, "rope_parameters", None) or {}
    if rope.get("rope_type", "default") != "default" or getattr(base.rotary_emb, "rope_type", None) != "default":
        raise ValueError("packed executor supports default fixed RoPE only")
    if getattr(config, "use_sliding_window", False) or getattr(base, "has_sliding_layers", False):
        raise ValueError("packed executor requires full attention")
    if any(kind != "full_attention" for kind in getattr(config, "layer_types", []) or []):
        raise ValueError("packed executor rejects sliding/hybrid attention")
    if hooked:
        raise ValueError("packed executor does not support dispatch/offload hooks")
    if overridden:
        raise ValueError("packed executor does not support per-instance decoder forward overrides")
    key = layer_kv(base_cache, 0)[0]
    if key.dtype not in _native.DTYPE_CODES:
        raise ValueError("packed HIP executor supports float32, float16 and bfloat16 caches")
    if key.shape[-1] % 2 or key.shape[-1] > 256:
        raise ValueError("packed HIP executor requires an even head dimension <= 256")
    if config.num_attention_heads % config.num_key_value_heads:
        raise ValueError("query head count must be divisible by KV head count")
    # Device checks last: every rejection above is host-only and names its cause.
    if device.type != "cuda" or torch.version.hip is None:
        raise ValueError("packed HIP executor requires one ROCm GPU device")
    if off_device:
        raise ValueError("packed executor requires all model parameters on the request device")
    same = uniform_layers(base_cache.layers)  # one layout: one device for every layer
    if (same is None or same[2].get_device() != index) and True in [
            t.get_device() != index for i in range(len(base_cache.layers)) for t in layer_kv(base_cache, i)]:
        raise ValueError("packed executor requires all cache layers on the request device")
    _require_gfx950(device)
    with _PLAN_LOCK:
        _QUALIFIED[base] = (fingerprint, index)
    return fingerprint, forward_hooked


class _PackedLayer(DynamicLayer):
    """Cache layer that scatters the fresh rows, then exposes the full mixed K/V."""

    def __init__(self, key, value, context, backend):
        super().__init__()
        self.keys, self.values = key, value
        self.dtype, self.device = key.dtype, key.device
        self.is_initialized = True
        self._context = context
        self._backend = backend
        self.updated = False

    def get_mask_sizes(self, query_length):
        return self._context.logical_length, 0

    def update(self, key_states, value_states, *args, **kwargs):
        if self.updated:
            raise RuntimeError("packed native forward updated one layer more than once")
        positions = self._context.positions
        expected = (*self.keys.shape[:2], positions.numel(), self.keys.shape[-1])
        for source, target in ((key_states, self.keys), (value_states, self.values)):
            if source.shape != expected or source.dtype != target.dtype or source.device != target.device:
                raise RuntimeError("packed native projection geometry/dtype/device drifted")
        if self._backend != "hip":
            raise RuntimeError("unknown packed writeback backend")
        self._context.launcher.scatter(self.keys, self.values, key_states, value_states)
        self.updated = True
        return self.keys, self.values

    def fused_update(self, query, query_out, key_states, value_states, cos, sin, norms=None):
        """Fresh-row epilogue: rotate queries (into ``query_out``) and keys at the
        context positions, scatter the keys and values into this layer; with
        ``norms`` = (q_norm, k_norm), RMS-normalise q and k per head first."""
        if self.updated:
            raise RuntimeError("packed native forward updated one layer more than once")
        positions = self._context.positions
        n_sel = positions.numel()
        expected = (*self.keys.shape[:2], n_sel, self.keys.shape[-1])
        for source, target in ((key_states, self.keys), (value_states, self.values)):
            if source.shape != expected or source.dtype != target.dtype or source.device != target.device:
                raise RuntimeError("packed native projection geometry/dtype/device drifted")
        if (query.shape != query_out.shape or query.shape[2:] != (n_sel, self.keys.shape[-1])
                or query.dtype != self.keys.dtype):
            raise RuntimeError("packed native query geometry/dtype drifted")
        for table in (cos, sin):
            if table.shape[-2:] != (n_sel, self.keys.shape[-1]) or table.dtype != self.keys.dtype \
                    or table.numel() != n_sel * self.keys.shape[-1]:
                raise RuntimeError("packed native rotary embedding geometry/dtype drifted")
        if self._backend != "hip":
            raise RuntimeError("unknown packed writeback backend")
        self._context.launcher.rope_scatter(query, query_out, key_states, value_states, self.keys, self.values,
                                            cos, sin, norms)
        self.updated = True


def _rounded_probabilities(dtype: torch.dtype) -> bool:
    """The reference executor's SDPA rounds probabilities to the 16-bit input
    dtype before PV (packed_cache.py:60-67); this path keeps that precision."""
    return dtype in (torch.bfloat16, torch.float16)


def _launcher(device_plan: DeviceIndexedPlan, config, key: torch.Tensor) -> _Launcher:
    q_heads, kv_heads, dim = int(config.num_attention_heads), int(key.shape[1]), int(key.shape[3])
    rounded = _rounded_probabilities(key.dtype)
    host, dev = device_plan.attention_schedule(q_heads, kv_heads, dim, key.dtype, rounded=rounded)
    ws_bytes = int(_native.lib().kvr_attention_workspace_bytes(host, len(host), q_heads, dim))
    _native.check(ws_bytes, "kvr_attention_workspace_bytes")
    workspace = torch.empty(ws_bytes, dtype=torch.uint8, device=key.device) if ws_bytes else None
    return _Launcher(device=key.device, n_sel=device_plan.selected_count, n_keys=device_plan.logical_length,
                     q_heads=q_heads, kv_heads=kv_heads, head_dim=dim, dtype_code=_native.DTYPE_CODES[key.dtype],
                     host_schedule=host, device_schedule=dev, workspace=workspace, workspace_bytes=ws_bytes,
                     positions_ptr=device_plan.positions.data_ptr())


def _check_backends(attention_backend, writeback_backend) -> tuple[str, str]:
    """The backends that run: always the HIP kernels. The reference's default
    names ("sdpa" attention, "torch" writeback, packed_cache.py:225-231) are
    accepted so callers that pass them explicitly keep working; they select the
    same kernels as "hip" (the receipt names what ran). The reference's
    experimental "triton"/"flex" backends and unknown names are rejected."""
    if attention_backend not in _BACKENDS + ("sdpa",):
        raise ValueError("attention_backend must be 'hip' (or the reference default 'sdpa', served by the same "
                         "HIP kernel)")
    if writeback_backend not in _BACKENDS + ("torch",):
        raise ValueError("writeback_backend must be 'hip' (or the reference default 'torch', served by the same "
                         "HIP kernel)")
    return "hip", "hip"


def _check_ids(edited_ids_t):
    if not isinstance(edited_ids_t, torch.Tensor) or edited_ids_t.ndim != 2 or edited_ids_t.shape[0] != 1:
        raise ValueError("edited_ids_t must be a single-batch rank-two tensor")
    if edited_ids_t.dtype not in (torch.int32, torch.int64):
        raise ValueError("edited_ids_t must contain int32 or int64 IDs")


def _receipt(intervals, selected, length, layer_count, attention_backend, writeback_backend):
    return {
        "executor": "packed_interval_repair",
        "schedule": "packed_selected_rows_layer_major",
        "attention_backend": attention_backend,
        "writeback_backend": writeback_backend,
        "interval_count": len(intervals),
        "recomputed_tokens": len(selected),
        "logical_length": length,
        "layer_count": layer_count,
        "base_cache_ownership": "borrowed_immutable",
        "output_cache_ownership": "independent" if selected else "borrowed_base",
        "selected_absolute_positions": list(selected),
        "native_model_mutated": False,
        "numerical_contract": "separate_schedule_qualification_required",
    }


@torch.no_grad()
def _fused_layers_for(fused_layers, dtype: torch.dtype) -> bool:
    """Default: fuse the layer elementwise ops for 16-bit caches only. Their fp32
    mean of squares may differ from the eager chain by an ulp, which is below
    16-bit storage precision; fp32 runs keep the eager ops unless asked."""
    if fused_layers is None:
        return dtype in (torch.float16, torch.bfloat16)
    return bool(fused_layers)


def _projection_plans_for(base, fused_projections, dtype: torch.dtype, selected: int, fingerprint=None):
    """Per-layer projection plans, or None for the modules' own linear layers.
    Default (None): on for fp16/bf16 caches when the selected rows fit one
    kvr_linear_multi launch (at most 64); fp32 has no such kernel.
    ``fingerprint`` (what _qualify returned for this call): when the plans were
    built for the same module tree they are reused without per-layer checks."""
    if fused_projections is None:
        fused_projections = dtype in (torch.float16, torch.bfloat16) and selected <= _projection.MAX_ROWS
    if not fused_projections or dtype not in (torch.float16, torch.bfloat16) or selected > _projection.MAX_ROWS:
        return None
    return _model_plans(base, fingerprint)


def _model_plans(base, fingerprint=None):
    """One _LayerPlans or None per decoder layer of ``base``."""
    if fingerprint is not None:
        with _PLAN_LOCK:
            cached = _MODEL_PLANS.get(base)
        if cached is not None and cached[0] is fingerprint:
            return cached[1]
    plans = _PlanList(_layer_plans(layer) for layer in base.layers)
    if fingerprint is not None:
        with _PLAN_LOCK:
            _MODEL_PLANS[base] = (fingerprint, plans)
    return plans


def _one_geometry(plans) -> tuple | None:
    """The geometry (_set_geometry) that all of ``plans`` share, or None. Kept with a plan
    list, as the weights it was built from are."""
    geometry = getattr(plans, "geometry", None)
    if geometry is None:
        found = {p.geometry for p in plans}
        geometry = found.pop() if len(found) == 1 else None
        if isinstance(plans, _PlanList):
            plans.geometry = geometry
    return geometry


def _native_layers_for(native_layers, base, plans, fused_epilogue: bool, fused_layers: bool, launcher=None):
    """Whether every layer runs as one kvr_decoder_layer call. Default (None): yes
    when the projection plans, fused epilogue and fused layer ops are all in use
    and every layer has a native descriptor and the same attention scale. One
    refresh descriptor gives the shapes of all layers, so layers of several
    widths, or of other heads than the cache's (``launcher``), run as modules."""
    possible = (plans is not None and fused_epilogue and fused_layers
                and all(p is not None and p.desc is not None for p in plans)
                and _one_geometry(plans) is not None
                and (launcher is None or _one_geometry(plans)[:3] == (
                    launcher.q_heads * launcher.head_dim, launcher.kv_heads * launcher.head_dim, launcher.head_dim))
                and len({float(layer._modules["self_attn"].scaling) for layer in base.layers}) == 1)
    if native_layers is None:
        return possible
    if native_layers and not possible:
        raise ValueError("native_layers=True needs fp16/bf16 plain-linear Llama/Qwen3 layers, <= 64 selected rows, "
                         "and the fused epilogue, layer ops and projections")
    return bool(native_layers)


def _tiled_weights(plans) -> bool:
    """Whether the tiled kernel takes every weight of the plans: k in whole 64s,
    rows in whole 8s, rows neither overlapping nor more than 2^21 elements apart.
    Kept with a plan list, as the weights it was built from are."""
    ok = getattr(plans, "tiled", None)
    if ok is None:
        projections = [q for p in plans for q in (p.qkv, p.q, p.k, p.v, p.o, p.gate_up, p.down) if q is not None]
        ok = all(q.k % 64 == 0 and all(rows % 8 == 0 for rows in q._rows)
                 and all(q.k <= ld <= 1 << 21 for ld in q._ldw) for q in projections)
        if isinstance(plans, _PlanList):
            plans.tiled = ok
    return ok


def _tiled_plans_for(base, launcher: _Launcher, fused_projections, native_layers, fused_epilogue: bool,
                     fused_layers: bool, fingerprint=None):
    """Layer plans of a refresh whose layers run as one kvr_decoder_tiled_forward
    call, or None: more rows than kvr_linear_multi takes, every fusion left on
    (none asked for one by one: ``native_layers=True`` stays an error here),
    layers with native descriptors, weights that kernel takes, and a size at which
    it is not slower than the modules' library GEMMs. Measured per call in bf16 at
    65 to 15104 rows of hidden sizes 1024 to 8192 (fp16 within 2% of it): 1.5 to
    5.8x faster at 65 rows, 1.1 to 4.6x at 512, 0.97 to 2.7x at 2048, 0.95 to 1.25x
    above for up to 5120 wide (1.07x on average). At 8192 wide it runs at 0.95 to
    1.11x from 4096 rows on, level on average: there the modules stay."""
    if (native_layers is not None or fused_projections not in (None, True) or not fused_epilogue or not fused_layers
            or launcher.n_sel <= _projection.MAX_ROWS or launcher.dtype_code == _native.DTYPE_CODES[torch.float32]):
        return None
    plans = _model_plans(base, fingerprint)
    if not _native_layers_for(None, base, plans, True, True, launcher):
        return None
    if _one_geometry(plans)[3] >= _TILED_WIDE and launcher.n_sel >= _TILED_WIDE_ROWS:
        return None
    return plans if launcher.n_sel <= _TILED_MAX_ROWS and _tiled_weights(plans) else None


# int64 word offsets of the cache fields in kvr_layer_desc (a multiple of 8 bytes long)
_DESC_K = _native.LayerDesc.cache_k.offset // 8
_DESC_V = _native.LayerDesc.cache_v.offset // 8
_DESC_STRIDES = _native.LayerDesc.cache_strides.offset // 8
if ctypes.sizeof(_native.LayerDesc) % 8 or (_native.LayerDesc.cache_k.offset | _native.LayerDesc.cache_v.offset
                                             | _native.LayerDesc.cache_strides.offset) % 8:
    raise RuntimeError("kvr_layer_desc layout is not 8-byte aligned")


def _native_layer_descs(plans, output, layer_count):
    """Per-refresh array of the layers' descriptors with this cache's pointers;
    each layer but the last computes the next layer's input norm in its down
    projection's reduction, and the next layer skips it. The cache-independent
    part is built once per plan list and copied."""
    template = getattr(plans, "descs_template", None)
    if template is None or len(template) != layer_count:
        template = (_native.LayerDesc * layer_count)()
        for i in range(layer_count):
            template[i] = plans[i].desc
            desc = template[i]
            if i + 1 < layer_count:
                desc.next_norm, desc.eps_next = plans[i + 1].desc.input_norm, plans[i + 1].desc.eps_input
            desc.input_normed = 1 if i > 0 else 0
        if isinstance(plans, _PlanList):
            plans.descs_template = template
    descs = (_native.LayerDesc * layer_count).from_buffer_copy(template)
    # the per-layer cache fields through one int64 view of the descriptor array
    words = np.frombuffer(descs, dtype=np.int64).reshape(layer_count, -1)
    layers = output.layers
    same = uniform_layers(layers)
    if same is not None and len(same[0]) == 8 * layer_count:  # one layout: addresses from one pass, shared strides
        k_raw, v_raw, first = same
        words[:, _DESC_K] = np.frombuffer(k_raw, dtype=np.int64)
        words[:, _DESC_V] = np.frombuffer(v_raw, dtype=np.int64)
        words[:, _DESC_STRIDES:_DESC_STRIDES + 6] = first.stride()[1:] * 2
        return descs
    words[:, _DESC_K] = [layer.keys.data_ptr() for layer in layers]
    words[:, _DESC_V] = [layer.values.data_ptr() for layer in layers]
    words[:, _DESC_STRIDES:_DESC_STRIDES + 6] = [layer.keys.stride()[1:] + layer.values.stride()[1:] for layer in layers]
    return descs


def _native_inputs(base, d, edited_ids_t, positions):
    """(hidden, cos, sin) of the selected rows from ONE kvr_refresh_inputs launch:
    the embedding rows and the rotary tables the model's own modules would
    produce (a plain nn.Embedding and the default-RoPE rotary module, whose
    fp32 operations the kernel repeats: bit-identical tables). None when the
    modules are not of that plain form; the caller then runs them."""
    embed, rotary = base.embed_tokens, base.rotary_emb
    weight = embed.__dict__["_parameters"].get("weight")
    inv_freq = rotary.__dict__["_buffers"].get("inv_freq")
    if (type(embed) is not torch.nn.Embedding or embed.max_norm is not None or weight is None
            or _native.DTYPE_CODES.get(weight.dtype) != d.dtype or weight.ndim != 2 or weight.stride(1) != 1
            or int(weight.shape[1]) != d.hidden or inv_freq is None or 2 * inv_freq.numel() != d.head_dim
            or type(rotary).__name__ not in ("LlamaRotaryEmbedding", "Qwen3RotaryEmbedding")):
        return None
    inv_freq = inv_freq.to(device=weight.device, dtype=torch.float32).contiguous()
    n, hidden_size, head_dim = int(d.rows), int(d.hidden), int(d.head_dim)
    buf = torch.empty(n * (hidden_size + 2 * head_dim), dtype=weight.dtype, device=weight.device)
    hidden = buf[:n * hidden_size].view(1, n, hidden_size)
    cos = buf[n * hidden_size:n * (hidden_size + head_dim)].view(1, n, head_dim)
    sin = buf[n * (hidden_size + head_dim):].view(1, n, head_dim)
    ids = edited_ids_t[0]
    if ids.stride(0) != 1:
        ids = ids.contiguous()
    status = _native.lib().kvr_refresh_inputs(
        ids.data_ptr(), 1 if ids.dtype == torch.int32 else 0, int(ids.shape[0]), positions.data_ptr(), n,
        weight.data_ptr(), int(weight.shape[0]), int(weight.stride(0)), hidden_size, hidden.data_ptr(), hidden_size,
        inv_freq.data_ptr(), head_dim, float(getattr(rotary, "attention_scaling", 1.0)), cos.data_ptr(),
        sin.data_ptr(), d.dtype, _native.stream_handle(weight.device))
    _native.check(status, "kvr_refresh_inputs")
    return hidden, cos, sin


def _native_refresh(base, launcher: _Launcher, plans, output, layer_count: int, edited_ids_t, positions,
                    tiled: bool = False) -> None:
    """The packed forward as ONE kvr_decoder_forward (or, for more than 64 rows,
    kvr_decoder_tiled_forward) call over all layers.

    One kvr_refresh_inputs launch makes the selected rows' input hidden states
    and cos/sin tables (what the model's embedding and rotary modules compute in
    LlamaModel/Qwen3Model.forward, transformers 5.15.0 modeling_llama.py:377-398,
    bit for bit; other module forms run the modules); then every decoder layer
    runs as kvr_decoder_layer -- the same kernels with the same arguments as the
    Python-dispatched fused shells, so the cache is bit-identical. The final
    norm is skipped: the refresh consumes only the K/V the layers scatter.
    """
    first = base.layers[0]
    native = _NativeForward(launcher, int(first.mlp.down_proj.weight.shape[0]),
                            int(first.mlp.gate_proj.weight.shape[0]), float(first.self_attn.scaling), tiled)
    descs = _native_layer_descs(plans, output, layer_count)
    inputs = _native_inputs(base, native.desc, edited_ids_t, positions)
    if inputs is None:
        hidden = base.embed_tokens(edited_ids_t.index_select(1, positions)).contiguous()
        native.bind_tables(base.rotary_emb(hidden, positions.unsqueeze(0)))
    else:
        hidden, cos, sin = inputs
        native.bind_tables((cos, sin))
    d = native.desc
    if hidden.shape != (1, d.rows, d.hidden) or _native.DTYPE_CODES.get(hidden.dtype) != d.dtype:
        raise RuntimeError("packed native hidden-state geometry/dtype drifted")
    name = "kvr_decoder_tiled_forward" if tiled else "kvr_decoder_forward"
    status = getattr(_native.lib(), name)(descs, layer_count, ctypes.byref(d), hidden.data_ptr(), native.stream)
    _native.check(status, name)


def _refresh_into(shim, output, edited_ids_t, host_plan: IndexedPlan, layer_count: int,
                  attention_backend: str, writeback_backend: str, fused_epilogue: bool = True,
                  fused_layers: bool | None = None, fused_projections: bool | None = None,
                  native_layers: bool | None = None, qualified=(None, False)) -> None:
    """Run the packed forward, scattering into the caller-owned ``output`` cache
    (``qualified``: what _qualify returned for this call). With forward hooks
    present the projections, norms and layers run as the modules themselves
    (the fused kernels would skip the hooks); asking for them then is an error."""
    fingerprint, forward_hooked = qualified
    if forward_hooked:
        if fused_layers or fused_projections or native_layers:
            raise ValueError("module forward hooks need the module path: fused_layers, fused_projections and "
                             "native_layers must not be requested")
        fused_layers = fused_projections = native_layers = False
    base = shim._base_transformer(shim.generator)
    key0 = layer_kv(output, 0)[0]
    # the plan and the attention schedule _launcher asks for, in one upload
    device_plan = host_plan.to(edited_ids_t.device, attention=(
        int(base.config.num_attention_heads), int(key0.shape[1]), int(key0.shape[3]), key0.dtype,
        _rounded_probabilities(key0.dtype)))
    positions = device_plan.positions
    launcher = _launcher(device_plan, base.config, key0)
    plans = _projection_plans_for(base, fused_projections, key0.dtype, device_plan.selected_count, fingerprint)
    fused_layers = _fused_layers_for(fused_layers, key0.dtype)
    if _native_layers_for(native_layers, base, plans, fused_epilogue, fused_layers, launcher):
        _native_refresh(base, launcher, plans, output, layer_count, edited_ids_t, positions)
        return
    tiled_plans = _tiled_plans_for(base, launcher, fused_projections, native_layers, fused_epilogue, fused_layers,
                                   fingerprint)
    if tiled_plans is not None:
        _native_refresh(base, launcher, tiled_plans, output, layer_count, edited_ids_t, positions, tiled=True)
        return
    context = _PackedContext(positions, host_plan.logical_length, attention_backend, device_plan, launcher)
    native_view = _make_native_view(base, fused_epilogue, fused_layers, plans)
    layers = [_PackedLayer(*layer_kv(output, i), context, writeback_backend) for i in range(layer_count)]
    cache = Cache(layers=layers)
    result = native_view(input_ids=edited_ids_t.index_select(1, positions), position_ids=positions.unsqueeze(0),
                         past_key_values=cache, use_cache=True, return_dict=True, sur_packed_context=context)
    if result.past_key_values is not cache or not all(layer.updated for layer in layers):
        raise RuntimeError("native packed forward did not update each cache layer exactly once")


@torch.no_grad()
def packed_interval_repair(shim: Any, base_cache: Any, edited_ids_t: torch.Tensor,
                           intervals: Sequence[tuple[int, int]], *, attention_backend: str = "sdpa",
                           writeback_backend: str = "torch", plan: Any = None, fused_epilogue: bool = True,
                           fused_layers: bool | None = None, fused_projections: bool | None = None,
                           native_layers: bool | None = None) -> tuple[Any, dict[str, Any]]:
    """Recompute sorted selected rows in one native layer-major forward.

    Same signature, validation order, receipt and ownership contract as the
    reference executor (packed_cache.py:225-298), including its default backend
    names; every accepted backend name runs the gfx950 HIP kernels (the receipt
    records "hip"). ``plan`` optionally supplies a reusable host IndexedPlan for
    exactly these intervals and length. The borrowed ``base_cache`` is never
    mutated: a nonempty repair returns an independently owned cache (one
    libkvrepair copy launch), an empty one returns ``base_cache`` itself.
    ``fused_epilogue`` (default) fuses each layer's fresh-row RoPE with the
    K/V scatter (one launch); False runs the native RoPE ops and the registered
    cache-update/attention plugin points. Both give bit-identical caches.
    ``fused_layers`` runs each decoder layer's RMSNorms (with the residual
    add) and MLP activation as single launches; its fp32 mean of squares can
    differ from the eager chain by an ulp, so the default (None) fuses them for
    fp16/bf16 caches only. ``fused_projections`` runs each layer's projections
    as kvr_linear_multi launches (q/k/v in one, gate/up with the SiLU gate in
    one; fp32 accumulation rounded once, like the library GEMM up to summation
    order); the default (None) uses them for fp16/bf16 caches with at most 64
    selected rows, where the modules' GEMMs are weight-streaming bound, and runs
    more rows through kvr_tiled_linear_multi's kernel inside one native forward
    (_tiled_plans_for). ``native_layers`` runs the whole packed forward as one kvr_decoder_forward
    call after the model's embedding and rotary modules (the same kernels with
    the same arguments, bit-identical to the Python-dispatched fused shells);
    the default (None) does so whenever the three fusions above are active.
    """
    attention_backend, writeback_backend = _check_backends(attention_backend, writeback_backend)
    _check_ids(edited_ids_t)
    length = int(edited_ids_t.shape[1])
    layer_count = _validate_cache(base_cache, length)
    intervals = _validate_intervals(intervals, length)
    selected = tuple(p for start, end in intervals for p in range(start, end))
    if plan is not None:
        if not isinstance(plan, IndexedPlan) or tuple(plan.positions) != selected or plan.logical_length != length:
            raise ValueError("supplied IndexedPlan must match exact selected positions and cache length")
    receipt = _receipt(intervals, selected, length, layer_count, attention_backend, writeback_backend)
    if not selected:
        return base_cache, receipt
    qualified = _qualify(shim, edited_ids_t, base_cache, attention_backend, writeback_backend)
    host_plan = plan if plan is not None else IndexedPlan(selected, length)
    from ..cache import clone_cache

    output = clone_cache(base_cache)
    _refresh_into(shim, output, edited_ids_t, host_plan, layer_count, attention_backend, writeback_backend,
                  bool(fused_epilogue), fused_layers, fused_projections, native_layers, qualified)
    return output, receipt


@torch.no_grad()
def packed_refresh_owned_(shim: Any, owned_cache: Any, edited_ids_t: torch.Tensor,
                          intervals: Sequence[tuple[int, int]], *, plan: Any = None,
                          fused_epilogue: bool = True, fused_layers: bool | None = None,
                          fused_projections: bool | None = None, native_layers: bool | None = None) -> dict[str, Any]:
    """Packed refresh that scatters IN PLACE into a cache the caller owns.

    For a cache the caller has just built and nobody else references (the
    shifted cache of build_halo_cache inside repair_after_deletion) the
    ownership copy of packed_interval_repair is redundant; this entry skips it.
    The result equals packed_interval_repair's output bit for bit.
    """
    _check_ids(edited_ids_t)
    length = int(edited_ids_t.shape[1])
    layer_count = _validate_cache(owned_cache, length)
    intervals = _validate_intervals(intervals, length)
    selected = tuple(p for start, end in intervals for p in range(start, end))
    if plan is not None:
        if not isinstance(plan, IndexedPlan) or tuple(plan.positions) != selected or plan.logical_length != length:
            raise ValueError("supplied IndexedPlan must match exact selected positions and cache length")
    receipt = _receipt(intervals, selected, length, layer_count, "hip", "hip")
    receipt["base_cache_ownership"] = "owned_in_place"
    if not selected:
        return receipt
    qualified = _qualify(shim, edited_ids_t, owned_cache, "hip", "hip")
    host_plan = plan if plan is not None else IndexedPlan(selected, length)
    _refresh_into(shim, owned_cache, edited_ids_t, host_plan, layer_count, "hip", "hip", bool(fused_epilogue),
                  fused_layers, fused_projections, native_layers, qualified)
    return receipt
