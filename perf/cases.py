"""The work that is timed: refreshes of a stale KV cache and the operators a program calls by themselves.

Kinds of case, each through the entry points that a user's program calls:

``refresh``    the repair of one prompt after an edit, as the API runs it once the support is chosen:
               ``build_halo_cache`` (prefix copy, rotated suffix), then ``packed_refresh_owned_``.
``attention``  one layer of ``indexed_causal_attention``.
``scatter``    one layer of ``indexed_kv_scatter_``.
``rotate``     ``shifted_suffix_keys`` of one layer.
``build``      ``build_halo_cache`` alone: a repair at a budget of 0%.
``linear``     one projection of a few rows (``linear`` or ``silu_gate_linear``).
``score``      ``dense_query_relevance_scores`` of a prompt, which ranks tokens for a budget.

Shapes are the benchmark's (an 8B Llama and an 8B Qwen3 decoder) or generic; a decoder of fewer layers stands
for the same call on the whole model where the whole one would only repeat the same layers. The vocabulary is
small: no case reads more of the embedding table than the rows of its prompt.
"""

from __future__ import annotations

import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "budgeted-kv-cache-repair_amd"))

from kv_cache_repair_amd.cache import (OperatorShim, build_halo_cache, cache_from_tensors,  # noqa: E402
                                       shifted_suffix_keys)
from kv_cache_repair_amd.kernels.indexed_attention import (IndexedPlan, indexed_causal_attention,  # noqa: E402
                                                           indexed_kv_scatter_)
from kv_cache_repair_amd.kernels import packed_cache  # noqa: E402
from kv_cache_repair_amd.kernels.projection import linear, silu_gate_linear  # noqa: E402
from kv_cache_repair_amd.scoring import dense_query_relevance_scores  # noqa: E402

# the model library the executor serves, as the package itself imported it
_hf = packed_cache.transformers

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
FAMILIES = {  # hidden, intermediate, query heads, KV heads, head dim, RoPE base
    "llama": (4096, 14336, 32, 8, 128, 500000.0),
    "qwen3": (4096, 12288, 32, 8, 128, 1000000.0),
}
VOCAB = 32768


def _refresh(name, family, layers, dtype, total, delete_at, delete_span, rows, intervals):
    return {"name": name, "kind": "refresh", "family": family, "layers": layers, "dtype": dtype, "total": total,
            "delete_at": delete_at, "delete_span": delete_span, "rows": rows, "intervals": intervals}


def listed():
    return [
        # the benchmark's headline: an 8k prompt, 64 rows in 16 places, every layer
        _refresh("refresh_llama_8k_64rows", "llama", 32, "bf16", 8192, 2048, 512, 64, 16),
        # the API's default budget, 5% of the retained suffix, on a 2k prompt ...
        _refresh("refresh_llama_2k_71rows", "llama", 32, "bf16", 2048, 512, 128, 71, 4),
        # ... and on the 8k prompt
        _refresh("refresh_llama_8k_282rows", "llama", 32, "bf16", 8192, 2048, 512, 282, 16),
        # 10% of a 2k prompt in fp16
        _refresh("refresh_fp16_2k_141rows", "llama", 16, "fp16", 2048, 512, 128, 141, 6),
        # a long prompt at the default budget, with per-head norms
        _refresh("refresh_qwen3_32k_1383rows", "qwen3", 8, "bf16", 32768, 4096, 1024, 1383, 32),
        # a budget of 100%: the whole suffix of a 16k prompt
        _refresh("refresh_llama_16k_15104rows", "llama", 4, "bf16", 16384, 1024, 256, 15104, 1),
        # one attention layer as a program that owns its decoder calls it: few rows over a long cache
        {"name": "attention_8k_64rows", "kind": "attention", "dtype": "bf16", "q_heads": 32, "kv_heads": 8, "dim": 128,
         "keys": 7680, "rows": 64, "intervals": 16},
        # ... and an odd number of rows with the smaller head
        {"name": "attention_fp16_d64_16k_805rows", "kind": "attention", "dtype": "fp16", "q_heads": 16, "kv_heads": 8,
         "dim": 64, "keys": 16128, "rows": 805, "intervals": 19},
        # fresh rows of one layer written into its cache: the smallest call
        {"name": "scatter_8k_282rows", "kind": "scatter", "dtype": "bf16", "kv_heads": 8, "dim": 128, "keys": 7680,
         "rows": 282, "intervals": 16},
        # position shift alone
        {"name": "build_llama_16k", "kind": "build", "family": "llama", "layers": 16, "dtype": "bf16", "total": 16384,
         "delete_at": 1024, "delete_span": 256},
        # an MLP's gated front half over a few rows
        {"name": "gate_up_37rows", "kind": "linear", "gated": True, "dtype": "bf16", "rows": 37, "n": 14336, "k": 4096},
        # ranking a long prompt's tokens before any repair below 100%
        {"name": "score_32k", "kind": "score", "dtype": "bf16", "tokens": 31744, "query": 12, "hidden": 4096},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choices(["refresh", "attention", "scatter", "rotate", "build", "linear", "score"],
                       [10, 3, 1, 1, 1, 2, 1])[0]
    dtype = rng.choices(["bf16", "fp16"], [4, 1])[0]
    family = rng.choice(["llama", "qwen3"])
    if kind in ("refresh", "build"):
        total = _log_int(rng, 1024, 32768)
        span = _log_int(rng, 16, total // 8)
        at = rng.randint(total // 16, total // 3)
        suffix = total - at - span
        case = {"kind": kind, "family": family, "layers": rng.choice([4, 8, 16]), "dtype": dtype, "total": total,
                "delete_at": at, "delete_span": span}
        if kind == "build":
            return case
        rows = min(suffix // 2, max(3, math.ceil(suffix * math.exp(rng.uniform(math.log(0.005), math.log(0.2))))))
        rows = min(rows, 4096)
        case["layers"] = min(case["layers"], 4 if rows > 1536 else 16)
        return {**case, "rows": rows, "intervals": rng.randint(1, max(1, min(32, rows // 3)))}
    if kind in ("attention", "scatter"):
        dim = rng.choices([128, 64], [3, 1])[0]
        kv_heads = rng.choice([4, 8])
        keys = _log_int(rng, 1024, 32768)
        rows = _log_int(rng, 3, min(2048, keys // 3))
        case = {"kind": kind, "dtype": dtype, "kv_heads": kv_heads, "dim": dim, "keys": keys, "rows": rows,
                "intervals": rng.randint(1, max(1, min(32, rows // 3)))}
        return {**case, "q_heads": kv_heads * rng.choice([2, 4])} if kind == "attention" else case
    if kind == "rotate":
        return {"kind": kind, "family": family, "dtype": dtype, "tokens": _log_int(rng, 512, 32768),
                "shift": -_log_int(rng, 1, 2048)}
    if kind == "linear":
        gated = rng.random() < 0.4
        n, k = rng.choice([(14336, 4096), (12288, 4096)] if gated else
                          [(4096, 4096), (1024, 4096), (4096, 14336), (4096, 12288)])
        return {"kind": kind, "gated": gated, "dtype": dtype, "rows": rng.randint(1, 64), "n": n, "k": k}
    return {"kind": kind, "dtype": dtype, "tokens": _log_int(rng, 1024, 32768), "query": rng.randint(3, 40),
            "hidden": 4096}


# ----------------------------------------------------------------------------- inputs
def _device():
    return torch.device("cuda", 0)


def _generator(seed):
    return torch.Generator(device=_device()).manual_seed(int(seed))


def _fill(tensor, std, gen):
    flat = tensor.view(-1)
    for start in range(0, flat.numel(), 1 << 28):
        flat[start:start + (1 << 28)].normal_(0.0, std, generator=gen)


def _model(family, layers, dtype, positions, gen):
    """A decoder of that shape as its library initialises it: weights ~ N(0, 0.02), norms 1, default RoPE."""
    hidden, mlp, hq, hkv, dim, theta = FAMILIES[family]
    common = dict(vocab_size=VOCAB, hidden_size=hidden, intermediate_size=mlp, num_hidden_layers=layers,
                  num_attention_heads=hq, num_key_value_heads=hkv, head_dim=dim, rope_theta=theta,
                  max_position_embeddings=positions, tie_word_embeddings=True)
    if family == "qwen3":
        config, ctor = _hf.Qwen3Config(layer_types=["full_attention"] * layers, **common), _hf.Qwen3ForCausalLM
    else:
        config, ctor = _hf.LlamaConfig(**common), _hf.LlamaForCausalLM
    before = torch.get_default_dtype()
    torch.set_default_dtype(DTYPES[dtype])
    try:
        with torch.device("meta"):
            model = ctor(config)
    finally:
        torch.set_default_dtype(before)
    model = model.to_empty(device=_device()).eval().requires_grad_(False)
    model.tie_weights()
    for name, param in model.named_parameters():
        if name.endswith("norm.weight"):
            param.data.fill_(1.0)
        else:
            _fill(param.data, 0.02, gen)
    rotary = model.model.rotary_emb
    inv_freq, rotary.attention_scaling = rotary.compute_default_rope_parameters(config, _device())
    rotary.inv_freq = inv_freq.to(device=_device(), dtype=torch.float32)
    rotary.original_inv_freq = rotary.inv_freq.clone()
    return model


def _intervals(rng, start, end, rows, count):
    """`count` runs of rows that touch nowhere in [start, end), `rows` in all."""
    base, extra = divmod(rows, count)
    lengths = [base + (i < extra) for i in range(count)]
    rng.shuffle(lengths)
    spare = end - start - rows - (count - 1)
    gaps = sorted(rng.randint(0, spare) for _ in range(count))
    at, before, out = start, 0, []
    for i, (length, gap) in enumerate(zip(lengths, gaps)):
        at += gap - before + (i > 0)
        before = gap
        out.append((at, at + length))
        at += length
    return out


def _rows(case, seed):
    intervals = _intervals(random.Random(seed), 0, case["keys"], case["rows"], case["intervals"])
    return tuple(p for s, e in intervals for p in range(s, e))


def _normal(shape, dtype, gen, std=1.0):
    out = torch.empty(shape, dtype=DTYPES[dtype], device=_device())
    _fill(out, std, gen)
    return out


def prepare(case, seed):
    kind, gen = case["kind"], _generator(seed)
    if kind in ("refresh", "build"):
        total, at, span = case["total"], case["delete_at"], case["delete_span"]
        _, _, _, hkv, dim, _ = FAMILIES[case["family"]]
        if kind == "refresh":
            model = _model(case["family"], case["layers"], case["dtype"], total, gen)
        else:  # the build reads the model's rotary frequencies and table size only
            model = _model(case["family"], 1, case["dtype"], total, gen)
        old = cache_from_tensors([tuple(_normal((1, hkv, total, dim), case["dtype"], gen) for _ in range(2))
                                  for _ in range(case["layers"])])
        old_ids = torch.randint(0, VOCAB, (1, total), generator=torch.Generator().manual_seed(int(seed)))
        old_ids[0, at] = (old_ids[0, at + span] + 1) % VOCAB  # the edit begins where it is said to
        new_ids = torch.cat((old_ids[:, :at], old_ids[:, at + span:]), dim=1)
        state = {"kind": kind, "shim": OperatorShim(model), "old": old, "old_ids": old_ids, "new_ids": new_ids}
        if kind == "refresh":
            state["device_ids"] = new_ids.to(_device())
            state["intervals"] = _intervals(random.Random(seed), at, total - span, case["rows"], case["intervals"])
        return state
    if kind == "rotate":
        _, _, _, hkv, dim, _ = FAMILIES[case["family"]]
        return {"kind": kind, "shim": OperatorShim(_model(case["family"], 1, case["dtype"], case["tokens"], gen)),
                "key": _normal((1, hkv, case["tokens"], dim), case["dtype"], gen), "shift": case["shift"]}
    if kind in ("attention", "scatter"):
        hkv, dim, keys, rows = case["kv_heads"], case["dim"], case["keys"], case["rows"]
        plan = IndexedPlan(_rows(case, seed), keys).to(_device())
        k, v = (_normal((1, hkv, keys, dim), case["dtype"], gen) for _ in range(2))
        state = {"kind": kind, "plan": plan, "k": k, "v": v}
        if kind == "attention":  # queries lie token by token, as a projection leaves them
            state["q"] = _normal((1, rows, case["q_heads"], dim), case["dtype"], gen).transpose(1, 2)
        else:
            state["fresh_k"], state["fresh_v"] = (
                _normal((1, rows, hkv, dim), case["dtype"], gen).transpose(1, 2) for _ in range(2))
        return state
    if kind == "linear":
        weights = [_normal((case["n"], case["k"]), case["dtype"], gen, 0.02) for _ in range(1 + case["gated"])]
        return {"kind": kind, "weights": weights, "x": _normal((1, case["rows"], case["k"]), case["dtype"], gen)}
    table = torch.nn.Embedding(VOCAB, case["hidden"], device=_device(), dtype=DTYPES[case["dtype"]])
    table.requires_grad_(False)
    _fill(table.weight.data, 0.02, gen)

    class Model:  # what the scorer asks of a model
        @staticmethod
        def get_input_embeddings():
            return table

    rng = random.Random(seed)
    return {"kind": kind, "shim": OperatorShim(Model()),
            "ids": torch.randint(0, VOCAB, (1, case["tokens"]), generator=gen, device=_device()),
            "query": [rng.randrange(VOCAB) for _ in range(case["query"])]}


# ----------------------------------------------------------------------------- one pass
def run(state):
    kind = state["kind"]
    if kind in ("refresh", "build"):
        cache, _ = build_halo_cache(state["shim"], state["old"], state["old_ids"], state["new_ids"], 0)
        if kind == "refresh":
            packed_cache.packed_refresh_owned_(state["shim"], cache, state["device_ids"], state["intervals"])
        return [t for layer in cache.layers for t in (layer.keys, layer.values)]
    if kind == "rotate":
        return shifted_suffix_keys(state["shim"], state["key"], state["shift"])
    if kind == "attention":
        return indexed_causal_attention(state["q"], state["k"], state["v"], state["plan"])
    if kind == "scatter":
        indexed_kv_scatter_(state["k"], state["v"], state["fresh_k"], state["fresh_v"], state["plan"])
        return [state["k"], state["v"]]
    if kind == "linear":
        if len(state["weights"]) == 2:
            return silu_gate_linear(state["x"], *state["weights"])
        return linear(state["x"], state["weights"][0])
    scores, _ = dense_query_relevance_scores(model=state["shim"], edited_input_ids=state["ids"],
                                             query_token_ids=state["query"])
    return np.asarray(scores, dtype=np.float32)


# ----------------------------------------------------------------------------- what a pass cannot do without
def work(case):
    kind = case["kind"]
    if kind in ("refresh", "build"):
        hidden, mlp, hq, hkv, dim, _ = FAMILIES[case["family"]]
        length = case["total"] - case["delete_span"]
        cache = 2 * case["layers"] * hkv * dim * 2
        moved = 2 * length * cache
        if kind == "build":
            return {"bytes": moved, "flops": 0}
        weights = case["layers"] * (hidden * dim * (2 * hq + 2 * hkv) + 3 * hidden * mlp)
        rows, start = case["rows"], case["delete_at"]
        seen = rows * (start + length) / 2  # keys that the rows attend to, on average
        return {"bytes": moved + 2 * weights + 2 * rows * hidden,
                "flops": 2 * rows * weights + case["layers"] * 4 * hq * dim * seen}
    if kind == "rotate":
        _, _, _, hkv, dim, _ = FAMILIES[case["family"]]
        return {"bytes": 2 * 2 * hkv * dim * case["tokens"], "flops": 0}
    if kind == "attention":
        hq, hkv, dim, keys, rows = (case[n] for n in ("q_heads", "kv_heads", "dim", "keys", "rows"))
        return {"bytes": 2 * dim * (2 * hkv * keys + 2 * hq * rows), "flops": 4 * hq * dim * rows * keys / 2}
    if kind == "scatter":
        return {"bytes": 2 * 2 * 2 * case["kv_heads"] * case["dim"] * case["rows"], "flops": 0}
    if kind == "linear":
        n, k, m = case["n"] * (1 + case["gated"]), case["k"], case["rows"]
        return {"bytes": 2 * (n * k + m * k + m * case["n"]), "flops": 2 * m * n * k}
    tokens, hidden = case["tokens"], case["hidden"]
    rows = VOCAB * (1 - math.exp(-tokens / VOCAB))  # different rows of the table among the prompt's tokens
    return {"bytes": 2 * rows * hidden + 12 * tokens, "flops": 2 * tokens * case["query"] * hidden}


def tolerance(case):
    """Relative to each output as a whole. Of a refresh only the refreshed rows can differ, but through all the
    layers: a quarter of what is stated is what the path is off 64 bits by (0.02 at most in bf16, of a refreshed
    row 0.05 after 32 layers), and an element's own error is up to a fifth of the row's size."""
    kind = case["kind"]
    if kind in ("scatter", "build", "rotate"):
        return "exact" if kind == "scatter" else {"rel": 1e-3, "max": 0.02}
    if kind == "score":
        return {"rel": 4e-6, "max": 1e-4}
    if kind == "linear":
        return {"rel": 4e-3, "max": 0.04}
    if kind == "attention":
        return {"rel": 5e-3, "max": 0.05} if case["dtype"] == "bf16" else {"rel": 6e-4, "max": 6e-3}
    return {"rel": 0.03, "max": 0.8} if case["dtype"] == "bf16" else {"rel": 6e-3, "max": 0.1}


# ----------------------------------------------------------------------------- the same in 64 bits
def _half_turn(x):
    a, b = x.chunk(2, dim=-1)
    return torch.cat((-b, a), dim=-1)


def _rope(x, positions, inv_freq):
    angle = positions.double().unsqueeze(-1) * torch.cat((inv_freq, inv_freq)).double()
    return x * angle.cos() + _half_turn(x) * angle.sin()


def _rms(x, weight, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * weight.double()


def _attend(q, k, v, positions, scale):
    """[heads, rows, dim] over [KV heads, keys, dim], a block of rows at a time."""
    hq, rows, dim = q.shape
    hkv, keys, _ = k.shape
    out = torch.empty_like(q)
    step = max(1, (1 << 27) // (keys * (hq // hkv)))
    at = torch.arange(keys, device=q.device)
    for h in range(hkv):
        heads = slice(h * (hq // hkv), (h + 1) * (hq // hkv))
        kt = k[h].t().contiguous()
        for r in range(0, rows, step):
            last = int(positions[min(r + step, rows) - 1]) + 1
            score = torch.matmul(q[heads, r:r + step], kt[:, :last].contiguous()).mul_(scale)
            score.masked_fill_(at[:last] > positions[r:r + step, None], -math.inf)
            out[heads, r:r + step] = torch.matmul(score.softmax(-1), v[h, :last].contiguous())
    return out


def _shift(state, case):
    at, span, length = case["delete_at"], case["delete_span"], case["total"] - case["delete_span"]
    inv_freq = state["shim"].generator.model.rotary_emb.inv_freq
    out = []
    for layer in state["old"].layers:
        k, v = layer.keys.double(), layer.values.double()
        tail = _rope(k[:, :, at + span:], torch.full((length - at,), -span, device=k.device), inv_freq)
        out.append([torch.cat((k[:, :, :at], tail), dim=2), torch.cat((v[:, :, :at], v[:, :, at + span:]), dim=2)])
    return out


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    state = prepare(case, seed)
    if kind == "scatter":
        indices = torch.tensor(_rows(case, seed), device=_device())
        return [state[n].double().index_copy(2, indices, state["fresh_" + n].double()) for n in ("k", "v")]
    if kind == "attention":
        positions = torch.tensor(_rows(case, seed), device=_device())
        return _attend(state["q"][0].double(), state["k"][0].double(), state["v"][0].double(), positions,
                       case["dim"] ** -0.5)[None]
    if kind == "rotate":
        key = state["key"].double()
        return _rope(key, torch.full((key.shape[2],), state["shift"], device=key.device),
                     state["shim"].generator.model.rotary_emb.inv_freq)
    if kind == "linear":
        out = [torch.matmul(state["x"].double(), w.double().t().contiguous()) for w in state["weights"]]
        return out[0] * torch.sigmoid(out[0]) * out[1] if len(out) == 2 else out[0]
    if kind == "score":
        table = state["shim"].generator.get_input_embeddings().weight.double()
        table = table / table.norm(dim=-1, keepdim=True).clamp_min(1e-12)
        query = torch.tensor(state["query"], device=_device())
        score = torch.matmul(table[state["ids"][0]], table[query].t().contiguous()).amax(-1)
        return score + 0.25 * torch.isin(state["ids"][0], query)
    cache = _shift(state, case)
    if kind == "build":
        return [t for pair in cache for t in pair]
    model = state["shim"].generator.model
    inv_freq = model.rotary_emb.inv_freq
    positions = torch.tensor([p for s, e in state["intervals"] for p in range(s, e)], device=_device())
    x = model.embed_tokens.weight[state["device_ids"][0, positions]].double()
    rows = x.shape[0]
    for layer, (keys, values) in zip(model.layers, cache):
        attn, mlp, eps = layer.self_attn, layer.mlp, model.config.rms_norm_eps

        def project(module, value):
            return torch.matmul(value, module.weight.double().t().contiguous())

        normed = _rms(x, layer.input_layernorm.weight, eps)
        q, k, v = (project(m, normed).view(rows, -1, attn.head_dim).transpose(0, 1)
                   for m in (attn.q_proj, attn.k_proj, attn.v_proj))
        if hasattr(attn, "q_norm"):
            q, k = _rms(q, attn.q_norm.weight, eps), _rms(k, attn.k_norm.weight, eps)
        q, k = _rope(q, positions, inv_freq), _rope(k, positions, inv_freq)
        keys[0, :, positions], values[0, :, positions] = k, v
        seen = _attend(q.contiguous(), keys[0], values[0], positions, attn.head_dim ** -0.5)
        x = x + project(attn.o_proj, seen.transpose(0, 1).reshape(rows, -1))
        normed = _rms(x, layer.post_attention_layernorm.weight, eps)
        gate = project(mlp.gate_proj, normed)
        x = x + project(mlp.down_proj, gate * torch.sigmoid(gate) * project(mlp.up_proj, normed))
    return [t for pair in cache for t in pair]
