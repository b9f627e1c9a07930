"""Packed attention over every row-group size of the head-pair kernel: one and
two pairs of query heads per KV head, groups of 16, 32 and 64 rows, whole and
ragged groups, chunked and single key ranges, against the fp64 oracle."""

from __future__ import annotations

import ctypes
import random

import pytest
import torch

from test_gpu_operators import assert_attention_close, attention_problem, oracle_attention

H_GROUP_ROWS = 16

# query heads, KV heads, head dim, rows, keys, rows per group the schedule picks
CASES = [
    (4, 2, 64, 5, 90, 16), (4, 2, 128, 16, 700, 16), (8, 4, 64, 47, 600, 16),
    (16, 8, 128, 33, 9000, 32), (16, 8, 64, 300, 4000, 32), (8, 4, 128, 282, 5000, 32), (12, 2, 128, 200, 9000, 32),
    (16, 8, 64, 500, 6001, 64), (8, 4, 128, 1400, 3000, 64), (4, 2, 64, 2100, 2200, 64), (24, 4, 128, 700, 900, 64),
    (8, 2, 128, 40, 3000, 16), (8, 2, 64, 640, 4000, 16), (16, 4, 128, 600, 9000, 64), (32, 8, 64, 290, 6000, 64),
]


def spread(rows, keys, seed):
    """Runs of rows over the whole range, the first and the last key among them."""
    rng = random.Random(seed)
    return sorted({0, keys - 1, *rng.sample(range(1, keys - 1), rows - 2)})


def group_rows(positions, keys, heads, kv_heads, dim, flags=0):
    from kv_cache_repair_amd import _native

    lib, pos = _native.lib(), (ctypes.c_int64 * len(positions))(*positions)
    args = (pos, len(positions), keys, heads, kv_heads, dim, 2, 0, flags)
    need = lib.kvr_attention_schedule_ex(*args, None, 0)
    buf = (ctypes.c_int32 * need)()
    assert lib.kvr_attention_schedule_ex(*args, buf, need) == need
    return buf[H_GROUP_ROWS]


@pytest.mark.parametrize("case", CASES)
def test_schedule_picks_the_group_size(case):
    heads, kv_heads, dim, rows, keys, expected = case
    assert group_rows(spread(rows, keys, rows), keys, heads, kv_heads, dim) == expected


@pytest.mark.parametrize("heads,kv_heads,dim,rows,keys,flags", [
    (16, 4, 64, 161, 20682, 1), (64, 8, 128, 455, 1248, 1), (32, 8, 128, 235, 7181, 0), (8, 2, 64, 867, 4522, 0),
    (8, 2, 64, 1143, 2692, 1), (2, 1, 128, 250, 9083, 0), (4, 2, 128, 57, 26798, 0)])
def test_schedule_keeps_16_rows_where_larger_groups_measured_slower(heads, kv_heads, dim, rows, keys, flags):
    """The last rows of the keys, 6 to 18% slower in 32- or 64-row groups than in 16."""
    assert group_rows(range(keys - rows, keys), keys, heads, kv_heads, dim, flags) == 16


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", CASES)
def test_every_group_size_agrees_with_the_fp64_oracle(gpu_device, case, dtype):
    from kv_cache_repair_amd.kernels import indexed_attention as ia

    heads, kv_heads, dim, rows, keys, _ = case
    positions = spread(rows, keys, rows)
    q, k, v = attention_problem(gpu_device, dtype, heads, kv_heads, rows, keys, dim, ("token_major",) * 3, seed=rows)
    plan = ia.IndexedPlan(positions, keys).to(gpu_device)
    actual = ia.indexed_causal_attention(q, k, v, plan)
    assert torch.isfinite(actual).all()
    # the oracle takes rows one by one: both ends, the rows around tile and group edges, some others
    edges = {0, 1, rows - 2, rows - 1, *(e + d for e in (16, 32, 64, 128) for d in (-1, 0)), *range(5, rows, 97)}
    picked = sorted(r for r in edges if 0 <= r < rows)
    assert_attention_close(actual[:, :, picked], oracle_attention(q[:, :, picked], k, v, [positions[r] for r in picked]))
    assert torch.equal(actual, ia.indexed_causal_attention(q, k, v, plan))


@pytest.mark.gpu
@pytest.mark.parametrize("layouts", [("sparse", "token_major", "token_major"), ("token_major", "padded", "sparse")])
@pytest.mark.parametrize("case", [CASES[3], CASES[4], CASES[6], CASES[7]])
def test_group_sizes_on_layouts_of_the_generic_kernel(gpu_device, case, layouts):
    """The schedule is made for a geometry, before any strides are seen: rows that
    the matrix kernels do not read take its 32- and 64-row groups to the generic one."""
    from kv_cache_repair_amd.kernels import indexed_attention as ia

    heads, kv_heads, dim, rows, keys, _ = case
    positions = spread(rows, keys, rows)
    q, k, v = attention_problem(gpu_device, torch.bfloat16, heads, kv_heads, rows, keys, dim, layouts, seed=rows)
    actual = ia.indexed_causal_attention(q, k, v, ia.IndexedPlan(positions, keys).to(gpu_device))
    picked = sorted({0, 1, 15, 16, 31, 32, rows - 2, rows - 1} & set(range(rows)))
    assert_attention_close(actual[:, :, picked], oracle_attention(q[:, :, picked], k, v, [positions[r] for r in picked]))
    assert_attention_close(actual[:, :, rows // 2:rows // 2 + 8],
                           oracle_attention(q[:, :, rows // 2:rows // 2 + 8], k, v, positions[rows // 2:rows // 2 + 8]))
    plan = ia.IndexedPlan(positions, keys).to(gpu_device)
    dense = ia.indexed_causal_attention(*(t.contiguous() for t in (q, k, v)), plan)
    # the same sums in another order, rounded to bf16
    torch.testing.assert_close(actual, dense, rtol=2 ** -6, atol=2 ** -9)
