"""The streaming projections' walk over k (kvr_linear_multi, at most 64 rows).
Without a K split, over weight rows of whole 2048 k or at least 6656, tiles 1344
streamed rows apart start at different 256-k chunks and come round, so some start
at a last chunk that k leaves ragged; all other launches start at k 0."""

from __future__ import annotations

import pytest
import torch

from test_gpu_operators import assert_linear_close, bits_equal, exact_linear, ulp_distance
from test_gpu_tiled import assert_gate_close

# (n, k, splits). From k 0: one ragged chunk; three, the last 8, 8 and 248 k long; a slice of two chunks and a ragged
# second slice; more than 256 blocks (128-k chunks), the last chunk 8 and 248 k long. Staggered, over 128-k chunks
# (more than 256 blocks) and, over 28672 rows of blocks of seven waves, 256-k ones: eight whole chunks, starts 0 to 7
# and round again; a last chunk 8 and 120 k long, reached in the middle
SHAPES = [(1400, 200, 1), (5400, 520, 1), (4040, 520, 1), (4100, 760, 1), (6000, 1288, 2), (16400, 520, 1),
          (17000, 1016, 1), (16400, 2048, 1), (17000, 6664, 1), (16400, 6904, 1), (28672, 2048, 1), (28672, 6664, 1)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("rows", [3, 64])
def test_every_start_of_the_walk_gives_the_product(gpu_device, dtype, shape, rows):
    from kv_cache_repair_amd import _native
    from kv_cache_repair_amd.kernels import projection

    n, k, splits = shape
    assert _native.lib().kvr_linear_splits(rows, n, k) == splits
    torch.manual_seed(n + k)
    x = torch.randn(1, rows, k + 8, device=gpu_device).to(dtype)[..., :k]
    w = (torch.randn(n, k + 8, device=gpu_device) * 0.03).to(dtype)[:, 8:]
    y = projection.linear(x, w)
    assert_linear_close(y, x, w)
    assert bits_equal(projection.linear(x, w), y)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,k", [(2760, 520), (8200, 776), (8200, 2048), (14336, 2048), (8200, 6664), (14336, 6904)])
def test_every_start_of_the_gated_walk(gpu_device, dtype, n, k):
    """Within the two roundings of the projections and that of the gate, as for the other gated shapes."""
    from kv_cache_repair_amd.kernels import projection

    torch.manual_seed(n)
    x = torch.randn(1, 37, k, device=gpu_device).to(dtype)
    gate, up = ((torch.randn(n, k, device=gpu_device) * 0.05).to(dtype) for _ in range(2))
    y = projection.silu_gate_linear(x, gate, up)
    eager = torch.nn.functional.silu(exact_linear(x, gate)) * exact_linear(x, up)
    assert_gate_close(y[0], x[0], gate, up)
    assert (ulp_distance(y, eager) <= 2).float().mean().item() >= 0.99
