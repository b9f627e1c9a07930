"""Every kernel that a projection of more than 64 rows can reach: each block tile,
with its weights streamed (one x tile) or shared by several x tiles, writing whole
sums, split-K partials or the gated product, at rows and features that end inside
a tile, against fp64 products."""

from __future__ import annotations

import ctypes

import pytest
import torch

from test_gpu_operators import assert_linear_close, exact_linear, ulp_distance
from test_gpu_tiled import CONCAT, RESIDUAL, SILU_GATE, assert_gate_close, tiled

# (tile rows, tile columns, streamed) -> rows of x, weight rows (gated: of gate and up together) and k that reach it
TILE_SHAPES = {
    (80, 64, True): {"whole": (76, 5328, 576), "split": (65, 72, 576), "gated": (65, 80, 576)},
    (80, 96, False): {"whole": (2289, 176, 576), "split": (81, 72, 576), "gated": (81, 80, 576)},
    (80, 96, True): {"whole": (65, 16424, 576), "split": (65, 4136, 1088), "gated": (66, 16464, 576)},
    (80, 112, False): {"whole": (81, 12344, 576), "split": (82, 3128, 1024), "gated": (81, 12464, 576)},
    (80, 112, True): {"whole": (66, 24648, 576), "split": (65, 6240, 1600), "gated": (65, 24880, 576)},
    (80, 128, False): {"whole": (81, 14480, 576), "split": (81, 3728, 1024), "gated": (81, 14496, 576)},
    (80, 128, True): {"whole": (65, 28832, 576), "split": (67, 4496, 3136), "gated": (68, 28752, 576)},
    (96, 112, False): {"whole": (244, 7200, 576), "split": (1442, 120, 2112), "gated": (163, 9616, 576)},
    (96, 112, True): {"whole": (82, 16392, 576), "split": (85, 2152, 2368), "gated": (82, 16432, 576)},
    (96, 128, False): {"whole": (482, 4720, 576), "split": (2785, 120, 3392), "gated": (485, 4752, 576)},
    (96, 128, True): {"whole": (81, 28920, 576), "split": (84, 7352, 1472), "gated": (81, 29264, 576)},
    (128, 64, False): {"split": (3076, 64, 3968)},
    (128, 64, True): {"whole": (97, 16360, 2112), "gated": (88, 15968, 5504)},
    (128, 96, False): {"whole": (195, 10936, 576), "split": (1563, 136, 4416), "gated": (195, 10992, 576)},
    (128, 96, True): {"whole": (97, 16440, 576), "split": (98, 2064, 4096), "gated": (97, 16400, 576)},
    (128, 128, False): {"whole": (291, 8232, 576), "split": (3077, 120, 4096), "gated": (290, 8224, 576)},
    (128, 128, True): {"whole": (98, 24600, 576), "split": (102, 4168, 2688), "gated": (97, 25328, 576)},
    (128, 256, False): {"whole": (260, 16488, 576), "split": (294, 4128, 9856), "gated": (257, 16688, 576)},
    (128, 256, True): {"whole": (97, 33048, 576), "split": (97, 12904, 12480), "gated": (65, 33184, 576)},
    (144, 112, False): {"whole": (257, 10888, 576), "split": (2081, 144, 13248), "gated": (264, 10960, 576)},
    (144, 112, True): {"whole": (129, 16464, 576), "split": (142, 2064, 10752), "gated": (129, 16528, 576)},
    (144, 128, False): {"whole": (772, 4760, 576), "split": (835, 568, 7104), "gated": (772, 4784, 576)},
    (144, 128, True): {"whole": (130, 28720, 576), "split": (131, 3728, 6144), "gated": (129, 28896, 576)},
    (160, 128, False): {"whole": (726, 5416, 576), "split": (3207, 352, 6080), "gated": (728, 5456, 576)},
    (160, 256, False): {"whole": (289, 21840, 576), "split": (2312, 392, 13120), "gated": (295, 21776, 576)},
    (160, 256, True): {"whole": (129, 32944, 576), "split": (151, 4312, 13760), "gated": (129, 32864, 576)},
    (192, 128, False): {"whole": (289, 10960, 576), "split": (2654, 136, 9536), "gated": (291, 11088, 576)},
    (192, 128, True): {"whole": (147, 16400, 576), "split": (161, 3632, 6976), "gated": (149, 16400, 576)},
    (192, 256, False): {"whole": (323, 21792, 576), "gated": (321, 21984, 576)},
    (192, 256, True): {"whole": (161, 33048, 576), "gated": (166, 32848, 576)},
    (224, 128, False): {"whole": (193, 16432, 576), "split": (3196, 136, 11776), "gated": (193, 16848, 576)},
    (224, 256, False): {"whole": (1160, 9808, 576), "split": (3108, 400, 13632), "gated": (1172, 9808, 576)},
    (256, 128, False): {"whole": (227, 16568, 576), "split": (2758, 552, 7680), "gated": (226, 16656, 576)},
    (256, 256, False): {"whole": (579, 16424, 576), "split": (581, 4376, 8192), "gated": (386, 24624, 576)},
    (288, 128, False): {"whole": (257, 21856, 576), "split": (4403, 136, 11648), "gated": (257, 22640, 576)},
    (288, 192, False): {"whole": (193, 32920, 576), "split": (4118, 272, 11776), "gated": (193, 33648, 576)},
}
SHAPES = [(*tile, form, *shape) for tile, forms in TILE_SHAPES.items() for form, shape in forms.items()]
# weight rows, k and gate of the projections of the 8B decoders: q/k/v, q/k/v apart, o, gate/up, down
DECODERS = [(6144, 4096, 0), (4096, 4096, 0), (1024, 4096, 0), (28672, 4096, 1), (4096, 14336, 0), (24576, 4096, 1),
            (4096, 12288, 0)]


def choice(m, rows, k, gated):
    from kv_cache_repair_amd import _native

    out = (ctypes.c_int32 * 4)()
    assert _native.lib().kvr_internal_tiled_choice(m, rows, k, gated, out) == 0
    return out[0], out[1], bool(out[2]), "gated" if gated else "split" if out[3] > 1 else "whole"


def test_the_shapes_reach_their_kernels():
    for bm, bn, streamed, form, m, rows, k in SHAPES:
        assert choice(m, rows, k, form == "gated") == (bm, bn, streamed, form)
        assert m % 16 or rows % 64


@pytest.mark.parametrize("rows,k,gated", DECODERS)
def test_the_shapes_cover_what_the_decoders_reach(rows, k, gated):
    covered = {shape[:4] for shape in SHAPES}
    for m in (*range(65, 1600), *range(1600, 16500, 41)):
        assert choice(m, rows, k, gated) in covered, m


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "-".join(map(str, s)))
def test_every_tile_gives_the_product(gpu_device, shape, dtype):
    _, _, _, form, m, rows, k = shape
    gen = torch.Generator(device=gpu_device).manual_seed(m + rows + k)
    x = torch.randn(m, k, device=gpu_device, generator=gen).to(dtype)
    if form == "gated":
        gate, up = ((torch.randn(rows // 2, k, device=gpu_device, generator=gen) * 0.04).to(dtype) for _ in range(2))
        y = tiled(x, [gate, up], SILU_GATE)
        assert_gate_close(y, x, gate, up)
        eager = torch.nn.functional.silu(exact_linear(x, gate)) * exact_linear(x, up)
        assert (ulp_distance(y, eager) <= 2).float().mean().item() >= 0.99
        return
    cut = rows // 3 // 8 * 8
    w = (torch.randn(rows, k, device=gpu_device, generator=gen) * 0.03).to(dtype)
    y = tiled(x, [w[:cut], w[cut:2 * cut], w[2 * cut:]], CONCAT)
    assert_linear_close(y, x, w)
    residual = torch.randn(m, rows, device=gpu_device, generator=gen).to(dtype)
    assert torch.equal(tiled(x, [w], RESIDUAL, residual), y + residual)
