"""The weight-streaming grouped GEMM at the edges of its tiles.

Work items are up to 64 rows in row tiles of 16. test_stream_tile_edges has two
experts of which every token takes both, so every group (the shared expert's
too) has exactly T rows: two row tiles of which the second holds one row, two,
three and four full ones, a second item of one row, and a third item. The shapes
leave column tiles that are not full, one, three and five 64-deep chunks of K,
and shared widths that do (128, 384) and do not (192) split their reduction in
two. test_stream_uneven_groups has groups of no row, of one (under
DynamicActivations the W8A8 units inside the same launches) and of many."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle as orc  # noqa: E402
import uocr_moe as um  # noqa: E402
from test_gpu_parity import Case, check_layer, ctx  # noqa: E402,F401
from uocr_moe import synthetic as syn  # noqa: E402

pytestmark = pytest.mark.gpu

# An activation enters as hi + lo bf16 terms with a residual of at most
# 2^-18 of it. A projection's error is then at most 2^-18 sum|x w|, and
# sum|x w| is about 0.64 sqrt(K) <= 13 times the norm of a sum of K <= 384
# Gaussian products; gate, up and down: 3 x 13 x 2^-18.
FP32_CLASS = 1.5e-4
# One bf16 term: 2^-9 in place of 2^-18, and random signs (a sum of K
# rounding errors grows with sqrt(K), not K): 3 x 3 x 2^-9.
BF16_CLASS = 2e-2

# Under DynamicActivations a hidden value of a single-row group that is one ulp
# away from the oracle's can land on the next int8 step, 1/127 of its block's
# largest value (up to some 5 times their rms). Times a weight of at most 1.7
# times the weights' rms (uniform int8), against the largest of the outputs,
# some 3 sqrt(K) rms products with K >= 128: 5/127 x 1.7 / (3 sqrt(128)) = 2e-3.
W8A8_CLASS = 3e-3

SHAPES = [dict(hidden=64, inter=64, experts=2, shared=2),
          dict(hidden=320, inter=192, experts=2, shared=1),
          dict(hidden=192, inter=128, experts=2, shared=3)]


@pytest.mark.parametrize("quant", [orc.QUANT_NONE, orc.QUANT_WEIGHTS_ONLY, orc.QUANT_DYNAMIC])
@pytest.mark.parametrize("shape", range(len(SHAPES)))
def test_stream_tile_edges(ctx, shape, quant):  # noqa: F811
    case = Case(ctx, SHAPES[shape], 2, seed=900 + shape, quant=quant)
    for T in (17, 32, 33, 48, 49, 64, 65, 129, 257):
        x = syn.activations(T, SHAPES[shape]["hidden"], seed=910 + T)
        print(f"stream shape={shape} quant={quant} T={T}", flush=True)
        y = check_layer(case, ctx, x, tol=FP32_CLASS)
        check_layer(case, ctx, x, tol=BF16_CLASS, flags=um.FLAG_BF16_ACTIVATIONS)
        # A row does not depend on its place or on the other rows of its tile
        # (of batches of one size: the split of K goes by the token count).
        y1, _ = case.run(ctx, np.ascontiguousarray(x[::-1]))
        assert np.array_equal(y1[::-1], y)


UNEVEN = [dict(hidden=320, inter=192, experts=24, shared=1),
          dict(hidden=192, inter=128, experts=24, shared=3)]


@pytest.mark.parametrize("quant", [orc.QUANT_NONE, orc.QUANT_WEIGHTS_ONLY, orc.QUANT_DYNAMIC])
@pytest.mark.parametrize("shape", range(len(UNEVEN)))
def test_stream_uneven_groups(ctx, shape, quant):  # noqa: F811
    scale = syn.route_profile(syn.zipf_share(24, 2), 2, samples=4096)
    case = Case(ctx, UNEVEN[shape], 2, seed=931, quant=quant, router_scale=scale)
    tol = W8A8_CLASS if quant == orc.QUANT_DYNAMIC else FP32_CLASS
    for T in (17, 40, 300):
        x = syn.activations(T, UNEVEN[shape]["hidden"], seed=940 + T)
        print(f"uneven groups shape={shape} quant={quant} T={T}", flush=True)
        check_layer(case, ctx, x, tol=tol)
        check_layer(case, ctx, x, tol=BF16_CLASS, flags=um.FLAG_BF16_ACTIVATIONS)
        if T == 40:
            rows = np.diff(case.run(ctx, x)[1]["expert_offsets"])
            assert (rows == 0).any() and (rows == 1).any() and (rows >= 16).any()
