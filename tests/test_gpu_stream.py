"""The weight-streaming grouped GEMM at the edges of its tiles.

Two experts of which every token takes both, so every group (the shared
expert's too) has exactly T rows: one row tile of 32, the step to 64, a full
64, a second tile of one row and a third. The shapes leave column tiles that
are not full, one, three and five 64-deep chunks of K, and shared widths that
do (1, 3 x 128) and do not (192) split their reduction in two."""
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
