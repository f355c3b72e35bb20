"""The 256 x 256 grouped GEMM at the edges of its tiles, and which BF16 batches
take it: those above 896 tokens (640 with BF16 activations), and above a number
of operations in wide layers; the rest take the weight-streaming kernel."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import uocr_moe as um  # noqa: E402
from test_gpu_parity import Case, check_layer, ctx  # noqa: E402,F401
from test_gpu_stream import BF16_CLASS, FP32_CLASS  # noqa: E402
from uocr_moe import synthetic as syn  # noqa: E402

pytestmark = pytest.mark.gpu

BF16 = um.FLAG_BF16_ACTIVATIONS
# Two experts that every token takes (each group has T rows), and eight of which
# it takes two (uneven groups). Column tiles of 256 and 512 that are not full, 2,
# 6 and 10 stages of K.
SHAPES = [dict(hidden=64, inter=64, experts=2, shared=2),
          dict(hidden=320, inter=192, experts=8, shared=1)]


@pytest.mark.parametrize("T,flags", [(897, 0), (1025, 0), (1531, 0), (641, BF16), (1025, BF16),
                                     (1531, BF16), (2305, BF16)])
@pytest.mark.parametrize("shape", range(len(SHAPES)))
def test_tile_edges(ctx, shape, T, flags):  # noqa: F811
    """Last row tiles of 1, 129 and 251 rows (each form has its own items for
    128 or fewer), up to 2048 tokens with the shared expert on a second stream;
    BF16 activations have square items only beyond that."""
    case = Case(ctx, SHAPES[shape], 2, seed=950 + shape)
    x = syn.activations(T, SHAPES[shape]["hidden"], seed=960 + T)
    print(f"tiles shape={shape} T={T} flags={flags}", flush=True)
    y = check_layer(case, ctx, x, tol=BF16_CLASS if flags else FP32_CLASS, flags=flags)
    # A row does not depend on its place or on the other rows of its tile.
    back, _ = case.run(ctx, np.ascontiguousarray(x[::-1]), flags)
    assert np.array_equal(back[::-1], y)


@pytest.mark.parametrize("T,flags", [(896, 0), (897, 0), (640, BF16), (641, BF16)])
def test_last_streaming_and_first_tiled_batch(ctx, T, flags):  # noqa: F811
    """Row tiles, work lists and streams change from one size to the next."""
    shape = dict(hidden=192, inter=128, experts=16, shared=3)
    case = Case(ctx, shape, 4, seed=970)
    print(f"engine boundary T={T} flags={flags}", flush=True)
    check_layer(case, ctx, syn.activations(T, 192, seed=971),
                tol=BF16_CLASS if flags else FP32_CLASS, flags=flags)


@pytest.mark.parametrize("H,T,larger,flags", [(2048, 832, 1024, 0), (2048, 608, 672, BF16),
                                              (4096, 190, 1024, 0), (4096, 190, 1024, BF16)],
                         ids=["fp32-class", "bf16-activations", "wider", "wider-bf16-activations"])
def test_wide_layer_takes_the_tiles(ctx, H, T, larger, flags):  # noqa: F811
    """A wide layer (23 or 46 M multiply-adds a token; the streaming kernel was up
    to 70% slower on such layers) runs on the 256 x 256 tiles at T tokens, as it
    does at `larger`, where every layer does: rows of the two batches have the
    same bits, since a tile sums a row's products in one order whatever the
    batch. So does the router: up to hidden 2048 it splits its sums alike at both
    sizes (4 ways at 817 to 1024 tokens, 6 at 577 to 672), beyond not at all. The
    streaming kernel sums in another order."""
    inter, E, K = 1408, 8, 6
    w = syn.moe_weights_device(H, inter, E, 2, seed=71)
    torch.cuda.synchronize()  # the library copies on its own stream
    layer = um.MoeLayer(ctx, um.config(H, inter, E, 2, K), w, um.MEMORY_DEVICE)
    g = torch.Generator(device="cuda").manual_seed(72)
    x = torch.randn((larger, H), generator=g, device="cuda")
    y, part = torch.empty_like(x), torch.empty((T, H), device="cuda")
    torch.cuda.synchronize()
    print(f"wide layer H={H} T={T} against {larger} flags={flags}", flush=True)
    um.forward(ctx, layer, x, y, flags)
    um.forward(ctx, layer, x[:T].contiguous(), part, flags)
    layer.close()
    assert torch.isfinite(y).all()
    assert torch.equal(part, y[:T])
