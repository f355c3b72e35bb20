"""Which grouped GEMM a BF16 batch takes: the weight-streaming kernel or the
256 x 256 tiles."""
import pytest

torch = pytest.importorskip("torch")

import uocr_moe as um  # noqa: E402
from test_gpu_parity import ctx  # noqa: E402,F401
from uocr_moe import synthetic as syn  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,larger,flags", [(832, 1024, 0),
                                            (608, 672, um.FLAG_BF16_ACTIVATIONS)],
                         ids=["fp32-class", "bf16-activations"])
def test_wide_layer_takes_the_tiles(ctx, T, larger, flags):  # noqa: F811
    """A wide layer (23 M multiply-adds a token; the streaming kernel was up to
    70% slower on such layers) runs on the 256 x 256 tiles at T tokens, as it
    does at `larger`, where every layer does: rows of the two batches have the
    same bits, since a tile sums a row's products in one order whatever the
    batch (and the router splits its sums alike at both sizes: 4 ways at 817 to
    1024 tokens, 6 at 577 to 672). The streaming kernel sums in another."""
    H, inter, E, K = 2048, 1408, 8, 6
    w = syn.moe_weights_device(H, inter, E, 2, seed=71)
    torch.cuda.synchronize()  # the library copies on its own stream
    layer = um.MoeLayer(ctx, um.config(H, inter, E, 2, K), w, um.MEMORY_DEVICE)
    g = torch.Generator(device="cuda").manual_seed(72)
    x = torch.randn((larger, H), generator=g, device="cuda")
    y, part = torch.empty_like(x), torch.empty((T, H), device="cuda")
    torch.cuda.synchronize()
    print(f"wide layer T={T} against {larger} flags={flags}", flush=True)
    um.forward(ctx, layer, x, y, flags)
    um.forward(ctx, layer, x[:T].contiguous(), part, flags)
    layer.close()
    assert torch.isfinite(y).all()
    assert torch.equal(part, y[:T])
