"""Workloads of the MoE feed-forward path, for timing and for comparing results.

Shapes are the decoder's: hidden 1280, 64 routed experts of width 896 of which a
token takes 6, two shared experts (one of width 1792), vocabulary 129280. A case
is one of

* "experts": the expert layer of `layers` decoder layers, one call per layer, each
  on its own input (attention stands between them in a decoder);
* "block": the same with the residual and the RMSNorm (the post-attention half of
  a layer), one call per layer;
* "stack": the post-attention halves of `layers` layers in one call, layer after
  layer;
* "lm_head": the vocabulary projection of the last row.

`weights` is "bf16", "int8" (block-32 overlay, FP32 activations) or "w8a8" (the
overlay with dynamic activations). `mode` is the precision the caller asks for:
"fp32", "bf16" (bf16 activations) or "int8" (every group W8A8). Routing is
"even" (Gaussian router), "zipf" (capped Zipf popularity) or "hot" (80% of the
assignments on 8 experts).
"""
import functools
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "unlimited-ocr-kernel_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
import uocr_moe as um  # noqa: E402
from uocr_moe import synthetic as syn  # noqa: E402

H, I, E, SHARED, K, V = 1280, 896, 64, 2, 6, 129280
S = I * SHARED
MAX_TOKENS, MAX_LAYERS = 4096, 12
EPS = 1e-6
STD = 0.02
# Least distance of a token's last chosen logit from the first one not chosen.
# Logits are sums of 1280 FP32 products: an implementation that sums them in
# another order may choose differently where two of them are closer than their
# rounding (about 1e-6), and the row's result is then another one. Rows that
# close are drawn again, so that results can be compared.
LEAST_GAP = 1e-4

MATRICES = ("gate", "up", "down", "shared_gate", "shared_up", "shared_down")


def _case(name, op, weights, mode, tokens, layers=1, routing="even", normalize=True):
    return {"name": name, "op": op, "weights": weights, "mode": mode, "tokens": tokens,
            "layers": layers, "routing": routing, "normalize": normalize}


def listed():
    return [
        # One generated token: the expert layers of a decode step. Four layers,
        # so that the weights come from memory and not from a cache, as in a
        # decoder that passes through all of its layers for each token.
        _case("decode_bf16", "experts", "bf16", "fp32", 1, layers=4),
        _case("decode_int8", "experts", "int8", "fp32", 1, layers=4),
        # A few sequences decoded together with dynamic activations: most groups
        # hold one row.
        _case("batch5_w8a8", "block", "w8a8", "fp32", 5, layers=2),
        # Sixteen sequences decoded together from the INT8 overlay.
        _case("batch16_int8", "experts", "int8", "fp32", 16),
        # A larger decode batch, or a short prompt: few rows for each expert.
        _case("batch61_bf16", "block", "bf16", "fp32", 61),
        # The image tokens of one page in the W8A8 overlay.
        _case("prefill273_w8a8", "experts", "w8a8", "fp32", 273, normalize=False),
        # A prompt of 512 tokens from the INT8 overlay, and with every group W8A8.
        _case("prefill512_int8", "experts", "int8", "fp32", 512),
        _case("prefill512_int8_activations", "experts", "w8a8", "int8", 512),
        # A prompt of 1024 tokens with uneven expert popularity.
        _case("prefill1024_zipf", "experts", "bf16", "fp32", 1024, routing="zipf"),
        # A longer prompt of odd length where the caller allows bf16 activations.
        _case("prefill1531_bf16_activations", "block", "bf16", "bf16", 1531),
        # A long prompt through all layers, most of it on a few experts.
        _case("stack4096_hot", "stack", "bf16", "fp32", 4096, layers=12, routing="hot"),
        # The vocabulary projection that ends each decode step.
        _case("lm_head_bf16", "lm_head", "bf16", "fp32", 1),
    ]


def draw(rng):
    # One in ten is a vocabulary projection; the others spread the token count
    # over its logarithm.
    if rng.random() < 0.1:
        tokens = rng.randint(1, 64)  # rows in hand; the last one is projected
        return _unnamed("lm_head", rng.choice(["bf16", "int8", "w8a8"]), "fp32", tokens, 1, "even",
                        True)
    tokens = min(MAX_TOKENS, max(1, int(round(math.exp(rng.uniform(0, math.log(MAX_TOKENS)))))))
    weights = rng.choice(["bf16", "int8", "w8a8"])
    mode = "fp32"
    if weights == "w8a8":
        mode = rng.choice(["fp32", "int8"])
    elif tokens > 1:
        mode = rng.choice(["fp32", "fp32", "bf16"])
    op = rng.choice(["experts", "block"])
    layers = 4 if tokens <= 2 else rng.randint(1, 2)
    routing = rng.choice(["even", "zipf", "hot"])
    return _unnamed(op, weights, mode, tokens, layers, routing, rng.random() < 0.5)


def _unnamed(*a):
    c = _case("", *a)
    del c["name"]
    return c


# ------------------------------------------------------------------- inputs

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _bf16(t):
    return t.to(torch.bfloat16)


def _quantize(w):
    """Round-to-nearest int8 blocks of 32 with an f32 scale each."""
    blocks = w.float().reshape(*w.shape[:-1], w.shape[-1] // 32, 32)
    s = blocks.abs().amax(-1) / 127.0
    q = torch.round(blocks / s.unsqueeze(-1).clamp_min(1e-30)).clamp(-127, 127)
    return q.to(torch.int8).reshape(w.shape), s.contiguous()


@functools.lru_cache(maxsize=None)
def _zipf_rows():
    """Row norms of a router whose experts are chosen with Zipf shares."""
    return torch.as_tensor(syn.route_profile(syn.zipf_share(E, K), K, samples=4096),
                           dtype=torch.float32)


HOT, HOT_MEAN, HOT_TILT, GROWTH = 8, 4.0, 20.4, 0.0655


def _direction():
    d = torch.randn(H, generator=torch.Generator().manual_seed(4242))
    return (d / d.norm()).cuda()


def _router(case, layer, g):
    r = torch.randn((E, H), generator=g, device="cuda")
    if case["routing"] == "zipf":
        r *= _zipf_rows().cuda()[:, None]
    elif case["routing"] == "hot":
        # The first experts lean towards a direction that every input carries;
        # deeper layers of a stack carry less of it after their norm.
        tilt = HOT_TILT * (math.sqrt(1 + layer * GROWTH) if case["op"] == "stack" else 1.0)
        r[:HOT] += tilt * _direction()
    return _bf16(r * STD)


def _layer_weights(case, seed, layer):
    g = _generator(seed * 64 + layer)

    def normal(*shape):
        return _bf16(torch.randn(shape, generator=g, device="cuda") * STD)

    return {"router": _router(case, layer, g),
            "norm_weight": _bf16(1 + 0.1 * torch.randn(H, generator=g, device="cuda")),
            "gate": normal(E, I, H), "up": normal(E, I, H), "down": normal(E, H, I),
            "shared_gate": normal(S, H), "shared_up": normal(S, H), "shared_down": normal(H, S)}


def _rows(case, n, g):
    x = torch.randn((n, H), generator=g, device="cuda")
    return x + HOT_MEAN * _direction() if case["routing"] == "hot" else x


def _norm(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _least_gap(x64, router):
    top = (x64 @ router.double().T).topk(K + 1, dim=-1).values if K < E else None
    return top[:, K - 1] - top[:, K]


def _inputs(case, weights, seed):
    """The input rows: [layers] tensors, or one for a stack."""
    g = _generator(seed * 64 + 63)
    T, stack = case["tokens"], case["op"] == "stack"

    def gaps(x, layers):
        x, least = x.double(), None
        for w in layers:
            z = x if case["op"] == "experts" else _norm(x, w["norm_weight"].double())
            gap = _least_gap(z, w["router"])
            least = gap if least is None else torch.minimum(least, gap)
            if w is not layers[-1]:
                x = x + _experts64(z, w, case)
        return least

    got = []
    for layers in ([weights] if stack else [[w] for w in weights]):
        x = _rows(case, T, g)
        for _ in range(20):
            close = (gaps(x, layers) < LEAST_GAP).nonzero().flatten()
            if close.numel() == 0:
                break
            x[close] = _rows(case, close.numel(), g)
        got.append(x)
    return got


def _config(case):
    return um.config(H, I, E, SHARED, K, normalize=case["normalize"], eps=EPS)


@functools.lru_cache(maxsize=None)
def _context():
    """A program's one context: device, stream and scratch for its longest prompt."""
    return um.Context(0, um.scratch_bytes(um.config(H, I, E, SHARED, K), MAX_TOKENS) + (64 << 20))


def _head_inputs(case, seed):
    g = _generator(seed)
    w = _bf16(torch.randn((V, H), generator=g, device="cuda") * STD)
    norm = _bf16(1 + 0.1 * torch.randn(H, generator=g, device="cuda")).float()
    hidden = torch.randn((case["tokens"], H), generator=g, device="cuda")
    return w, norm, hidden


FLAGS = {"fp32": um.FLAG_FP32_CLASS, "bf16": um.FLAG_BF16_ACTIVATIONS, "int8": um.FLAG_INT8_MFMA}
MODES = {"int8": um.QUANT_WEIGHTS_ONLY, "w8a8": um.QUANT_DYNAMIC}


def prepare(case, seed):
    ctx = _context()
    if case["op"] == "lm_head":
        w, norm, hidden = _head_inputs(case, seed)
        if case["weights"] == "bf16":
            more = {"weight": w.view(torch.int16)}
        else:
            q, s = _quantize(w)
            more = {"q": q, "scales": s, "mode": MODES[case["weights"]]}
        torch.cuda.synchronize()  # the library copies on its own stream
        head = um.LmHead(ctx, norm, EPS, where=um.MEMORY_DEVICE, **more)
        return {"case": case, "ctx": ctx, "head": head, "hidden": hidden,
                "out": torch.empty(V, device="cuda")}
    cfg, layers, kept = _config(case), [], []
    for l in range(case["layers"]):
        w = _layer_weights(case, seed, l)
        torch.cuda.synchronize()
        layer = um.MoeLayer(ctx, cfg, {n: t.view(torch.int16) for n, t in w.items()},
                            um.MEMORY_DEVICE)
        if case["weights"] != "bf16":
            q = {n: _quantize(w[n]) for n in MATRICES}
            torch.cuda.synchronize()
            layer.attach_int8(ctx, q, um.MEMORY_DEVICE, MODES[case["weights"]])
        layers.append(layer)
        # The inputs of a stack depend on all of its layers' weights.
        kept.append(w if case["op"] == "stack" else
                    {n: w[n] for n in ("router", "norm_weight")})
        del w
    xs = _inputs(case, kept, seed)
    return {"case": case, "ctx": ctx, "layers": layers, "x": xs,
            "y": [torch.empty_like(x) for x in xs], "flags": FLAGS[case["mode"]]}


def run(state):
    op, ctx = state["case"]["op"], state["ctx"]
    if op == "lm_head":
        state["head"].logits(ctx, state["hidden"], state["out"], sync=False)
        return state["out"]
    if op == "stack":
        um.block_forward(ctx, state["layers"], state["x"][0], state["y"][0], state["flags"],
                         sync=False)
    else:
        for layer, x, y in zip(state["layers"], state["x"], state["y"]):
            if op == "experts":
                um.forward(ctx, layer, x, y, state["flags"], sync=False)
            else:
                um.block_forward(ctx, [layer], x, y, state["flags"], sync=False)
    return state["y"]


# ----------------------------------------------------------- work, tolerance

def _shares(routing):
    if routing == "zipf":
        return [float(q) for q in syn.zipf_share(E, K)]
    if routing == "hot":
        return [0.8 * K / HOT] * HOT + [0.2 * K / (E - HOT)] * (E - HOT)
    return [K / E] * E


def work(case):
    T = case["tokens"]
    per_weight = 2.0 if case["weights"] == "bf16" else 1.0 + 4.0 / 32
    if case["op"] == "lm_head":
        return {"bytes": V * H * per_weight + H * 8 + V * 4, "flops": 2.0 * V * H}
    unique = sum(1 - (1 - q) ** T for q in _shares(case["routing"])) if T > 1 else K
    layer = (unique * I + S) * 3 * H * per_weight + E * H * 2
    rows = case["layers"] if case["op"] != "stack" else 1
    return {"bytes": case["layers"] * layer + rows * 2.0 * T * H * 4,
            "flops": case["layers"] * 2.0 * T * ((K * I + S) * 3 * H + E * H)}


def tolerance(case):
    """About four times the distance from exact() that was measured."""
    if case["weights"] == "w8a8":
        # A value next to a rounding boundary of its int8 block lands on the
        # other side when a sum is taken in another order: one step of one
        # value is 1/127 of its block's largest, about 2e-4 of a single row's
        # result. Without such a step: 1e-6 (2.6e-5 over 512 rows).
        return {"rel": 5e-4}
    if case["mode"] == "bf16":
        return {"rel": 1.2e-2}  # measured 2.9e-3
    if case["tokens"] == 1 or case["op"] == "lm_head":
        return {"rel": 2e-6}  # FP32 products and sums: measured 3.2e-7
    return {"rel": 2e-5}  # activations as two bf16 terms: measured 4.4e-6


# -------------------------------------------------------------------- exact

def _dequantized(q, s):
    return (q.double().reshape(*s.shape, 32) * s.double().unsqueeze(-1)).reshape(q.shape)


def _matrix(w, case):
    return w.double() if case["weights"] == "bf16" else _dequantized(*_quantize(w))


def _project(x, w, case):
    """x [rows, k] . w^T; the rows as int8 blocks where the path quantises them."""
    if case["weights"] == "w8a8" and (case["mode"] == "int8" or x.shape[0] == 1):
        x = _dequantized(*_quantize(x))
    return x @ _matrix(w, case).T


def _feed_forward(x, gate, up, down, case):
    g = _project(x, gate, case)
    return _project(g * torch.sigmoid(g) * _project(x, up, case), down, case)


def _experts64(x, w, case):
    p = torch.softmax(x @ w["router"].double().T, dim=-1)
    top, ids = p.topk(K, dim=-1)
    if case["normalize"]:
        top = top / top.sum(-1, keepdim=True)
    y = _feed_forward(x, w["shared_gate"], w["shared_up"], w["shared_down"], case)
    for e in range(E):
        rows, slot = (ids == e).nonzero(as_tuple=True)
        if rows.numel():
            out = _feed_forward(x[rows], w["gate"][e], w["up"][e], w["down"][e], case)
            y[rows] += top[rows, slot].unsqueeze(-1) * out
    return y


def exact(case, seed):
    if case["op"] == "lm_head":
        w, norm, hidden = _head_inputs(case, seed)
        x = _norm(hidden[-1:].double(), norm.double())
        return _project(x, w, case).flatten()
    weights = [_layer_weights(case, seed, l) for l in range(case["layers"])]
    xs = _inputs(case, weights, seed)
    if case["op"] == "stack":
        x = xs[0].double()
        for w in weights:
            x = x + _experts64(_norm(x, w["norm_weight"].double()), w, case)
        return [x]
    if case["op"] == "block":
        return [x.double() + _experts64(_norm(x.double(), w["norm_weight"].double()), w, case)
                for x, w in zip(xs, weights)]
    return [_experts64(x.double(), w, case) for x, w in zip(xs, weights)]
