"""Performance cases of the library: what its users run, through the public handles.

Three chains of dependent kernels make up the library's work, and each has one handle in ``cusync_amd.api``:

* ``Mlp``: the MLP block of one GPU's shard, GPT-3 (hidden 12288, inner 6144, GeLU) or LLaMA (hidden 8192, inner 2752 or
  2816, SwiGLU), at any number of rows: a decode step has few, a prefill or a training batch up to 2048;
* ``AttnLayer``: projection to Q|K|V, causal attention over the cached and the new rows, output projection, for 12 heads of
  128 (GPT-3's shard): prefill has no cached rows, decode has many and few new ones;
* ``ConvChain``: dependent 3x3 convolutions of ResNet and VGG blocks.

A pass is one ``run`` of the handle on operands resident on the device, which returns when the outputs are there.
"""
import math

import torch

from cusync_amd import api

GPT3_HIDDEN, GPT3_INNER = 12288, 6144
LLAMA_HIDDEN, LLAMA_INNERS = 8192, (2752, 2816)
HEADS, HEAD_DIM = 12, 128
MOST_ROWS = 2048
MOST_CACHED = 8192
# image side and channels of a ResNet stage
CONV_STAGES = ((56, 64), (28, 128), (14, 256), (7, 512))


def _mlp(model, rows, sync, inner=0):
    return {"chain": "mlp", "model": model, "rows": rows, "sync": sync, "inner": inner or (GPT3_INNER if model == "gpt3" else LLAMA_INNERS[0])}


def _attention(rows, cached, sync):
    return {"chain": "attention", "rows": rows, "cached": cached, "sync": sync}


def _conv(images, side, channels, layers, sync):
    return {"chain": "conv", "images": images, "side": side, "channels": channels, "layers": layers, "sync": sync}


def listed():
    return [
        # one token of one sequence: what interactive decoding costs per layer
        dict(_mlp("gpt3", 1, "tile"), name="gpt3_mlp_1"),
        # decoding a batch of sequences in step
        dict(_mlp("gpt3", 64, "tile"), name="gpt3_mlp_64"),
        # a large decoding batch or a short prompt
        dict(_mlp("gpt3", 256, "row"), name="gpt3_mlp_256"),
        # a prompt of no particular length
        dict(_mlp("gpt3", 777, "row"), name="gpt3_mlp_777"),
        # a full context, or one step's rows of a training batch
        dict(_mlp("gpt3", 2048, "row"), name="gpt3_mlp_2048"),
        # decoding on the gated MLP, under the policy made for it
        dict(_mlp("llama", 16, "strided"), name="llama_mlp_16"),
        # prefill on the gated MLP
        dict(_mlp("llama", 1000, "row"), name="llama_mlp_1000"),
        # decoding: a few sequences' new rows behind a context
        dict(_attention(16, 2048, "row"), name="attention_16_behind_2048"),
        # prefill of a short and of a full context
        dict(_attention(500, 0, "strided"), name="attention_500"),
        dict(_attention(2048, 0, "row"), name="attention_2048"),
        # the pair of convolutions of a ResNet block, first and third stage, at the usual batch
        dict(_conv(32, 56, 64, 2, "row"), name="conv_56x56x64"),
        dict(_conv(32, 14, 256, 2, "tile"), name="conv_14x14x256"),
    ]


def _spread(rng, low, high):
    """A whole number between low and high, even over the logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(("gpt3", "gpt3", "gpt3", "llama", "llama", "prefill", "prefill", "decode", "conv", "conv"))
    if kind == "gpt3":
        return _mlp("gpt3", _spread(rng, 1, MOST_ROWS), rng.choice(("stream", "row", "tile")))
    if kind == "llama":
        return _mlp("llama", _spread(rng, 1, MOST_ROWS), rng.choice(("stream", "row", "tile", "strided")), rng.choice(LLAMA_INNERS))
    if kind == "prefill":
        return _attention(_spread(rng, 64, MOST_ROWS), 0, rng.choice(("stream", "row", "tile", "strided")))
    if kind == "decode":
        return _attention(_spread(rng, 1, 64), _spread(rng, 64, MOST_CACHED), rng.choice(("stream", "row", "tile", "strided")))
    side, channels = rng.choice(CONV_STAGES)
    return _conv(_spread(rng, 1, 32), side + rng.choice((-1, 0, 0, 1)), channels, rng.choice((2, 2, 4)), rng.choice(("stream", "row", "tile")))


SYNC = {"stream": api.SYNC.STREAM, "row": api.SYNC.ROW, "tile": api.SYNC.TILE, "strided": api.SYNC.STRIDED}


class _State:
    """The handle, the operands it works on and the call that makes a pass; the handle is given back with the state."""

    def __init__(self, handle, call, outputs, keep):
        self.handle, self.call, self.outputs, self.keep = handle, call, outputs, keep

    def __del__(self):
        self.handle.destroy()


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def uniform(*shape):       # activations, U[-1, 1]
        return torch.empty(shape, device="cuda", dtype=torch.float16).uniform_(-1, 1, generator=gen)

    def normal(std, *shape):   # weights, cached projections
        return torch.empty(shape, device="cuda", dtype=torch.float16).normal_(0, std, generator=gen)

    def zeros(*shape):
        return torch.zeros(shape, device="cuda", dtype=torch.float16)

    sync = SYNC[case["sync"]]
    if case["chain"] == "mlp":
        llama = case["model"] == "llama"
        rows, inner, hidden = case["rows"], case["inner"], LLAMA_HIDDEN if llama else GPT3_HIDDEN
        x, w1, w2 = uniform(rows, hidden), normal(0.02, hidden, inner * (2 if llama else 1)), normal(0.02, inner, hidden)
        h, y = zeros(rows, inner), zeros(rows, hidden)
        torch.cuda.synchronize()      # the handle works on streams of its own
        mlp = api.Mlp(api.MODEL.LLAMA if llama else api.MODEL.GPT3, rows, hidden, inner, sync, w1.data_ptr(), w2.data_ptr())
        return _State(mlp, lambda: mlp.run(x.data_ptr(), h.data_ptr(), y.data_ptr()), {"h": h, "y": y}, (x, w1, w2))
    if case["chain"] == "attention":
        rows, cached, width = case["rows"], case["cached"], HEADS * HEAD_DIM
        x, wqkv, wo = uniform(rows, GPT3_HIDDEN), normal(0.02, GPT3_HIDDEN, 3 * width), normal(0.02, width, GPT3_HIDDEN)
        # cached rows as the projection leaves them: a sum of 12288 products of U[-1, 1] and N(0, 0.02)
        qkv = normal(0.02 * math.sqrt(GPT3_HIDDEN / 3), cached + rows, 3 * width)
        o, y = zeros(rows, width), zeros(rows, GPT3_HIDDEN)
        torch.cuda.synchronize()
        layer = api.AttnLayer(rows, GPT3_HIDDEN, HEADS, sync, wqkv.data_ptr(), wo.data_ptr(), cached_rows=cached)
        return _State(layer, lambda: layer.run(x.data_ptr(), qkv.data_ptr(), o.data_ptr(), y.data_ptr()),
                      {"qkv": qkv[cached:], "o": o, "y": y}, (x, wqkv, wo))
    images, side, channels, layers = case["images"], case["side"], case["channels"], case["layers"]
    x = uniform(images, side, side, channels)
    ws = [normal(math.sqrt(2.0 / (9 * channels)), channels, 3, 3, channels) for _ in range(layers)]
    ys = [zeros(images, side, side, channels) for _ in range(layers)]
    torch.cuda.synchronize()
    chain = api.ConvChain(images, side, side, channels, [w.data_ptr() for w in ws], sync)
    return _State(chain, lambda: chain.run(x.data_ptr(), [y.data_ptr() for y in ys]), {"y": ys}, (x, ws))


def run(state):
    state.call()
    return state.outputs


def work(case):
    """Operands and results once each, in halfs; a chain's intermediates are written once and read once."""
    if case["chain"] == "mlp":
        llama = case["model"] == "llama"
        rows, inner, hidden = case["rows"], case["inner"], LLAMA_HIDDEN if llama else GPT3_HIDDEN
        weights = hidden * inner * (3 if llama else 2)
        return {"bytes": 2.0 * (weights + 2 * rows * hidden + 2 * rows * inner), "flops": 2.0 * rows * weights}
    if case["chain"] == "attention":
        rows, cached, width = case["rows"], case["cached"], HEADS * HEAD_DIM
        weights = 4 * width * GPT3_HIDDEN
        pairs = rows * cached + rows * (rows + 1) / 2      # (query, key) under the causal mask
        return {"bytes": 2.0 * (weights + 2 * rows * GPT3_HIDDEN + 2 * rows * 3 * width + 2 * cached * width + 2 * rows * width),
                "flops": 2.0 * rows * weights + 4.0 * pairs * width}
    pixels, channels, layers = case["images"] * case["side"] ** 2, case["channels"], case["layers"]
    return {"bytes": 2.0 * layers * (2 * pixels * channels + 9 * channels * channels), "flops": 2.0 * layers * pixels * 9 * channels * channels}


def tolerance(case):
    """About four times the largest error of the outputs against the same chain in float64: rel 2.9e-4 and max 1.3e-3 for the
    MLPs and a pair of convolutions (4.2e-4 and 2.0e-3 for four), 5.6e-4 and 1.0e-2 for attention, whose probabilities are
    rounded to halfs as well."""
    if case["chain"] == "attention":
        return {"rel": 2.2e-3, "max": 0.04}
    return {"rel": 1.6e-3 if case["chain"] == "conv" else 1.2e-3, "max": 8e-3}
