"""Performance cases of the BERT encoder forward: what a serving program has this package run, through the
package's public entry points.

A pass is one complete forward of a stack of encoder layers over one batch of variable-length sequences, in the
five ways a program can ask for it:

  op       torch.ops.ByteTransformer.BertTransformer, one call per layer (the measurement of bert_bench.py)
  class    torch.classes.ByteTransformer.BertTransformer objects, one per layer
  layer    BertEncoderLayer objects through encoder_forward
  encoder  BertEncoder: every layer in one call, weights packed once when it is made
  graph    GraphedBertEncoder: a captured BertEncoder forward, called with new inputs

Keys of a case: api; batch, seq_len, heads, head_size, layers; dtype (fp16, fp32); lens ("uniform": integer-uniform
on [0.2 S, S], 0.6 S on average, as the package's workloads draw them; "full": every sequence S long); packed
(is_remove_padding); mask ("prefix": the first len_b keys; "blocks": several texts share one row, each token
attends to its own text, which only the padded rows support); bias (an additive [heads, S, S] attention bias).
"""
import math

import torch

import bytetransformer_amd as bt

DTYPES = {"fp16": torch.float16, "fp32": torch.float32}
LAYER_TENSORS = 12


def _case(name, api, batch, seq_len, heads=12, head_size=64, layers=12, dtype="fp16", lens="uniform", packed=True,
          mask="prefix", bias=False):
    case = dict(api=api, batch=batch, seq_len=seq_len, heads=heads, head_size=head_size, layers=layers, dtype=dtype,
                lens=lens, packed=packed, mask=mask, bias=bias)
    return dict(case, name=name) if name else case


def listed():
    return [
        # a single short query, answered at once: nothing but launches and the weights
        _case("op_1x32", "op", 1, 32),
        # a single paragraph
        _case("op_1x256", "op", 1, 256),
        # a small online batch behind a captured graph, ragged
        _case("graph_4x96", "graph", 4, 96),
        # an ordinary online batch of odd sizes, bound layer objects
        _case("class_7x217", "class", 7, 217),
        # the headline batch
        _case("op_16x512", "op", 16, 512),
        # long documents
        _case("op_16x1024", "op", 16, 1024),
        # many short texts in one batch (offline scoring)
        _case("encoder_100x120", "encoder", 100, 120),
        # the large encoder at its usual fine-tuning length: the largest case
        _case("encoder_large_32x384", "encoder", 32, 384, heads=16, layers=24),
        # several texts packed into one row, told apart by the mask: padded rows, the mask applied
        _case("op_blocks_6x250", "op", 6, 250, lens="full", packed=False, mask="blocks"),
        # a relative-position bias in every layer
        _case("encoder_bias_12x380", "encoder", 12, 380, bias=True),
        # full precision
        _case("op_fp32_16x256", "op", 16, 256, dtype="fp32"),
        # wide heads
        _case("layer_d128_8x300", "layer", 8, 300, heads=6, head_size=128),
    ]


def draw(rng):
    """One more case: tokens spread over the logarithm of 32 .. 16384 and the length over that of 16 .. 1024."""
    kind = rng.choice(["base", "base", "base", "encoder", "graph", "large", "blocks", "padded", "bias", "fp32", "head"])
    most = {"base": 16384, "encoder": 16384, "graph": 4096, "large": 6144, "blocks": 6144, "padded": 8192, "bias": 8192,
            "fp32": 2560, "head": 3072}[kind]
    tokens = math.exp(rng.uniform(math.log(32), math.log(most)))
    seq_len = round(math.exp(rng.uniform(math.log(16), math.log(min(1024.0, tokens)))))
    batch = max(1, min(128, int(tokens / seq_len)))
    lens = rng.choice(["uniform", "uniform", "uniform", "full"])
    per_layer = rng.choice(["op", "op", "class", "layer"])
    if kind == "base":
        return _case(None, per_layer, batch, seq_len, lens=lens)
    if kind in ("encoder", "graph"):
        return _case(None, kind, batch, seq_len, lens=lens)
    if kind == "large":
        return _case(None, rng.choice(["encoder", "op"]), batch, seq_len, heads=16, layers=24, lens=lens)
    if kind == "blocks":
        return _case(None, rng.choice(["encoder", per_layer]), batch, seq_len, lens="full", packed=False, mask="blocks")
    if kind == "padded":
        return _case(None, per_layer, batch, seq_len, lens=lens, packed=False)
    if kind == "bias":
        return _case(None, "encoder", batch, seq_len, lens=lens, bias=True)
    if kind == "fp32":
        return _case(None, rng.choice(["encoder", per_layer]), batch, seq_len, dtype="fp32", lens=lens)
    head_size = rng.choice([32, 96, 128])
    return _case(None, rng.choice(["encoder", per_layer]), batch, seq_len, heads=768 // head_size, head_size=head_size,
                 lens=lens)


def _layer_shapes(hidden, ffn):
    return [(hidden, 3 * hidden), (3 * hidden,), (hidden, hidden), (hidden,), (hidden,), (hidden,),
            (hidden, ffn), (ffn,), (ffn, hidden), (hidden,), (hidden,), (hidden,)]


def _lengths(case, gen):
    batch, seq_len = case["batch"], case["seq_len"]
    if case["lens"] == "full":
        return torch.full((batch,), seq_len, device="cuda")
    return torch.randint(math.ceil(0.2 * seq_len), seq_len + 1, (batch,), generator=gen, device="cuda")


def _mask(case, lens, gen, dtype):
    batch, seq_len = case["batch"], case["seq_len"]
    at = torch.arange(seq_len, device="cuda")
    if case["mask"] == "blocks":
        # text boundaries at about one position in 64
        cuts = torch.rand(batch, seq_len, generator=gen, device="cuda") < 1.0 / 64
        text = cuts.cumsum(1)
        return (text[:, :, None] == text[:, None, :]).to(dtype)
    return (at[None, None, :] < lens[:, None, None]).to(dtype).expand(batch, seq_len, seq_len).contiguous()


def prepare(case, seed):
    """Input, mask and the bound layers, as a program that serves one model holds them."""
    dtype = DTYPES[case["dtype"]]
    heads, head_size = case["heads"], case["head_size"]
    hidden = heads * head_size
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)

    def normal(shape, std, mean=0.0):
        t = torch.empty(shape, dtype=dtype, device="cuda")
        return t.normal_(mean, std, generator=gen)

    layers = []
    for _ in range(case["layers"]):
        w = [normal(s, 0.02) for s in _layer_shapes(hidden, 4 * hidden)]
        for i in (4, 10):      # LayerNorm gamma
            w[i] = normal(w[i].shape, 0.05, 1.0)
        layers.append(w)
    x = normal((case["batch"], case["seq_len"], hidden), 1.0)
    mask = _mask(case, _lengths(case, gen), gen, dtype)
    bias = normal((heads, case["seq_len"], case["seq_len"]), 0.5) if case["bias"] else None
    api = case["api"]
    if api in ("op", "class"):
        bt.load_th_op()
    if api == "class":
        model = [torch.classes.ByteTransformer.BertTransformer(heads, head_size, *w) for w in layers]
    elif api == "layer":
        model = [bt.BertEncoderLayer(heads, head_size, w, is_remove_padding=case["packed"]) for w in layers]
    elif api in ("encoder", "graph"):
        model = bt.BertEncoder(heads, head_size, layers, is_remove_padding=case["packed"])
        model.prepack()
        if api == "graph":
            model = model.graph(case["batch"], case["seq_len"])
    else:
        model = layers
    return dict(api=api, heads=heads, head_size=head_size, packed=case["packed"], model=model, x=x, mask=mask, bias=bias)


def run(state):
    api, model, mask = state["api"], state["model"], state["mask"]
    h = state["x"]
    if api == "op":
        layer = torch.ops.ByteTransformer.BertTransformer
        heads, head_size, packed = state["heads"], state["head_size"], state["packed"]
        for w in model:
            h = layer(heads, head_size, *w, h, mask, packed, True)
        return h
    if api == "class":
        for layer in model:
            h = layer.forwardv2(h, mask, state["packed"], True)
        return h
    if api == "layer":
        return bt.encoder_forward(model, h, mask)
    if api == "graph":
        return model(h, mask)
    return model(h, mask, attention_bias=state["bias"])


def work(case):
    """Weights, input, output and the mask entries that matter (row 0 of a prefix mask, every entry of another) once;
    four products on the valid rows and attention over the valid keys. Uniform lengths by their expected values."""
    size = 2 if case["dtype"] == "fp16" else 4
    batch, seq_len = case["batch"], case["seq_len"]
    hidden = case["heads"] * case["head_size"]
    weights = sum(math.prod(s) for s in _layer_shapes(hidden, 4 * hidden)) * case["layers"]
    mask = batch * seq_len * (seq_len if case["mask"] == "blocks" else 1)
    bias = case["heads"] * seq_len * seq_len if case["bias"] else 0
    full = case["lens"] == "full" or not case["packed"]
    rows = batch * seq_len * (1.0 if full else 0.6)
    pairs = batch * seq_len * seq_len * (1.0 if full else 0.36 + 0.64 / 12)
    return {"bytes": size * (weights + 2 * batch * seq_len * hidden + mask + bias),
            "flops": case["layers"] * (24.0 * rows * hidden * hidden + 4.0 * pairs * hidden)}


def tolerance(case):
    """fp16 keeps 11 bits of every tensor between two launches, over up to 24 layers; float sums run in any order."""
    return {"rel": 1e-5} if case["dtype"] == "fp32" else {"rel": 5e-3}
