"""The work that is timed when this package is tuned, as plain cases over its public entry points.

`listed()` names twelve cases, `draw(rng)` gives further ones of the same ranges; a case is prepared
once (`prepare`: weights from a seed, quantized and warmed as a serving program keeps them, and the
inputs of one call) and then run many times (`run`: one pass, no synchronisation of its own).

Kinds of case
  dense      a quantized `Dense` called eagerly: int8 (activations quantised per row on the fly) or
             int4 (grouped by 128 as `quantize("int4")` does by default, or per channel), float32
             (the default policy) or bfloat16 compute, one row (decode) to thousands (prefill)
  einsum     the attention projections `btd,dnh->btnh` / `btnh,nhd->btd` as a quantized `EinsumDense`
  decoder    a Llama-style decoder replayed from a HIP graph the program captured: the prompt's
             forward or one decode step, logits out
  quantize   the conversion of a float layer: build, `quantize(mode)`, the quantized variables out
  embedding  token ids into a quantized `Embedding`
"""

import math
import warnings

import torch

from keras_amd.decoder_harness import LlamaStyleDecoder
from keras_amd.layers import Dense, EinsumDense, Embedding
from keras_amd.quantization_config import Int4QuantizationConfig

# The largest listed Dense product; a drawn case stays at or below it.
DENSE_MOST_MACS = 4096 * 8192 * 8192
DENSE_MOST_WEIGHTS = 8192 * 8192

# Widths met in practice: model and feed-forward widths, multiples of 128 or not.
WIDTHS = (768, 960, 1024, 1280, 1600, 2048, 2560, 3072, 3200, 4096, 4544, 5120, 5632, 6400, 8192,
          11008, 13824, 14336)


def listed():
    return [
        # one layer of a served model under the default float32 policy, a small batch
        dict(name="dense_int8_f32_16", kind="dense", mode="int8", group=0, dtype="float32",
             rows=16, k=4096, n=4096),
        # weight-only int4, one token: the smallest call, all latency and weight bytes
        dict(name="dense_int4_bf16_1", kind="dense", mode="int4", group=-1, dtype="bfloat16",
             rows=1, k=8192, n=8192),
        # the default policy and the default grouping at a small decode batch
        dict(name="dense_int4_f32_8", kind="dense", mode="int4", group=128, dtype="float32",
             rows=8, k=4096, n=14336),
        # a short prompt, or a large decode batch, through a feed-forward layer
        dict(name="dense_int4_bf16_96", kind="dense", mode="int4", group=128, dtype="bfloat16",
             rows=96, k=4096, n=14336),
        # a model width that is no multiple of the group (1600 = 12.5 groups of 128)
        dict(name="dense_int4_bf16_300_ragged", kind="dense", mode="int4", group=128, dtype="bfloat16",
             rows=300, k=1600, n=6400),
        # the same widths, int8, default policy, a batch that is no multiple of a tile
        dict(name="dense_int8_f32_1000_ragged", kind="dense", mode="int8", group=0, dtype="float32",
             rows=1000, k=1600, n=6400),
        # attention projection of eight prompts of 512 tokens
        dict(name="einsum_int8_bf16_8x512", kind="einsum", mode="int8", group=0, dtype="bfloat16",
             equation="btd,dnh->btnh", batch=8, tokens=512, d=4096, heads=32),
        # the large int8 product (4096 tokens of prefill)
        dict(name="dense_int8_bf16_4096", kind="dense", mode="int8", group=0, dtype="bfloat16",
             rows=4096, k=8192, n=8192),
        # one greedy step of a decoder at batch 1 (eight blocks of the 32: time per block is the same)
        dict(name="decoder_int4_step_b1", kind="decoder", mode="int4", phase="step", batch=1,
             tokens=128, layers=8, d=4096, ffn=14336),
        # its prompt at batch 8: 1024 rows through every layer
        dict(name="decoder_int4_prompt_b8", kind="decoder", mode="int4", phase="prompt", batch=8,
             tokens=128, layers=8, d=4096, ffn=14336),
        # conversion of a feed-forward layer that lives on the device
        dict(name="quantize_int4_4096x14336", kind="quantize", mode="int4", group=128, k=4096, n=14336),
        # the token embedding of eight prompts of 512 tokens
        dict(name="embedding_int8_8x512", kind="embedding", mode="int8", group=0, dtype="float32",
             vocab=32000, d=4096, tokens=4096),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _mode(rng):
    mode = rng.choice(("int8", "int4"))
    return mode, 0 if mode == "int8" else rng.choice((128, 128, -1))


def draw(rng):
    kind = rng.choice(("dense",) * 6 + ("einsum", "decoder", "quantize", "embedding"))
    if kind == "dense":
        mode, group = _mode(rng)
        while True:
            k, n = rng.choice(WIDTHS), rng.choice(WIDTHS)
            if rng.random() < 0.2:
                n = _log(rng, 1000, 8000)  # a head of any size
            if k * n <= DENSE_MOST_WEIGHTS:
                break
        rows = _log(rng, 1, min(4096, DENSE_MOST_MACS // (k * n)))
        return dict(kind=kind, mode=mode, group=group, dtype=rng.choice(("float32", "bfloat16")),
                    rows=rows, k=k, n=n)
    if kind == "einsum":
        mode, group = _mode(rng)
        tokens = rng.choice((1, _log(rng, 2, 512)))
        return dict(kind=kind, mode=mode, group=group, dtype=rng.choice(("float32", "bfloat16")),
                    equation=rng.choice(("btd,dnh->btnh", "btnh,nhd->btd")), batch=rng.randint(1, 8),
                    tokens=tokens, d=rng.choice((1024, 2048, 4096)), heads=rng.choice((8, 16, 32)))
    if kind == "decoder":
        d, ffn = rng.choice(((2048, 5632), (4096, 11008), (4096, 14336)))
        # (prompts in int4 only: a bfloat16 ulp between two layers moves int8 activations by a step, so
        # the logits of two correct int8 decoders are 5 % apart and their outputs say little)
        mode, phase = rng.choice((("int4", "step"), ("int4", "prompt"), ("int8", "step")))
        return dict(kind=kind, mode=mode, phase=phase, batch=rng.randint(1, 8), tokens=_log(rng, 16, 128),
                    layers=rng.randint(2, 8), d=d, ffn=ffn)
    if kind == "quantize":
        mode, group = _mode(rng)
        while True:
            k, n = rng.choice(WIDTHS), rng.choice(WIDTHS)
            if k * n <= DENSE_MOST_WEIGHTS:
                break
        return dict(kind=kind, mode=mode, group=group, k=k, n=n)
    mode, group = _mode(rng)
    return dict(kind=kind, mode=mode, group=group, dtype=rng.choice(("float32", "bfloat16")),
                vocab=rng.choice((30522, 32000, 50257)), d=rng.choice((768, 1024, 1600, 4096)),
                tokens=_log(rng, 1, 8192))


# ---- what a program has in hand before the call ----------------------------------------------------
def _config(case):
    return Int4QuantizationConfig(block_size=case["group"]) if case["mode"] == "int4" else None


def _policy(dtype):
    # float32 variables either way; bfloat16 compute is the mixed policy
    return "mixed_bfloat16" if dtype == "bfloat16" else "float32"


def _uniform(gen, fan_in, fan_out):
    limit = math.sqrt(6.0 / (fan_in + fan_out))
    return lambda shape, dtype: ((torch.rand(shape, generator=gen, device="cuda") * 2 - 1) * limit).to(dtype)


def _bias(gen):
    return lambda shape, dtype: (torch.randn(shape, generator=gen, device="cuda") * 0.02).to(dtype)


def _torch_dtype(name):
    return torch.bfloat16 if name == "bfloat16" else torch.float32


def _prepare_dense(case, gen):
    layer = Dense(case["n"], dtype=_policy(case["dtype"]), device="cuda:0",
                  kernel_initializer=_uniform(gen, case["k"], case["n"]), bias_initializer=_bias(gen))
    layer.build((None, case["k"]))
    layer.quantize(case["mode"], config=_config(case))
    x = torch.randn(case["rows"], case["k"], generator=gen, device="cuda").to(_torch_dtype(case["dtype"]))
    layer(x)  # a server has called its layers before the first request
    return dict(call=layer, x=x)


def _prepare_einsum(case, gen):
    d, heads = case["d"], case["heads"]
    h = d // heads
    if case["equation"] == "btd,dnh->btnh":
        out, row = (None, heads, h), (d,)
    else:
        out, row = (None, d), (heads, h)
    layer = EinsumDense(case["equation"], out, dtype=_policy(case["dtype"]), device="cuda:0",
                        kernel_initializer=_uniform(gen, d, d))
    layer.build((None, None) + row)
    layer.quantize(case["mode"], config=_config(case))
    x = torch.randn(case["batch"], case["tokens"], *row, generator=gen, device="cuda")
    x = x.to(_torch_dtype(case["dtype"]))
    layer(x)
    return dict(call=layer, x=x)


class _Replay:
    """A forward of the decoder as a captured graph: inputs and logits are the graph's own buffers."""

    def __init__(self, model, ids, pos, cache):
        self.model, self.cache, self.ids, self.pos = model, cache, ids, pos
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            model.forward(ids, pos, cache)  # first-call set-up happens outside the capture
            self.graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(self.graph, stream=side):
                self.logits = model.forward(ids, pos, cache)
        torch.cuda.current_stream().wait_stream(side)

    def __call__(self, ids):
        self.ids.copy_(ids)
        self.graph.replay()
        return self.logits


def _prepare_decoder(case, gen, seed):
    model = LlamaStyleDecoder(vocab=32000, d_model=case["d"], n_heads=case["d"] // 128, ffn_dim=case["ffn"],
                              n_layers=case["layers"], max_len=256, dtype="mixed_bfloat16", device="cuda:0",
                              seed=seed, init_on_device=True)
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")  # the norms have no quantized form
        model.quantize(case["mode"])
    batch, tokens = case["batch"], case["tokens"]
    prompt = torch.randint(0, 32000, (batch, tokens), generator=gen, device="cuda")
    cache = model.new_cache(batch)
    if case["phase"] == "prompt":
        return dict(call=_Replay(model, prompt.clone(), torch.arange(tokens, device="cuda"), cache), x=prompt)
    model.forward(prompt, torch.arange(tokens, device="cuda"), cache)  # the rows a step attends to
    token = torch.randint(0, 32000, (batch, 1), generator=gen, device="cuda")
    pos = torch.full((1,), tokens, dtype=torch.int64, device="cuda")
    return dict(call=_Replay(model, token.clone(), pos, cache), x=token)


def _prepare_quantize(case, gen):
    kernel = _uniform(gen, case["k"], case["n"])((case["k"], case["n"]), torch.float32)

    def convert(kernel):
        layer = Dense(case["n"], dtype="mixed_bfloat16", device="cuda:0", use_bias=False,
                      kernel_initializer=lambda shape, dtype: kernel.to(dtype))
        layer.build((None, case["k"]))
        layer.quantize(case["mode"], config=_config(case))
        out = [layer._kernel.value, layer.kernel_scale.value]
        if case["group"] > 0:
            out.append(layer.kernel_zero.value)
        return out

    return dict(call=convert, x=kernel)


def _prepare_embedding(case, gen):
    layer = Embedding(case["vocab"], case["d"], dtype=_policy(case["dtype"]), device="cuda:0",
                      embeddings_initializer=_bias(gen))
    layer.build()
    layer.quantize(case["mode"], config=_config(case))
    layer.check_ids = False  # as a serving loop runs it: no read back from the device per call
    ids = torch.randint(0, case["vocab"], (case["tokens"],), generator=gen, device="cuda")
    layer(ids)
    return dict(call=layer, x=ids)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    kind = case["kind"]
    if kind == "dense":
        return _prepare_dense(case, gen)
    if kind == "einsum":
        return _prepare_einsum(case, gen)
    if kind == "decoder":
        return _prepare_decoder(case, gen, int(seed))
    if kind == "quantize":
        return _prepare_quantize(case, gen)
    return _prepare_embedding(case, gen)


def run(state):
    return state["call"](state["x"])


# ---- what a pass cannot do without -------------------------------------------------------------------
def _weight_bytes(mode, group, k, n):
    """Stored weights and their scales: a byte per weight, or half a byte (a pair per byte along n) with
    float32 scales and int8 zero points per group of k."""
    if mode == "int8":
        return k * n + 4 * n
    groups = -(-k // group) if group > 0 else 0
    return k * (-(-n // 2)) + (5 * groups * n if groups else 4 * n)


def _matmul_work(mode, group, size, rows, k, n, bias):
    return dict(bytes=_weight_bytes(mode, group, k, n) + size * rows * (k + n) + (4 * n if bias else 0),
                flops=2 * rows * k * n)


def work(case):
    kind = case["kind"]
    size = 2 if case.get("dtype") == "bfloat16" else 4
    if kind == "dense":
        return _matmul_work(case["mode"], case["group"], size, case["rows"], case["k"], case["n"], True)
    if kind == "einsum":
        return _matmul_work(case["mode"], case["group"], size, case["batch"] * case["tokens"], case["d"], case["d"],
                            False)
    if kind == "decoder":
        d, ffn, mode, group = case["d"], case["ffn"], case["mode"], 0 if case["mode"] == "int8" else 128
        new = 1 if case["phase"] == "step" else case["tokens"]
        seen = case["tokens"] + 1 if case["phase"] == "step" else case["tokens"]
        rows = case["batch"] * new
        layer_bytes = (4 * _weight_bytes(mode, group, d, d) + 2 * _weight_bytes(mode, group, d, ffn)
                       + _weight_bytes(mode, group, ffn, d))
        # keys and values of every position so far, read or written once
        cache_bytes = 2 * 2 * case["batch"] * seen * d
        head = _weight_bytes(mode, group, d, 32000)
        causal = seen if case["phase"] == "step" else (new + 1) / 2
        flops = case["layers"] * (2 * rows * (4 * d * d + 3 * d * ffn) + 4 * rows * causal * d)
        return dict(bytes=case["layers"] * (layer_bytes + cache_bytes) + head + 4 * case["batch"] * 32000,
                    flops=flops + 2 * case["batch"] * d * 32000)
    if kind == "quantize":
        k, n = case["k"], case["n"]
        return dict(bytes=4 * k * n + _weight_bytes(case["mode"], case["group"], k, n), flops=4 * k * n)
    d, tokens = case["d"], case["tokens"]
    row = _weight_bytes(case["mode"], 0, d, 1) if case["mode"] == "int8" else (
        -(-d // 2) + (5 * -(-d // case["group"]) if case["group"] > 0 else 4))
    return dict(bytes=tokens * (8 + 4 * d) + min(tokens, case["vocab"]) * row, flops=tokens * d)


def tolerance(case):
    """How far another correct implementation may be from this one.

    int8 layers, conversions and lookups reproduce the reference's rounding chain bit for bit (exact
    int32 sums, every later step one rounding), so nothing may differ.  Weight-only int4 sums in some
    order: against 64-bit sums a bfloat16 result is 2.9e-3 off (2-norm) and a float32 one, whose
    operands travel as pairs of bfloat16, 1.2e-5.  The decoder carries such differences through its
    blocks: eight of them with every sum in another order are 1.4e-2 to 1.7e-2 apart."""
    if case["kind"] == "decoder":
        return {"rel": 3e-2, "max": 0.3}
    if case["mode"] == "int8" or case["kind"] in ("quantize", "embedding"):
        return "exact"
    if case["dtype"] == "bfloat16":
        return {"rel": 1.1e-2, "max": 4.5e-2}
    return {"rel": 5e-5, "max": 2e-4}
