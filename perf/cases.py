"""The work a program that serves quantized models has this package do, as timed cases.

Four kinds, each through the public entry points on device tensors:

``linear``      one ``quantized_linear`` with the plan a program keeps: a decode step's contraction of one or a few
                vectors, a batch, a prompt's chunk; every codec, both activation modes, with and without bias
``attention``   paged key/value-cache attention of one layer: a decode step (one token per sequence), a prompt's chunk
                (many), every slab type, equal and ragged contexts
``decode``      one step of the batched decode loop as its captured graph: layers, output projection, greedy token
``embedding``   the lookup of a prompt's token ids in a packed table

Sizes: those of the benchmark configurations (``effect_torch_amd.synth.CONFIGS``, ``LlamaShape``) and, where they are
odd, generic ones near them.
"""
import importlib
import math

import torch

et = importlib.import_module("effect-torch_amd")

BLOCK = 16  # positions per block of the paged cache
SLABS = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "u8": torch.uint8}


# ---------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # One vector against a small square matrix: an attention projection of single-user decode. Latency.
        linear("linear_q8_0_m1", "Q8_0", 4096, 4096, 1),
        # One vector against a feed-forward matrix: the contraction the headline metric is quoted on.
        linear("linear_q4_k_m1", "Q4_K", 14336, 4096, 1),
        # A handful of sequences (or draft tokens being verified) on the wide down projection.
        linear("linear_q4_k_m5_wide", "Q4_K", 4096, 14336, 5),
        # An odd decode batch on the codec that mixed-precision files give their more sensitive matrices; with a bias.
        linear("linear_q6_k_m27", "Q6_K", 14336, 4096, 27, bias=True),
        # A prompt's chunk on a feed-forward matrix, f32 accuracy; not a whole number of tiles.
        linear("linear_q4_k_m1000", "Q4_K", 14336, 4096, 1000),
        # A prompt's chunk in the int8-activation mode on the down projection.
        linear("linear_q8_0_int8_m512", "Q8_0", 4096, 14336, 512, mode="int8"),
        # One decode step's attention for a full batch over half-float slabs.
        attention("attention_decode_32x2048", 32, 1, 2048, "f16"),
        # A few long sequences of different lengths over the int8-quantized slabs that long contexts are kept in.
        attention("attention_decode_long_u8", 3, 1, 30000, "u8", ragged=True),
        # Two prompts' chunks at the end of contexts of 2000 positions.
        attention("attention_chunk_2x500", 2, 500, 2000, "f16"),
        # Single-user decode: one token of one sequence through the layers and the output projection.
        decode("decode_step_1", 1, 1000),
        # The full decode batch of the end-to-end configuration (four of its layers).
        decode("decode_step_32", 32, 2048),
        # A long prompt's ids, looked up in a packed vocabulary table.
        embedding("embedding_q4_k_5000", "Q4_K", 128256, 4096, 5000),
    ]


def linear(name, codec, rows, columns, vectors, mode="f32", bias=False):
    return named(name, kind="linear", codec=codec, rows=rows, columns=columns, vectors=vectors, mode=mode, bias=bias)


def attention(name, slots, tokens, context, slab, ragged=False, heads=32, kv_heads=8, width=128):
    return named(name, kind="attention", slots=slots, tokens=tokens, context=context, slab=slab, ragged=ragged, heads=heads,
                 kv_heads=kv_heads, width=width)


def decode(name, slots, context, codec="Q4_K", layers=4, hidden=4096, ffn=14336, heads=32, kv_heads=8, vocab=128256):
    return named(name, kind="decode", slots=slots, context=context, codec=codec, layers=layers, hidden=hidden, ffn=ffn,
                 heads=heads, kv_heads=kv_heads, vocab=vocab)


def embedding(name, codec, rows, columns, ids):
    return named(name, kind="embedding", codec=codec, rows=rows, columns=columns, ids=ids)


def named(name, **case):
    return dict(case, name=name) if name else case


def log_int(rng, low, high):
    """An integer between ``low`` and ``high``, spread over its logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "attention", "attention", "decode", "embedding"])
    if kind == "linear":
        codec = rng.choice(["Q4_K", "Q4_K", "Q6_K", "Q5_K", "Q3_K", "Q2_K", "Q8_0", "Q4_0"])
        mode = "int8" if codec in ("Q8_0", "Q4_0", "Q4_K") and rng.random() < 0.3 else "f32"
        rows, columns = log_int(rng, 512, 16384), 256 * log_int(rng, 4, 56)
        most = 14336 * 4096 * 1000 // (rows * columns)
        # half of the calls belong to decode steps, half to prompts
        vectors = log_int(rng, 1, 64) if rng.random() < 0.5 else log_int(rng, 33, max(33, min(1000, most)))
        return linear(None, codec, rows, columns, vectors, mode, rng.random() < 0.25)
    if kind == "attention":
        heads, kv_heads, width = rng.choice([(32, 8, 128), (32, 8, 128), (16, 8, 64), (32, 32, 128), (24, 8, 128)])
        slab = rng.choice(["f16", "f16", "bf16", "u8", "f32"])
        if rng.random() < 0.5:
            slots = log_int(rng, 1, 64)
            return attention(None, slots, 1, log_int(rng, 64, 65536 // slots), slab, rng.random() < 0.5, heads, kv_heads, width)
        slots = log_int(rng, 1, 8)
        tokens = log_int(rng, 2, 1000 // slots)
        return attention(None, slots, tokens, log_int(rng, max(tokens, 64), 2000), slab, rng.random() < 0.5, heads, kv_heads, width)
    if kind == "decode":
        slots = log_int(rng, 1, 32)
        hidden, ffn, heads, kv_heads = rng.choice([(4096, 14336, 32, 8), (2048, 5632, 16, 4)])
        return decode(None, slots, log_int(rng, 64, 2048), rng.choice(["Q4_K", "Q4_K", "Q5_K", "Q8_0", "Q6_K"]),
                      rng.choice([2, 3]), hidden, ffn, heads, kv_heads, rng.choice([32000, 128256]))
    return embedding(None, rng.choice(["Q4_K", "Q6_K", "Q8_0", "Q5_K", "Q3_K"]), rng.choice([32000, 128256]),
                     rng.choice([2048, 4096]), log_int(rng, 1, 5000))


# ---------------------------------------------------------------------------------------------- inputs
def generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def packed_weight(codec, rows, columns, gen):
    """``[rows, row_bytes]`` u8: quants and sub-scales uniform over their range, half-float block scales |N(0, 1)| times
    the scale of the benchmark configurations."""
    synth = importlib.import_module("effect-torch_amd.synth")
    size = codec.block_bytes
    data = torch.randint(0, 256, (rows * (columns // codec.block_values), size), generator=gen, device="cuda", dtype=torch.uint8)
    if codec == et.GgmlQuant.Q8_0:  # -128 is never produced by a quantiser
        quants = data[:, 2:]
        quants[quants == 128] = 129
    for offset in synth._FP16_FIELDS[int(codec)]:
        scale = torch.randn(data.shape[0], generator=gen, device="cuda").abs() * synth.DEFAULT_SCALE[int(codec)]
        data[:, offset:offset + 2] = scale.to(torch.float16).view(torch.uint8).reshape(-1, 2)
    return data.reshape(rows, -1)


def contexts(case):
    """The context of every slot after the step: all alike, or between a third and the whole of ``context``."""
    most, slots = case["context"], case["slots"]
    if not case.get("ragged"):
        return [most] * slots
    least = max(case.get("tokens", 1), most // 3, 1)
    return [most - (i * 7919) % (most - least + 1) for i in range(slots)]


def pages(lengths, gen):
    """A block table that places every sequence's blocks anywhere in the pool, and the pool's positions."""
    per_slot = -(-max(lengths) // BLOCK)
    table = torch.randperm(len(lengths) * per_slot, generator=gen, device="cuda").reshape(len(lengths), per_slot)
    return table.to(torch.int32), len(lengths) * per_slot * BLOCK


def slabs(slab, positions, kv_heads, width, gen):
    """Filled K and V slabs and, for the int8-quantized tier, their scales."""
    shape = (positions, kv_heads, width)
    if slab == "u8":
        pair = [torch.randint(1, 256, shape, generator=gen, device="cuda", dtype=torch.uint8) for _ in range(2)]
        scales = [torch.rand(shape[:2], generator=gen, device="cuda") * 0.01 + 0.015 for _ in range(2)]
        return pair, {"k_scales": scales[0], "v_scales": scales[1]}
    return [torch.randn(shape, generator=gen, device="cuda").to(SLABS[slab]) for _ in range(2)], {}


def prepare(case, seed):
    return {"linear": prepare_linear, "attention": prepare_attention, "decode": prepare_decode,
            "embedding": prepare_embedding}[case["kind"]](case, generator(seed))


def prepare_linear(case, gen):
    codec, mode = et.GgmlQuant[case["codec"]], et.ActivationMode[case["mode"].upper()]
    shape = (case["rows"], case["columns"])
    weight = packed_weight(codec, *shape, gen)
    x = torch.randn(case["vectors"], case["columns"], generator=gen, device="cuda")
    bias = torch.randn(case["rows"], generator=gen, device="cuda") if case["bias"] else None
    plan = et.linear_requirements(x, weight, bias, codec, shape, mode)
    return {"run": run_linear, "codec": codec, "x": x, "weight": weight, "bias": bias, "plan": plan,
            "y": torch.empty(plan.output_shape, device="cuda"),
            "workspace": torch.empty(max(plan.workspace_bytes, 16), dtype=torch.uint8, device="cuda")}


def prepare_attention(case, gen):
    lengths, tokens = contexts(case), case["tokens"]
    table, positions = pages(lengths, gen)
    (k_slab, v_slab), scales = slabs(case["slab"], positions, case["kv_heads"], case["width"], gen)
    advances = torch.full((case["slots"],), tokens, dtype=torch.int32, device="cuda")
    cursors = torch.tensor(lengths, dtype=torch.int32, device="cuda") - tokens
    layer = et.KvLayer(k_slab, v_slab, BLOCK, table, cursors, advances, max(lengths), **scales)
    rows = lambda heads: torch.randn(case["slots"], heads, tokens, case["width"], generator=gen, device="cuda")  # noqa: E731
    q, k, v = rows(case["heads"]), rows(case["kv_heads"]), rows(case["kv_heads"])
    return {"run": run_attention, "layer": layer, "q": q, "k": k, "v": v, "out": torch.empty_like(q),
            "scale": case["width"] ** -0.5, "workspace": et.kv_attention_workspace(layer, case["heads"], tokens)}


def prepare_decode(case, gen):
    codec, slots = et.GgmlQuant[case["codec"]], case["slots"]
    shape = et.LlamaShape(hidden=case["hidden"], heads=case["heads"], kv_heads=case["kv_heads"], ffn=case["ffn"],
                          vocab=case["vocab"], layers=case["layers"])
    shapes = shape.linear_shapes()
    weights = [{name: packed_weight(codec, *size, gen) for name, size in shapes.items() if name != "head"}
               for _ in range(shape.layers)]
    head = packed_weight(codec, *shapes["head"], gen)
    # norm weights around 1/16 keep the residual stream of random weights inside the slabs' half floats
    norm = lambda *size: ((1 + 0.1 * torch.randn(*size, shape.hidden, generator=gen, device="cuda")) / 16).half()  # noqa: E731
    norms, final_norm = [norm(2) for _ in range(shape.layers)], norm()
    table_rows = torch.randn(shape.vocab, shape.hidden, generator=gen, device="cuda", dtype=torch.float16)
    lengths = contexts(case)
    table, positions = pages(lengths, gen)
    start = {"tokens": torch.randint(0, shape.vocab, (slots,), generator=gen, device="cuda", dtype=torch.int32),
             "cursors": torch.tensor(lengths, dtype=torch.int32, device="cuda") - 1}
    tokens, cursors = start["tokens"].clone(), start["cursors"].clone()
    advances = torch.ones(slots, dtype=torch.int32, device="cuda")
    kv = [et.KvLayer(*slabs("f16", positions, shape.kv_heads, shape.head_dim, gen)[0], BLOCK, table, cursors, advances,
                     max(lengths)) for _ in range(shape.layers)]
    # the fused step where every contraction takes prepared activations, else one launch sequence per operator
    fused = all(et.RawLinear(codec, *size, slots).prepared_input_bytes > 0 for size in shapes.values())
    decoder = et.LlamaDecoder(shape, codec, slots, weights, head, norms, final_norm, table_rows, kv, tokens, fused=fused)
    state = {"run": run_decode, "decoder": decoder, "start": start, "tokens": tokens, "cursors": cursors, "kv": kv}
    begin_step(state)
    decoder.step()
    begin_step(state)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        decoder.step()
    begin_step(state)
    return dict(state, graph=graph)


def prepare_embedding(case, gen):
    codec, shape = et.GgmlQuant[case["codec"]], (case["rows"], case["columns"])
    weight = packed_weight(codec, *shape, gen)
    ids = torch.randint(0, case["rows"], (case["ids"],), generator=gen, device="cuda")
    plan = et.embedding_requirements(ids, weight, codec, shape)
    return {"run": run_embedding, "codec": codec, "ids": ids, "weight": weight, "plan": plan,
            "out": torch.empty(plan.output_shape, device="cuda")}


# ---------------------------------------------------------------------------------------------- one pass
def run(state):
    return state["run"](state)


def run_linear(s):
    et.linear_into(s["x"], s["weight"], s["bias"], s["codec"], s["y"], s["plan"], workspace=s["workspace"])
    return s["y"]


def run_attention(s):
    layer = s["layer"]
    et.kv_attention_into(layer, s["q"], s["k"], s["v"], s["scale"], None, s["out"], workspace=s["workspace"],
                         synchronize=False)
    return {"out": s["out"], "k_slab": layer.k_slab, "v_slab": layer.v_slab, "k_scales": layer.k_scales,
            "v_scales": layer.v_scales}


def begin_step(s):
    """What a server writes before a step: which token every slot feeds, and at which position."""
    s["tokens"].copy_(s["start"]["tokens"])
    s["cursors"].copy_(s["start"]["cursors"])


def run_decode(s):
    begin_step(s)
    s["graph"].replay()
    return {"logits": s["decoder"].logits, "tokens": s["tokens"], "cursors": s["cursors"],
            "slabs": [(layer.k_slab, layer.v_slab) for layer in s["kv"]]}


def run_embedding(s):
    et.embedding_into(s["ids"], s["weight"], s["codec"], s["out"], s["plan"], synchronize=False)
    return s["out"]


# ---------------------------------------------------------------------------------------------- what a pass cannot do without
def packed_bytes(codec, rows, columns):
    return rows * et.GgmlQuant[codec].encoded_row_bytes(columns)


def attention_work(slots_tokens, lengths, heads, kv_heads, width, slab):
    """Every cached row of the contexts read once, the new rows written once; q.k and p.v over the causal positions."""
    row = width * {"f32": 4, "f16": 2, "bf16": 2, "u8": 1}[slab] + (4 if slab == "u8" else 0)
    new = slots_tokens * len(lengths)
    seen = sum(slots_tokens * n - slots_tokens * (slots_tokens - 1) // 2 for n in lengths)
    return {"bytes": 2 * kv_heads * row * sum(lengths) + 4 * width * new * (2 * heads + 2 * kv_heads),
            "flops": 4 * heads * width * seen}


def work(case):
    if case["kind"] == "linear":
        m, n, k = case["vectors"], case["rows"], case["columns"]
        return {"bytes": packed_bytes(case["codec"], n, k) + 4 * m * (k + n) + (4 * n if case["bias"] else 0), "flops": 2 * m * n * k}
    if case["kind"] == "attention":
        return attention_work(case["tokens"], contexts(case), case["heads"], case["kv_heads"], case["width"], case["slab"])
    if case["kind"] == "embedding":
        row = packed_bytes(case["codec"], 1, case["columns"])
        return {"bytes": case["ids"] * (8 + row + 4 * case["columns"]), "flops": 2 * case["ids"] * case["columns"]}
    shape = et.LlamaShape(hidden=case["hidden"], heads=case["heads"], kv_heads=case["kv_heads"], ffn=case["ffn"], vocab=case["vocab"])
    slots, layers = case["slots"], case["layers"]
    sizes = [size for name, size in shape.linear_shapes().items() for _ in range(1 if name == "head" else layers)]
    attended = attention_work(1, contexts(case), case["heads"], case["kv_heads"], shape.head_dim, "f16")
    return {"bytes": sum(packed_bytes(case["codec"], *size) for size in sizes) + layers * attended["bytes"] +
            slots * (2 * shape.hidden + 4 * shape.vocab) + layers * 4 * shape.hidden,
            "flops": sum(2 * slots * n * k for n, k in sizes) + layers * attended["flops"]}


def tolerance(case):
    """Against the same pass in 64 bits: contractions (integer sums, f32 scales) 0.9 to 2.0e-7, attention 1.6 to 3.3e-7. A
    decode step's logits differ by up to 2.6e-5 where a key or value of the step rounds to the next half float."""
    if case["kind"] == "embedding":
        return "exact"
    return {"rel": 1e-4 if case["kind"] == "decode" else 2e-6}
