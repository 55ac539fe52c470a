"""One-vector contractions with the operators around them in one launch (``LinearStep``), against the oracle's operators
one after the other, and the decode step of a single sequence that is made of them.

Sizes: one, two and four slices of columns (4096 each, the last one ragged), one to eight rows per wave and the loop above
that, matrices whose rows end inside a wave's rows or a workgroup's range. Bars: ``close`` of test_gpu_parity (f32 bars); the
sums alone: the bits of the launch per matrix. Chained steps against the same step with one operator per launch."""
import numpy as np
import pytest
import torch

import oracle
from effect_torch_amd import synth
import test_gpu_decode_step
from test_gpu_decode_step import test_decode_steps_follow_the_oracle_chain as _follow_the_oracle_chain
from test_gpu_parity import close

pytestmark = pytest.mark.gpu

CODECS = ["Q2_K", "Q3_K", "Q4_K", "Q5_K", "Q6_K", "Q4_0", "Q8_0"]


def tensors(device, *arrays):
    return [torch.from_numpy(a).to(device) for a in arrays]


def case(codec, rows, columns, seed):
    rng = np.random.default_rng(seed)
    code = getattr(synth, codec)
    weights = [synth.random_weight(code, r, columns, rng) for r in rows]
    x = synth.random_activations(1, columns, rng)
    norm = (1 + 0.1 * rng.standard_normal(columns)).astype(np.float16)
    residuals = [rng.standard_normal((1, r)).astype(np.float32) for r in rows]
    return code, weights, x, norm, residuals


def linear(code, weight, rows, columns, x):
    return oracle.linear_into(code, rows, columns, x, weight)


@pytest.mark.parametrize("codec", CODECS)
@pytest.mark.parametrize("rows,columns,normed", [((1,), 256, True), ((300, 77, 2049), 1792, True), ((2048, 513), 4096, False),
                                                 ((7, 2500, 40, 3000), 4352, True), ((4099, 61), 6144, False),
                                                 ((2047,), 14336, False), ((4500,), 8448, True)])
def test_contractions_with_norm_and_residuals(et, device, codec, rows, columns, normed):
    code, weights, x, norm, residuals = case(codec, rows, columns, 0x57E9 + columns + len(rows))
    step = et.LinearStep([et.RawLinear(et.GgmlQuant[codec], r, columns, 1) for r in rows])
    assert step.supported
    xd, nd = tensors(device, x, norm)
    wd, ys = tensors(device, *weights), tensors(device, *residuals)
    plain = len(rows) - 1  # the last of several members has no residual
    added = [y if i != plain or len(rows) == 1 else None for i, y in enumerate(ys)]  # in place
    step.enqueue(xd, wd, ys, norm=(nd, 1e-5) if normed else None, residuals=added)
    torch.cuda.synchronize()
    h = oracle.rms_norm(x, norm.astype(np.float32), 1e-5) if normed else x
    for i, r in enumerate(rows):
        want = linear(code, weights[i], r, columns, h)
        close(ys[i].cpu().numpy(), want if added[i] is None else want + residuals[i])


@pytest.mark.parametrize("codec", CODECS)
@pytest.mark.parametrize("rows,columns", [(1, 256), (1500, 2048), (2600, 4096), (4200, 4096), (700, 4352), (5632, 2048)])
def test_gate_and_up_with_silu(et, device, codec, rows, columns):
    code, (gate, up), x, norm, _ = case(codec, (rows, rows), columns, 0x51D + rows)
    plan = et.RawLinear(et.GgmlQuant[codec], rows, columns, 1)
    step = et.LinearStep([plan, plan], silu_mul=True)
    assert step.supported
    # an odd number of half floats into its buffer: a norm weight that is not 8-byte aligned
    xd, nd = tensors(device, x, np.concatenate([norm[:1], norm]))
    y = torch.empty(1, rows, device=device)
    step.enqueue(xd, tensors(device, gate, up), [y], norm=(nd[1:], 1e-6))
    torch.cuda.synchronize()
    h = oracle.rms_norm(x, norm.astype(np.float32), 1e-6)
    close(y.cpu().numpy(), oracle.silu_mul(linear(code, gate, rows, columns, h), linear(code, up, rows, columns, h)))


@pytest.mark.parametrize("codec", CODECS)
@pytest.mark.parametrize("rows,columns", [((1000, 77), 1792), ((14336,), 4096), ((2500, 40), 4352), ((4099,), 14336)])
def test_the_sums_are_those_of_a_launch_per_matrix(et, device, codec, rows, columns):
    # the same limbs, folds and order: the same bits, also where an activation is not finite
    code, weights, x, norm, _ = case(codec, rows, columns, 0xB175 + columns)
    plans = [et.RawLinear(et.GgmlQuant[codec], r, columns, 1) for r in rows]
    step, wd = et.LinearStep(plans), tensors(device, *weights)
    for spoilt in (None, np.nan, np.inf, -np.inf):
        if spoilt is not None:
            x[0, columns - 3] = spoilt
        xd, = tensors(device, x)
        ys, want = ([torch.full((1, r), 7.0, device=device) for r in rows] for _ in range(2))
        step.enqueue(xd, wd, ys)
        for plan, weight, y in zip(plans, wd, want):
            plan.enqueue(xd, weight, None, y, torch.empty(max(plan.requirements.workspace_bytes, 16), dtype=torch.uint8, device=device))
        for y, w in zip(ys, want):
            assert torch.equal(y.isnan(), w.isnan()) and torch.equal(y.nan_to_num(), w.nan_to_num())


@pytest.mark.parametrize("columns", [256, 1792, 4096, 4352, 14336])
@pytest.mark.parametrize("weight", ["f32", "none"])
def test_norms_with_float_weights_or_none(et, device, columns, weight):
    rows = 300
    code, (packed,), x, norm, (residual,) = case("Q4_K", (rows,), columns, 0xF32 + columns)
    step = et.LinearStep([et.RawLinear(et.GgmlQuant.Q4_K, rows, columns, 1)])
    norm = (norm.astype(np.float32) + np.float32(1e-5)) if weight == "f32" else None  # no half floats
    for spoilt in (False, True):
        if spoilt:
            x[:] = np.inf
        xd, wd, rd = tensors(device, x, packed, residual)
        nd = None
        if norm is not None:
            nd, = tensors(device, np.concatenate([norm[:1], norm]))
            nd = nd[1:]  # 4-byte aligned only
        y = torch.empty(1, rows, device=device)
        step.enqueue(xd, [wd], [y], norm=(nd, 1e-5), residuals=[rd])
        got = y.cpu().numpy()
        if spoilt:
            assert np.isnan(got).all()
        else:
            close(got, linear(code, packed, rows, columns, oracle.rms_norm(x, norm, 1e-5)) + residual)


def test_what_has_no_such_launch_is_refused(et, device):
    plan = lambda *a, **k: et.RawLinear(et.GgmlQuant.Q4_K, *a, **k)  # noqa: E731
    one = plan(512, 1024, 1)
    assert et.LinearStep([one]).supported
    refused = [([plan(512, 1024, 2)], False), ([plan(512, 1024, 1, True)], False), ([one, plan(512, 2048, 1)], False),
               ([one, et.RawLinear(et.GgmlQuant.Q5_K, 512, 1024, 1)], False), ([one, plan(513, 1024, 1)], True), ([one], True),
               ([plan(64, 16640, 1)], False), ([plan(64, 8448, 1)] * 2, True)]
    for plans, silu_mul in refused:
        assert not et.LinearStep(plans, silu_mul).supported
    x, weight = torch.ones(1, 1024, device=device), torch.zeros(512, 576, dtype=torch.uint8, device=device)
    with pytest.raises(et.QuantizedError, match="no launch with the operators"):
        et.LinearStep(refused[1][0]).enqueue(x, [weight], [torch.empty(1, 512, device=device)])
    with pytest.raises(et.QuantizedError, match="overlaps the activations"):
        et.LinearStep([one]).enqueue(x, [weight], [x[:, 512:]])


@pytest.mark.parametrize("contexts", [(40, 41), (2030, 2060)], ids=["one_attention_launch_or_more", "context_2048"])
def test_decode_steps_of_one_sequence_follow_the_oracle_chain(et, device, contexts, monkeypatch):
    made = []
    model = test_gpu_decode_step.Model
    monkeypatch.setattr(test_gpu_decode_step, "Model", lambda *args: made.append(model(*args)) or made[-1])
    _follow_the_oracle_chain(et, device, False, 1, contexts)
    assert made[0].decoder.chained and made[0].decoder.project_in_attention


def small_decoder(et, device, codec, slab, head_dim, bound, chain):
    """Two layers, one sequence, eight query heads over two kv heads; every call makes the same one."""
    rng = np.random.default_rng(0x5DEC + head_dim)
    code = getattr(synth, codec)
    shape = et.LlamaShape(hidden=8 * head_dim, heads=8, kv_heads=2, head_dim=head_dim, ffn=1280, vocab=1000, layers=2)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)  # noqa: E731
    shapes = shape.linear_shapes()
    weights = [{name: dev(synth.random_weight(code, *size, rng)) for name, size in shapes.items() if name != "head"} for _ in range(2)]
    head = dev(synth.random_weight(code, *shapes["head"], rng))
    norm = lambda *size: dev((1 + 0.1 * rng.standard_normal((*size, shape.hidden))).astype(np.float32))  # noqa: E731
    norms, final_norm = [norm(2) for _ in range(2)], norm()
    embedding = dev(rng.standard_normal((shape.vocab, shape.hidden)).astype(np.float16))
    cursors, advances = (torch.full((1,), n, dtype=torch.int32, device=device) for n in (77, 1))
    table = dev(rng.permutation(8).reshape(1, 8).astype(np.int32))

    def layer():
        size = (128, 2, head_dim)
        if slab == torch.uint8:
            values = [dev(rng.integers(1, 256, size).astype(np.uint8)) for _ in range(2)]
            scales = {name: dev(rng.uniform(0.01, 0.03, size[:2]).astype(np.float32)) for name in ("k_scales", "v_scales")}
        else:
            values, scales = [dev(rng.standard_normal(size).astype(np.float32)).to(slab) for _ in range(2)], {}
        return et.KvLayer(*values, 16, table, cursors, advances, bound, **scales)

    tokens = torch.full((1,), 5, dtype=torch.int32, device=device)
    return et.LlamaDecoder(shape, et.GgmlQuant[codec], 1, weights, head, norms, final_norm, embedding, [layer(), layer()], tokens,
                           fused=False, chain=chain)


@pytest.mark.parametrize("codec,slab,head_dim,bound,attention,bar", [
    ("Q4_K", torch.float32, 64, 100, "kv_attend", 2e-6),
    ("Q6_K", torch.float16, 128, 5000, "kv_attend+kv_merge", 2e-3),
    ("Q8_0", torch.bfloat16, 64, 100, "kv_attend", 1e-2),
    ("Q5_K", torch.uint8, 128, 40000, "kv_bytes+kv_merge", 1e-2),
    ("Q4_0", torch.uint8, 64, 40000, "kv_bytes+kv_merge", 1e-2),
    ("Q3_K", torch.float32, 96, 100, "kv_attend_any", 2e-6),          # q and k are rotated by a launch of their own
])
def test_a_chained_step_is_that_of_its_operators_one_by_one(et, device, codec, slab, head_dim, bound, attention, bar):
    # Bar: f32 sums; where a row of the step rounds to the slab's next value the two part by that step (2^-11, 2^-9, 1/254 of the
    # row's largest) in one of 78 positions.
    one = small_decoder(et, device, codec, slab, head_dim, bound, chain=False)
    chained = small_decoder(et, device, codec, slab, head_dim, bound, chain=True)
    assert chained.chained and not one.chained
    assert et.kv_attention_variant(chained.kv[0], 8, 1).startswith(attention)
    assert chained.project_in_attention == (not attention.startswith("kv_attend_any"))
    relative = lambda got, want: ((got - want).norm() / want.norm()).item()  # noqa: E731
    for decoder in (one, chained):
        for name in ("h", "q", "k", "v", "up", "projected", "down"):
            getattr(decoder, name).fill_(float("nan"))
        decoder.step()
    torch.cuda.synchronize()
    for decoder in (one, chained):
        et.gather_rows_status_check(1000, decoder.status[0])
        for index in range(2):
            et.kv_attention_status_check(decoder.kv[index], 1, decoder.status[1 + index])
    assert relative(chained.logits, one.logits) <= bar
    assert torch.isfinite(one.logits).all() and one.cursors.item() == chained.cursors.item() == 78
    # one operator per launch: each has left its result behind
    assert all(torch.isfinite(getattr(one, name)).all() for name in ("h", "q", "k", "v", "up", "projected", "down"))
    for name, source, result in (("wo", one.attended, one.projected), ("down", one.gate, one.down)):
        want = torch.empty_like(result)
        one.plans[name].enqueue(source, one.weights[1][name], None, want, one.linear_ws)
        assert torch.equal(result, want)


def test_a_chained_step_as_a_replayed_graph(et, device):
    eager, graphed = (small_decoder(et, device, "Q4_K", torch.uint8, 128, 40000, chain=True) for _ in range(2))
    start = [t.clone() for layer in graphed.kv for t in (layer.k_slab, layer.v_slab, layer.k_scales, layer.v_scales)]
    graphed.step()  # warm up, then back to the start
    for tensor, value in zip([t for layer in graphed.kv for t in (layer.k_slab, layer.v_slab, layer.k_scales, layer.v_scales)], start):
        tensor.copy_(value)
    graphed.tokens.fill_(5)
    graphed.cursors.fill_(77)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        graphed.step()
    for _ in range(4):
        eager.step()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in ((eager.logits, graphed.logits), (eager.tokens, graphed.tokens), (eager.cursors, graphed.cursors)):
            assert torch.equal(a, b)
    for a, b in zip(eager.kv, graphed.kv):
        assert torch.equal(a.k_slab, b.k_slab) and torch.equal(a.v_slab, b.v_slab) and torch.equal(a.k_scales, b.k_scales)
