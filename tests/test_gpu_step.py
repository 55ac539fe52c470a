"""One-vector contractions with the operators around them in one launch (``LinearStep``), against the oracle's operators
one after the other, and the decode step of a single sequence that is made of them.

Sizes: one, two and four slices of columns (4096 each, the last one ragged), one to eight rows per wave and the loop above
that, matrices whose rows end inside a wave's rows or a workgroup's range. Bars: ``close`` of test_gpu_parity (f32 bars)."""
import numpy as np
import pytest
import torch

import oracle
from effect_torch_amd import synth
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
def test_decode_steps_of_one_sequence_follow_the_oracle_chain(et, device, contexts):
    _follow_the_oracle_chain(et, device, False, 1, contexts)
