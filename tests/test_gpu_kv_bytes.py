"""Decode steps over u8 slabs on the int8 matrix cores, against the oracle: two, three and four query heads per kv head,
widths 64 and 128, contexts around a wave's tile of 64 positions and a workgroup's round, block sizes that are no powers of
two, splits of a context, sliding windows, scales and queries that are not finite; against the streaming kernel where the two
give the same; and q, k and v as shares of their projections, against the same call with tensors, bit for bit.

The declared bound on the context (``max_context``) picks the kernel, so that short contexts reach it; every test asserts that
it did. Bar against the oracle: 1e-5, of values of the slabs below 4. The error itself is compared with the streaming kernel's
in ``test_its_error_is_below_the_streaming_kernels``."""
import numpy as np
import pytest
import torch

from effect_torch_amd._native import EtGroupShares
from test_gpu_kv_attention import compare, make_case, run_gpu, run_oracle

pytestmark = pytest.mark.gpu
BOUND = 40000  # units * bound picks the kernel; 1 slot x 2 kv heads x 40000 positions are enough


def check(et, device, case, scale, heads, **options):
    got = run_gpu(et, device, case, scale, max_context=options.pop("max_context", BOUND), **options)
    assert et.kv_attention_variant(got[3], heads, 1).startswith("kv_bytes")
    want = run_oracle(case, scale, **options)
    compare(got, want)
    assert np.abs(got[0] - want[0]).max() <= 1e-5


@pytest.mark.parametrize("width", [64, 128])
@pytest.mark.parametrize("group", [2, 3, 4])
@pytest.mark.parametrize("slots", [9, 129])  # context splits of eight waves; 258 units: one workgroup each
def test_contexts_around_tiles_and_rounds(et, device, width, group, slots):
    rng = np.random.default_rng(width + group + slots)
    contexts = np.resize([0, 1, 15, 63, 64, 65, 127, 511, 700], slots)
    case = make_case(rng, slots=slots, query_heads=2 * group, kv_heads=2, width=width, block_size=16, contexts=contexts,
                     tokens=1, advances=[1] * slots, dtype="u8")
    check(et, device, case, 1.0 / np.sqrt(width), 2 * group)


@pytest.mark.parametrize("block_size", [1, 5, 64])
@pytest.mark.parametrize("window,context_window", [(0, 0), (70, 0), (0, 100)])
def test_blocks_of_any_size_and_windows(et, device, block_size, window, context_window):
    rng = np.random.default_rng(block_size + window)
    case = make_case(rng, slots=3, query_heads=8, kv_heads=2, width=128, block_size=block_size, contexts=[1300, 64, 333],
                     tokens=1, advances=[1, 1, 1], dtype="u8")
    check(et, device, case, -0.09, 8, window=window, context_window=context_window)


@pytest.mark.parametrize("bound", [1700, 140000])  # eight waves, and two workgroups of four to a compute unit
def test_long_contexts_in_splits(et, device, bound):
    rng = np.random.default_rng(bound)
    case = make_case(rng, slots=2, query_heads=64, kv_heads=16, width=64, block_size=16, contexts=[1099, 700], tokens=1,
                     advances=[1, 1], dtype="u8")
    check(et, device, case, 0.4, 64, max_context=bound)


def test_what_is_not_finite_stays_with_the_heads_that_see_it(et, device):
    rng = np.random.default_rng(3)
    slots, contexts = 6, [70, 257, 100, 300, 90, 80]
    case = make_case(rng, slots=slots, query_heads=8, kv_heads=2, width=128, block_size=16, contexts=contexts, tokens=1,
                     advances=[1] * slots, dtype="u8")
    row_of = lambda slot, position: case["table"][slot, position // 16] * 16 + position % 16  # noqa: E731
    case["v_scales"][row_of(0, 30), 0] = np.nan
    case["k_scales"][row_of(1, 200), 1] = np.inf
    case["q"][2, 3, 0, 1] = np.inf
    case["v_scales"][row_of(3, 5), 0] *= -1  # no writer leaves it, nothing refuses it
    case["k_scales"][row_of(3, 6), 1] = 0.0
    case["v_scales"][row_of(4, 7), 1] = -np.inf
    case["v"][5, 0, 0, 9] = np.inf           # the row that arrives: its scale is infinite
    got = run_gpu(et, device, case, 0.1, max_context=BOUND)
    assert et.kv_attention_variant(got[3], 8, 1) == "kv_bytes+kv_merge"
    streaming = run_gpu(et, device, case, 0.1)
    assert et.kv_attention_variant(streaming[3], 8, 1).startswith("kv_attend")
    want = run_oracle(case, 0.1)
    expected = np.zeros((slots, 8), bool)
    expected[0, :4] = expected[1, 4:] = expected[2, 3] = expected[4, 4:] = expected[5, :4] = True
    finite = np.broadcast_to(~expected[:, :, None, None], got[0].shape)
    assert np.isfinite(got[0][finite]).all() and np.abs(got[0][finite] - want[0][finite]).max() <= 1e-5
    # an infinite V scale makes every column NaN here and in the streaming kernel (byte * inf - 128 * inf); the oracle's are
    # infinities but for byte 128
    assert np.isnan(got[0][~finite]).all() and np.isnan(streaming[0][~finite]).all()
    assert not np.isfinite(want[0][~finite]).any() and np.isinf(want[0][4, 4:]).any()
    for mine, theirs in zip(got[1:3] + tuple(got[4]), streaming[1:3] + tuple(streaming[4])):
        assert np.array_equal(mine.view(np.uint8), theirs.view(np.uint8))


def attention_f64(case, scale):
    """One token per slot over u8 slabs in 64 bits."""
    out = np.empty(case["q"].shape)
    group = case["q"].shape[1] // case["k"].shape[1]
    for slot, context in enumerate(case["cursors"].astype(int)):
        positions = np.arange(context)
        rows = case["table"][slot, positions // case["block_size"]].astype(int) * case["block_size"] + positions % case["block_size"]
        for head in range(case["k"].shape[1]):
            cached = [(case[name + "_slab"][rows, head].astype(np.float64) - 128) * case[name + "_scales"][rows, head, None].astype(np.float64)
                      for name in "kv"]
            q = case["q"][slot, head * group:(head + 1) * group, 0].astype(np.float64)
            arriving = []
            for name in "kv":  # as the slab will hold it, in the writer's f32
                row = case[name][slot, head, 0]
                unit = np.abs(row).max() / np.float32(127.0) + np.float32(1e-12)
                byte = np.clip(np.trunc(row / unit + np.copysign(np.float32(0.5), row)), -127, 127)
                arriving.append(byte.astype(np.float64) * np.float64(unit))
            k, v = (np.concatenate([c, a[None]]) for c, a in zip(cached, arriving))
            scores = q @ k.T * scale
            p = np.exp(scores - scores.max(1, keepdims=True))
            out[slot, head * group:(head + 1) * group, 0] = p @ v / p.sum(1, keepdims=True)
    return out


@pytest.mark.parametrize("width,group", [(128, 4), (128, 2), (64, 4), (64, 3)])
def test_its_error_is_below_the_streaming_kernels(et, device, width, group):
    rng = np.random.default_rng(width + group)
    case = make_case(rng, slots=4, query_heads=2 * group, kv_heads=2, width=width, block_size=16, contexts=[900, 1500, 2000, 700],
                     tokens=1, advances=[1] * 4, dtype="u8")
    scale = width ** -0.5
    exact = attention_f64(case, scale)
    errors = {}
    for bound, kernel in ((2001, "kv_attend"), (BOUND, "kv_bytes")):
        got = run_gpu(et, device, case, scale, max_context=bound)
        assert et.kv_attention_variant(got[3], 2 * group, 1).startswith(kernel)
        errors[kernel] = np.linalg.norm(got[0] - exact) / np.linalg.norm(exact)
    print(errors, flush=True)
    assert errors["kv_bytes"] <= errors["kv_attend"] and errors["kv_bytes"] <= 2.5e-7


@pytest.mark.parametrize("group", [2, 3, 4])
@pytest.mark.parametrize("width", [64, 128])
@pytest.mark.parametrize("slots,kv_heads,bound,launch", [
    (130, 2, 300, "kv_bytes"),             # 260 units: one piece of eight waves
    (1, 2, 60000, "kv_bytes+kv_merge"),    # splits of eight waves
    (3, 8, 20000, "kv_bytes+kv_merge"),    # splits of four waves
])
@pytest.mark.parametrize("with_bias", [False, True])
def test_rows_as_shares_of_their_projections(et, device, group, width, slots, kv_heads, bound, launch, with_bias):
    # q, k and v as two shares to be summed, with biases, q and k to be rotated at the cursors: the bytes of the call that is given
    # the rows summed, then rotated by their own launch
    torch.manual_seed(width + group + slots)
    rng = np.random.default_rng(width + group + slots)
    heads = group * kv_heads
    case = make_case(rng, slots=slots, query_heads=heads, kv_heads=kv_heads, width=width, block_size=16,
                     contexts=rng.integers(0, 200, slots), tokens=1, advances=[1] * slots, dtype="u8")
    sizes = [heads * width, kv_heads * width, kv_heads * width]
    first = np.cumsum([0] + sizes)
    shares = torch.randn(2, slots, int(first[-1]), device=device)
    biases = [torch.randn(size, device=device) if with_bias else None for size in sizes]
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)  # noqa: E731
    results = []
    for projected in (False, True):
        tensors = {name: dev(case[name]) for name in ("k_slab", "v_slab", "k_scales", "v_scales")}
        cursors = dev(case["cursors"].view(np.int32))
        layer = et.KvLayer(tensors["k_slab"], tensors["v_slab"], 16, dev(case["table"].view(np.int32)), cursors,
                           dev(case["advances"].view(np.int32)), bound, k_scales=tensors["k_scales"], v_scales=tensors["v_scales"])
        assert et.kv_attention_variant(layer, heads, 1) == launch
        out = torch.full((slots, heads, 1, width), float("nan"), device=device)
        if projected:
            layout = EtGroupShares(shares.data_ptr(), 2, slots, int(first[-1]), (*(int(f) for f in first[:3]), 0))
            et.kv_attention_projected_into(layer, layout, (0, 1, 2), biases, cursors, 500000.0, 1.0, et.RotaryLayout.HALF_SPLIT,
                                           0.1, None, out)
        else:
            rows = [(shares[0] + shares[1])[:, first[i]:first[i + 1]].contiguous() for i in range(3)]
            rows = [row + bias if bias is not None else row for row, bias in zip(rows, biases)]
            q, k, v = (row.view(slots, -1, 1, width) for row in rows)
            et.rotary_pair_into(q, k, cursors, 500000.0, 1.0, et.RotaryLayout.HALF_SPLIT, q, k)
            et.kv_attention_into(layer, q, k, v, 0.1, None, out)
        results.append([out, *tensors.values()])
    assert torch.isfinite(results[0][0]).all()
    for one, other in zip(*results):
        assert torch.equal(one.view(torch.uint8), other.view(torch.uint8))


@pytest.mark.parametrize("exponent", [-60, -95, -117])
@pytest.mark.parametrize("width", [64, 128])
def test_small_scales_and_queries_keep_their_bits(et, device, width, exponent):
    # A slab may hold rows of any scale, and the limbs of q and of the weights are fixed point. Bar: f32 sums of 300 terms,
    # 300 * 2^-24 / sqrt(300) = 1e-6 of the result; the streaming kernel shows 2.6e-7.
    relative = lambda got, want: (np.linalg.norm((got.astype(np.float64) - want) / np.abs(want).max()) /  # noqa: E731
                                  np.linalg.norm(want / np.abs(want).max()))
    factor = np.float32(2.0 ** exponent)
    make = lambda: make_case(np.random.default_rng(width), slots=2, query_heads=8, kv_heads=2, width=width, block_size=16,  # noqa: E731
                             contexts=[300, 200], tokens=1, advances=[1, 1], dtype="u8")
    small_values = make()
    small_values["v_scales"] *= factor
    small_values["v"] *= factor * np.float32(0)
    small_queries = make()  # the scores are those of ordinary q and K
    small_queries["q"] *= factor
    small_queries["k_scales"] /= factor
    small_queries["k"] *= 0
    for case in (small_values, small_queries):
        got, want = run_gpu(et, device, case, 0.1, max_context=BOUND), run_oracle(case, 0.1)
        assert et.kv_attention_variant(got[3], 8, 1).startswith("kv_bytes")
        assert relative(got[0], want[0].astype(np.float64)) <= 1e-6
