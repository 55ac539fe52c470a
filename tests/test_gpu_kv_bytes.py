"""Decode steps over u8 slabs on the int8 matrix cores, against the oracle: two, three and four query heads per kv head,
widths 64 and 128, contexts around a wave's tile of 64 positions and a workgroup's round, block sizes that are no powers of
two, splits of a context, sliding windows, scales and queries that are not finite.

The declared bound on the context (``max_context``) picks the kernel, so that short contexts reach it. Bar: 1e-5 where the
outputs are below 4 (values of the slabs), twice the bar of the matrix-core kernel's other tests being met by 1e-6."""
import numpy as np
import pytest

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
    slots, contexts = 4, [70, 257, 100, 300]
    case = make_case(rng, slots=slots, query_heads=8, kv_heads=2, width=128, block_size=16, contexts=contexts, tokens=1,
                     advances=[1] * slots, dtype="u8")
    row_of = lambda slot, position: case["table"][slot, position // 16] * 16 + position % 16  # noqa: E731
    case["v_scales"][row_of(0, 30), 0] = np.nan
    case["k_scales"][row_of(1, 200), 1] = np.inf
    case["q"][2, 3, 0, 1] = np.inf
    case["v_scales"][row_of(3, 5), 0] *= -1  # no writer leaves it, nothing refuses it
    case["k_scales"][row_of(3, 6), 1] = 0.0
    got = run_gpu(et, device, case, 0.1, max_context=BOUND)
    want = run_oracle(case, 0.1)
    assert np.isnan(got[0][0, :4]).all() and np.isnan(got[0][1, 4:]).all() and np.isnan(got[0][2, 3]).all()
    assert np.isfinite(got[0]).mean() > 0.6
    finite = np.isfinite(got[0])
    assert np.isfinite(want[0][finite]).all()
    assert np.abs(got[0][finite] - want[0][finite]).max() <= 1e-5


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
