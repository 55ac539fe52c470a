"""GPU parity of the one-pass small-batch GEMV (2..8 activation vectors; Q4_K, Q5_K, Q4_0, Q8_0; the regime
crates/runtime-metal/src/quantized.rs:1204-1220 keeps in its GEMV family): the HIP path through the C
ABI against the CPU oracle (linear_into, crates/runtime-cpu/src/quantized.rs:419-499) on the same
seeded inputs. Bar: |a-b| <= 1e-3 * max(|b|, 1), once against the oracle and once, with no allowance,
against the f64-exact value of the same contraction; and the same bits on a second run.
"""
import numpy as np
import pytest
import torch

import oracle
from effect_torch_amd import synth
from test_gpu_parity import close, run_linear, to_dev

pytestmark = pytest.mark.gpu

CODECS = [oracle.Q4_K, oracle.Q4_0, oracle.Q5_K, oracle.Q8_0]


def planned_kernel(et, codec, rows, columns, vectors, bias=False):
    return et.RawLinear(et.GgmlQuant(codec), rows, columns, vectors, bias).requirements.kernel


def check(et, device, codec, rows, columns, vectors, rng, bias=None, x_scale=1.0, kernel="gemv_mma"):
    weight = synth.random_weight(codec, rows, columns, rng)
    x = synth.random_activations(vectors, columns, rng, x_scale)
    assert planned_kernel(et, codec, rows, columns, vectors, bias is not None) == kernel
    print(f"gemv_mma codec={codec} rows={rows} columns={columns} vectors={vectors}", flush=True)
    abandoned = et.handover_timeouts()
    got = run_linear(et, device, codec, rows, columns, x, weight, bias)
    again = run_linear(et, device, codec, rows, columns, x, weight, bias)
    assert np.array_equal(got, again)  # neither the arrival order of the copies nor that of the waves reaches the sums
    close(got, oracle.linear_into(codec, rows, columns, x, weight, bias))
    exact = x.astype(np.float64) @ oracle.decode_rows(codec, weight, columns).astype(np.float64).T
    if bias is not None:
        exact = exact + bias.astype(np.float64)
    close(got, exact, oracle_noise=0)
    assert et.handover_timeouts() == abandoned  # no wave gave up a wait
    return got


@pytest.mark.parametrize("codec", CODECS)
@pytest.mark.parametrize("vectors", [2, 3, 4, 5, 6, 7, 8])
def test_every_vector_count(et, device, codec, vectors):
    # 4099 rows: ranges of 17 rows (a whole group of sixteen and a group of one), a ragged last range
    rng = np.random.default_rng(100 * codec + vectors)
    check(et, device, codec, 4099, 4096, vectors, rng, rng.standard_normal(4099).astype(np.float32))


@pytest.mark.parametrize("codec", CODECS)
@pytest.mark.parametrize("vectors,rows,columns", [
    (2, 2048, 4096),     # half a group per range
    (4, 2100, 4096),     # ranges of 9 rows, the last of 6
    (3, 5003, 256),      # one unit per row: seven of the eight consumer waves hold no columns
    (8, 3000, 2048),     # four consumer waves hold columns
    (5, 30000, 512),     # 118 rows per range, images of 36 KiB
    (8, 40000, 4096),    # more rows than 256 images hold: three rounds of 256 ranges of 53 rows
    (6, 9000, 1024),
    (4, 12000, 3072),    # the last consumer waves hold one unit / none
    (7, 2300, 3840),     # fifteen units: the last wave holds one
])
def test_shapes(et, device, codec, vectors, rows, columns):
    rng = np.random.default_rng(7 * codec + vectors + rows + columns)
    bias = rng.standard_normal(rows).astype(np.float32) if rows % 2 else None
    check(et, device, codec, rows, columns, vectors, rng, bias)


@pytest.mark.parametrize("codec", CODECS)
@pytest.mark.parametrize("vectors,rows,columns", [
    (3, 2048, 4352),     # seventeen units: a last slice of one
    (2, 2048, 8448),     # two vectors: wider than 8192 columns
    (4, 2100, 8192),     # whole slices only; ranges of nine rows, the last of three
    (5, 4096, 6400),     # sixteen rows per range, a last slice of one unit
    (6, 4100, 5120),     # ranges of seventeen rows: a group of one; a half slice at the end
    (3, 4096, 14336),    # the widest configuration: seven slices (Q8_0: two rounds of ranges of eight rows)
])
def test_rows_wider_than_4096_columns(et, device, codec, vectors, rows, columns):
    rng = np.random.default_rng(17 * codec + vectors + rows + columns)
    bias = rng.standard_normal(rows).astype(np.float32) if rows % 8 else None
    check(et, device, codec, rows, columns, vectors, rng, bias, kernel="gemv_mma_prepare+gemv_mma_wide")


# Bytes of a 256-column unit that make its first 64 columns' weights zero: {offset: bytes}.
ZERO_FIRST_64 = {
    oracle.Q4_K: {2: [0] * 2, 16: [0] * 32},            # no minimum; nibbles of sub-blocks 0 and 1
    oracle.Q5_K: {2: [0] * 2, 16: None, 48: [0] * 32},  # None: their fifth bits
    oracle.Q4_0: {0: [0] * 2, 18: [0] * 2},             # the block scales: a quant of 8 is only zero after a subtraction
    oracle.Q8_0: {2: [0] * 32, 36: [0] * 32},
}


@pytest.mark.parametrize("codec", CODECS)
@pytest.mark.parametrize("vectors", [3, 6])
def test_wide_rows_beside_a_large_activation(et, device, codec, vectors):
    # One activation of 2^20 among each 256, its 64 columns' weights zero: the other columns keep 24 bits of their own
    # size. Fixed point with 127 * 2^16 units to the largest of 64 columns is off by at most 1.5 units (half a unit
    # of rounding, one of the scaled value's two roundings); the rest is f32 sums of at most 64 terms per chain.
    rows, columns = 2080, 8448
    rng = np.random.default_rng(400 + 10 * codec + vectors)
    weight = synth.random_weight(codec, rows, columns, rng)
    units = weight.reshape(rows, columns // 256, -1)
    for offset, values in ZERO_FIRST_64[codec].items():
        if values is None:
            units[:, :, offset:offset + 32] &= 0xFC
        else:
            units[:, :, offset:offset + len(values)] = values
    weight = units.reshape(rows, -1)
    x = synth.random_activations(vectors, columns, rng)
    x[:, 5::256] = 2.0 ** 20
    assert planned_kernel(et, codec, rows, columns, vectors) == "gemv_mma_prepare+gemv_mma_wide"
    got = run_linear(et, device, codec, rows, columns, x, weight)
    w = oracle.decode_rows(codec, weight, columns).astype(np.float64)
    assert not w.reshape(rows, -1, 256)[:, :, :64].any()
    unit = np.abs(x.astype(np.float64)).reshape(vectors, -1, 64).max(-1) / (127 * 65536)
    bound = 1.5 * unit @ np.abs(w).reshape(rows, -1, 64).sum(-1).T + 64 * 2.0 ** -24 * np.abs(x.astype(np.float64)) @ np.abs(w).T
    assert (np.abs(got - x.astype(np.float64) @ w.T) <= bound).all()


@pytest.mark.parametrize("codec", [oracle.Q4_K, oracle.Q5_K])
@pytest.mark.parametrize("rows,columns", [
    (2048, 256),    # one unit: seven consumer waves hold no columns
    (5000, 3840),   # a last group of four rows; the last wave holds one unit
    (2100, 4096),
    (2064, 4352),   # wider rows: a last slice of one unit
    (4096, 14336),  # seven whole slices
])
def test_a_fifth_vector_in_the_rows_of_four(et, device, codec, rows, columns):
    # Its limbs lie in the rows that the four others leave empty: it gets its own value whatever they hold. Fixed point is off
    # by at most 1.5 units (127 * 2^16 to the largest of 64 columns, 4161000 to that of 256 in rows of up to 4096), the rest
    # is f32 sums of at most 64 terms per chain, the minima's apart from the quants'.
    rng = np.random.default_rng(500 + codec + rows + columns)
    weight = synth.random_weight(codec, rows, columns, rng)
    x = synth.random_activations(5, columns, rng)
    x[4] += 0.5  # the minima weigh as much as the quants
    x[1] = 0.0
    x[2, ::7] = np.nan
    got = run_linear(et, device, codec, rows, columns, x, weight)
    w = oracle.decode_rows(codec, weight, columns).astype(np.float64)
    size, most = (256, 4161000) if columns <= 4096 else (64, 127 * 65536)
    unit = np.abs(x[4].astype(np.float64)).reshape(-1, size).max(-1) / most
    parts = np.abs(w) + 2 * np.abs(w).max(1, keepdims=True)
    bound = 1.5 * np.abs(w).reshape(rows, -1, size).sum(-1) @ unit + 64 * 2.0 ** -24 * parts @ np.abs(x[4].astype(np.float64))
    assert (np.abs(got[4] - w @ x[4].astype(np.float64)) <= bound).all()
    assert not got[1].any() and np.isnan(got[2]).all() and np.isfinite(got[[0, 3, 4]]).all()
    close(got[[0, 3]], x[[0, 3]].astype(np.float64) @ w.T)


def test_wide_rows_without_a_workspace(et, device):
    # aligned activations need no workspace in the vector kernels: the call then runs the launches that quantise themselves
    rows, columns, vectors = 2048, 8192, 5
    rng = np.random.default_rng(3)
    weight = synth.random_weight(oracle.Q4_K, rows, columns, rng)
    x = synth.random_activations(vectors, columns, rng)
    plan = et.RawLinear(et.GgmlQuant.Q4_K, rows, columns, vectors)
    y = torch.empty(vectors, rows, device=device)
    plan.enqueue(to_dev(x, device), to_dev(weight, device), None, y)
    close(y.cpu().numpy(), oracle.linear_into(oracle.Q4_K, rows, columns, x, weight))


@pytest.mark.parametrize("name", ["q4_0_gemv_11008x4096", "q4_k_gemv_14336x4096", "q8_0_gemv_4096x4096"])
@pytest.mark.parametrize("vectors", [2, 3, 4, 5, 6, 7, 8])
def test_full_size(et, device, name, vectors):
    cfg = synth.CONFIGS[name]
    rng = np.random.default_rng(cfg["seed"] + 50 + vectors)
    check(et, device, cfg["codec"], cfg["rows"], cfg["columns"], vectors, rng, None, cfg["x_scale"])


@pytest.mark.parametrize("codec", CODECS)
def test_special_activations(et, device, codec):
    # unit vectors select one decoded weight (every other product is an exact zero; what is left is the
    # rounding of d * (scale * quant) against the decoder's (d * scale) * quant, and for Q4_0 of d * quant - 8 * d: a
    # few 1e-8 of the largest weight); a vector of
    # zeros gives zeros; a vector whose 256-column units differ by 2^20 in size keeps every unit's precision
    rows, columns, vectors = 2304, 4096, 4
    rng = np.random.default_rng(31 + codec)
    weight = synth.random_weight(codec, rows, columns, rng)
    decoded = oracle.decode_rows(codec, weight, columns)
    x = np.zeros((vectors, columns), np.float32)
    picks = [5, 1000, 4095]
    for v, k in enumerate(picks):
        x[v, k] = 1.0
    got = run_linear(et, device, codec, rows, columns, x, weight)
    for v, k in enumerate(picks):
        np.testing.assert_allclose(got[v], decoded[:, k], rtol=5e-7, atol=1e-7 * np.abs(decoded[:, k]).max())
    assert not got[3].any()
    x = synth.random_activations(vectors, columns, rng)
    x[:, :256] *= 2.0 ** 20
    x[:, 256:512] *= 2.0 ** -20
    got = run_linear(et, device, codec, rows, columns, x, weight)
    exact = x.astype(np.float64) @ decoded.astype(np.float64).T
    close(got, exact)  # outputs that cancel to a millionth of the row's size: the allowance of an f32 sum
    small = x.copy()
    small[:, :256] = 0.0  # without the large unit the small one must come out to its own precision
    tail = run_linear(et, device, codec, rows, columns, small, weight)
    exact_tail = x[:, 256:].astype(np.float64) @ decoded[:, 256:].astype(np.float64).T
    close(tail, exact_tail, oracle_noise=0)


def test_strided_activation_rows(et, device):
    # rows of a wider tensor (unit trailing stride, 16-byte aligned): read in place
    rows, columns, vectors = 4096, 4096, 5
    rng = np.random.default_rng(77)
    weight = synth.random_weight(oracle.Q4_K, rows, columns, rng)
    wide = torch.from_numpy(rng.standard_normal((vectors, 2 * columns)).astype(np.float32)).to(device)
    view = wide[:, columns:]
    got = run_linear(et, device, oracle.Q4_K, rows, columns, view, weight)
    close(got, oracle.linear_into(oracle.Q4_K, rows, columns, view.cpu().numpy().copy(), weight))


def test_a_wait_that_is_given_up_ends_the_launch(et, device):
    # Every wait of a consumer wave on another wave is bounded. With the bound at zero polls a wave that
    # finds its rows not landed yet gives up at once: the launch must still end (every wave leaves the
    # kernel), the device word counts the waves, and the next launch with the library's own bound is right.
    codec, rows, columns, vectors = oracle.Q4_K, 14336, 4096, 4
    rng = np.random.default_rng(5)
    weight = synth.random_weight(codec, rows, columns, rng)
    x = synth.random_activations(vectors, columns, rng)
    before = et.handover_timeouts()
    et.set_handover_spin_limit(0)
    try:
        run_linear(et, device, codec, rows, columns, x, weight)  # returns: the launch has ended
        single = run_linear(et, device, codec, rows, columns, x[:1], weight)  # gemv_limb_dma, same bound
    finally:
        et.set_handover_spin_limit()
    assert single.shape == (1, rows)
    assert et.handover_timeouts() > before
    counted = et.handover_timeouts()
    got = run_linear(et, device, codec, rows, columns, x, weight)
    close(got, oracle.linear_into(codec, rows, columns, x, weight))
    one = run_linear(et, device, codec, rows, columns, x[:1], weight)
    close(one, oracle.linear_into(codec, rows, columns, x[:1], weight))
    assert et.handover_timeouts() == counted
