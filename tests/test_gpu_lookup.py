"""Bit-exact lookup at the sizes where its launch changes shape: rows of fewer spans than a workgroup has threads (several
rows to a workgroup, idle threads), rows that end inside a workgroup's part, and indexes just below and above what one
round, two rounds and no longer one launch check, with a bad one in every round."""
import numpy as np
import pytest
import torch

import oracle
from effect_torch_amd import synth

pytestmark = pytest.mark.gpu

# 1024 of Q4_0, 512 of Q8_0, 1024 and 2048 of the others are the widest rows that share a workgroup
WIDTHS = {"Q4_0": [32, 96, 1024, 1056, 2080, 2112], "Q8_0": [32, 160, 512, 544, 4128],
          **{c: [256, 768, 1024, 2048, 2304, 4352] for c in ("Q2_K", "Q3_K", "Q4_K", "Q5_K", "Q6_K")}}


@pytest.mark.parametrize("codec,columns", [(codec, columns) for codec, widths in WIDTHS.items() for columns in widths])
def test_rows_of_every_width_bit_exact(et, device, codec, columns):
    rng = np.random.default_rng(columns)
    rows = 61
    weight = synth.random_weight(getattr(synth, codec), rows, columns, rng)
    ids = rng.integers(0, rows, 150)
    want = oracle.decode_rows(getattr(synth, codec), weight, columns)[ids]
    idx, table = torch.from_numpy(ids).to(device), torch.from_numpy(weight).to(device)
    plan = et.embedding_requirements(idx, table, et.GgmlQuant[codec], (rows, columns))
    out = torch.full(plan.output_shape, np.nan, device=device)
    et.embedding_into(idx, table, et.GgmlQuant[codec], out, plan)
    assert np.array_equal(out.cpu().numpy().view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("count,bad", [(4096, 4095), (4097, 4096), (8192, 4000), (8192, 8191), (8193, 8192)])
def test_the_first_bad_index_is_reported(et, device, count, bad):
    rows, columns = 9, 32
    weight = synth.random_weight(synth.Q8_0, rows, columns, np.random.default_rng(5))
    ids = np.arange(count) % rows
    ids[bad] = 77
    ids[-1] = 78 if bad != count - 1 else 77
    idx, table = torch.from_numpy(ids).to(device), torch.from_numpy(weight).to(device)
    plan = et.embedding_requirements(idx, table, et.GgmlQuant.Q8_0, (rows, columns))
    out = torch.empty(plan.output_shape, device=device)
    with pytest.raises(et.QuantizedError, match="index 77 is outside 0..9"):
        et.embedding_into(idx, table, et.GgmlQuant.Q8_0, out, plan)
    good = np.arange(count) != bad
    good[-1] = False
    want = oracle.decode_rows(synth.Q8_0, weight, columns)
    assert np.array_equal(out.cpu().numpy()[good], want[ids[good]])
