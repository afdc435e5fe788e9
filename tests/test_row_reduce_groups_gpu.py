"""Long folds over the contiguous axis, which the generated reduce kernel reads in groups of consecutive elements: rows that divide
into groups of 8, 4 and 2 and odd ones, with partial last steps, against float64."""
import numpy as np
import pytest

import morok_amd.tensor as T
from morok_amd import synth, uop

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(1200, 1001), (1100, 1002), (1030, 1020), (4200, 520), (4200, 264), (600, 3608), (520, 12296), (2049, 16384)])
@pytest.mark.parametrize("op", ["sum", "max"])
def test_row_reductions_in_groups(rows, cols, op):
    x = synth.normal((rows, cols), 5, cols)
    t = T.Tensor.from_numpy(x).try_mul(2.0)
    got = (t.sum(1) if op == "sum" else t.max(1)).to_numpy()
    w = 2.0 * x.astype(np.float64)
    if op == "max":
        assert np.array_equal(got, w.max(1).astype(np.float32))
    else:  # the forward error of a sum of `cols` terms in any order
        assert np.all(np.abs(got - w.sum(1)) <= cols * 2.0 ** -24 / (1 - cols * 2.0 ** -24) * np.abs(w).sum(1))
    h = T.Tensor.from_numpy(synth.to_bf16(x), uop.BF16).cast(uop.F32)
    got = (h.sum(1) if op == "sum" else h.max(1)).to_numpy()
    w = synth.from_bf16(synth.to_bf16(x)).astype(np.float64)
    if op == "max":
        assert np.array_equal(got, w.max(1).astype(np.float32))
    else:
        assert np.all(np.abs(got - w.sum(1)) <= cols * 2.0 ** -24 / (1 - cols * 2.0 ** -24) * np.abs(w).sum(1))
