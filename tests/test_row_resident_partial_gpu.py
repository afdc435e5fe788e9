"""Row-resident kernels over rows that do not divide into whole workgroups of vectors: against the separate kernels of the same graph and
against numpy in 64 bits, with infinities in the rows."""
import os

import numpy as np
import pytest

from morok_amd import synth
from morok_amd import tensor as T, uop

pytestmark = pytest.mark.gpu


def _separate(build):
    os.environ["MOROK_NO_ROW_FUSION"] = "1"
    try:
        y = build().realize()
        assert len(y.kernels()) > 1
        return y.to_numpy()
    finally:
        del os.environ["MOROK_NO_ROW_FUSION"]


# one vector more and one less than a workgroup's, vectors of 8, 4, 2 and 1 element, sixteen loads per work-item, a single row, rows
# shorter than a wave, many rows
SHAPES = [(130, 520), (130, 504), (7, 1028), (64, 1026), (31, 8191), (200, 4097), (1, 5446), (64, 10), (3, 3), (3000, 264)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("bf16", [False, True])
def test_rms_norm_with_gain(dev, shape, bf16):
    x, g = synth.normal(shape, 3, 0), 1.0 + synth.normal((shape[1],), 3, 1, sigma=0.1)
    if bf16:
        x, g = synth.from_bf16(synth.to_bf16(x)), synth.from_bf16(synth.to_bf16(g))
    conv, tag = (synth.to_bf16, uop.BF16) if bf16 else (np.ascontiguousarray, uop.F32)
    build = lambda: T.Tensor.from_numpy(conv(x), tag).rms_norm(-1, 1e-6).try_mul(T.Tensor.from_numpy(conv(g), tag)).cast(tag)  # noqa: E731
    y = build().realize()
    assert len(y.kernels()) == 1 and y.kernels()[0].startswith("rE_"), y.kernels()
    want = x / np.sqrt((x.astype(np.float64) ** 2).mean(-1, keepdims=True) + 1e-6) * g
    got, other = y.to_numpy(), _separate(build)
    if bf16:
        got, other = synth.from_bf16(got), synth.from_bf16(other)
    # f32: the statistic's sum of C squares, two multiplications and a reciprocal square root; bf16: one rounding on top
    tol = 2.0 ** -8 if bf16 else 4e-6
    assert np.abs(got - want).max() <= tol * np.abs(want).max()
    assert np.abs(got - other).max() <= tol * np.abs(want).max()


@pytest.mark.parametrize("shape", SHAPES)
def test_log_softmax(dev, shape):
    x = synth.normal(shape, 4, 0, sigma=3.0)
    if shape[0] > 1 and shape[1] > 3:
        x[1, 0], x[1, -1] = -np.inf, -np.inf  # some of a row's values, among them its last
        x[0, -1] = 60.0
    build = lambda: T.Tensor.from_numpy(x).log_softmax(-1)  # noqa: E731
    y = build().realize()
    assert len(y.kernels()) == 1, y.kernels()
    m = x.astype(np.float64).max(-1, keepdims=True)
    want = x - (m + np.log(np.exp(x - m).sum(-1, keepdims=True)))
    np.testing.assert_allclose(y.to_numpy(), want, rtol=1e-5, atol=1e-5)  # (elementwise f32; the sum of up to 8191 terms in a row)
    np.testing.assert_allclose(y.to_numpy(), _separate(build), rtol=1e-5, atol=1e-5)


def test_side_output(dev):
    rows, cols = 150, 1000
    table, ids, w = synth.normal_bf16((300, cols), 5, 0), synth.randint((rows,), 5, 1, 300), synth.normal_bf16((cols,), 5, 2)
    h = T.Tensor.from_numpy(table, uop.BF16).embedding(T.Tensor.from_numpy(ids)).contiguous().keep()
    y = h.rms_norm(-1, 1e-6).try_mul(T.Tensor.from_numpy(w, uop.BF16)).cast(uop.BF16).realize()
    assert len(y.kernels()) == 1 and y.kernels()[0].endswith("_s1"), y.kernels()
    assert np.array_equal(h.to_numpy().view(np.uint16), table[ids])
    x = synth.from_bf16(table[ids])
    want = x / np.sqrt((x.astype(np.float64) ** 2).mean(-1, keepdims=True) + 1e-6) * synth.from_bf16(w)
    assert np.abs(synth.from_bf16(y.to_numpy()) - want).max() <= 2.0 ** -8 * np.abs(want).max()


# Rows that a product or another reduction leaves: that is computed first, the row's reductions and its elementwise part are one kernel
@pytest.mark.parametrize("shape", [(64, 256, 10), (1, 33, 2), (3, 700, 257), (512, 32, 1000), (17, 64, 65)])
@pytest.mark.parametrize("activation", [False, True])
def test_log_softmax_of_a_product(dev, shape, activation):
    b, k, c = shape
    x, w, bias = synth.normal((b, k), 6, 0), synth.normal((c, k), 6, 1, sigma=k ** -0.5), synth.normal((c,), 6, 2)

    def build():
        t = T.Tensor.from_numpy(x)
        if activation:
            t = t.maximum(0.0)
        return t.linear(T.Tensor.from_numpy(w), T.Tensor.from_numpy(bias)).log_softmax(-1)

    y = build().realize()
    assert y.kernels()[-1].startswith("rE_") and sum(n.startswith(("rE_", "r_")) for n in y.kernels()) <= 2, y.kernels()
    z = (np.maximum(x, 0) if activation else x).astype(np.float64) @ w.T.astype(np.float64) + bias
    m = z.max(-1, keepdims=True)
    # (products of K terms in f32, up to |z| of about 10)
    np.testing.assert_allclose(y.to_numpy(), z - (m + np.log(np.exp(z - m).sum(-1, keepdims=True))), rtol=1e-5, atol=2e-5)
    np.testing.assert_allclose(y.to_numpy(), _separate(build), rtol=1e-5, atol=1e-5)


def test_statistics_of_other_rows_and_columns_come_first(dev):
    x, o = synth.normal((130, 520), 7, 0), synth.normal((520, 130, 3), 7, 1)
    t, u = T.Tensor.from_numpy(x), T.Tensor.from_numpy(o)
    columns = u.sum([1, 2]).try_reshape([1, 520]).try_expand([130, 520])  # a reduction of another tensor
    build = lambda: t.try_add(columns).softmax(-1)  # noqa: E731
    z = x.astype(np.float64) + o.astype(np.float64).sum((1, 2))
    want = np.exp(z - z.max(-1, keepdims=True))
    want /= want.sum(-1, keepdims=True)
    np.testing.assert_allclose(build().to_numpy(), want, rtol=1e-4, atol=1e-7)  # (sums of 390 terms in f32 under an exponential)
    y = t.try_sub(t.sum(0, keepdim=True).try_expand([130, 520])).log_softmax(-1).to_numpy()  # one of the row's own tensor along columns
    z = x.astype(np.float64) - x.astype(np.float64).sum(0)
    m = z.max(-1, keepdims=True)
    np.testing.assert_allclose(y, z - (m + np.log(np.exp(z - m).sum(-1, keepdims=True))), rtol=1e-5, atol=1e-4)
