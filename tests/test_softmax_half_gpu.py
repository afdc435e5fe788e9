"""Softmax over bf16 and f16 rows that are no whole waves of vectors (one kernel, the row in registers), against
float64 on the same inputs."""
import numpy as np
import pytest

import morok_amd.tensor as T
from morok_amd import synth, uop

pytestmark = pytest.mark.gpu

COLS = [1, 7, 8, 9, 79, 511, 513, 712, 1023, 1025, 2047, 2052, 4090, 4099, 8191, 8200, 16380, 16390, 32767, 32776, 65528, 65535, 65536]


def _half(x, f16):
    return x.astype(np.float16) if f16 else synth.to_bf16(x)


def _wide(bits, f16):
    return bits.astype(np.float64) if f16 else synth.from_bf16(bits).astype(np.float64)


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("cols", COLS)
@pytest.mark.parametrize("rows", [1, 5])
def test_softmax_half(rows, cols, f16):
    x = _half(synth.normal((rows, cols), cols, rows, sigma=3.0), f16)
    t = T.Tensor.from_numpy(x, uop.F16 if f16 else uop.BF16).softmax(-1)
    got = _wide(t.to_numpy(), f16)
    assert len(t.kernels()) == 1, t.kernels()
    w = _wide(x, f16)
    e = np.exp(w - w.max(1, keepdims=True))
    ref = e / e.sum(1, keepdims=True)
    # one rounding to the type: half the spacing, which is 2^-10 (f16) or 2^-7 (bf16) of the power of two below the value, so at
    # most 2^-11 or 2^-8 of the value; the f32 exponential, sum and product add a hundredth of that at most; below f16's
    # normal range the spacing is 2^-24
    u = 2.0 ** -11 if f16 else 2.0 ** -8
    assert np.all(np.abs(got - ref) <= ref * u * 1.01 + (2.0 ** -25 if f16 else 1e-38))


def test_softmax_half_infinities_and_nan():
    x = np.zeros((4, 300), np.float32)
    x[0, 5:] = -np.inf
    x[1, :] = -np.inf
    x[2, 7] = np.nan
    got = synth.from_bf16(T.Tensor.from_numpy(synth.to_bf16(x), uop.BF16).softmax(-1).to_numpy())
    assert np.all(got[0, 5:] == 0) and np.allclose(got[0, :5], 0.2, atol=1e-3)
    assert np.all(np.isnan(got[1])) and np.all(np.isnan(got[2])) and np.allclose(got[3], 1 / 300, rtol=4e-3)


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("cols", [1, 2, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 121, 127, 128, 129])
def test_softmax_half_short_rows(dev, cols, f16):
    """Several rows to a wave: rows that fill a workgroup and rows beyond, NaNs right behind the input and a pattern behind the
    result, which has to stay."""
    import morok_amd

    rows = 1031
    x = _half(synth.normal((rows, cols), cols, 7, sigma=3.0), f16)
    guard = np.full(64, 0x7FFF, np.uint16)
    bx = morok_amd.Buffer.from_numpy(np.concatenate([x.view(np.uint16).reshape(-1), guard]), dev.device_id)
    by = morok_amd.Buffer.from_numpy(np.full(rows * cols + 64, 0x1234, np.uint16), dev.device_id)
    morok_amd.Program.builtin("softmax_f16" if f16 else "softmax_bf16", [rows, cols], dev.device_id).execute([by, bx])
    out = by.copyout(np.uint16)
    assert np.all(out[rows * cols:] == 0x1234)
    got = out[:rows * cols].reshape(rows, cols)
    got = _wide(got.view(np.float16) if f16 else got, f16)
    w = _wide(x, f16)
    e = np.exp(w - w.max(1, keepdims=True))
    ref = e / e.sum(1, keepdims=True)
    u = 2.0 ** -11 if f16 else 2.0 ** -8  # (the bound of test_softmax_half)
    assert np.all(np.abs(got - ref) <= ref * u * 1.01 + (2.0 ** -25 if f16 else 1e-38))
