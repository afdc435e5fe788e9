"""Kernels of an expression realized again with other inputs come from its structure: every form against numpy, first made, kept,
kept with other operands aliased, and made again after the kernel cache was cleared."""
import numpy as np
import pytest

from morok_amd import tensor as T
from morok_amd._ffi import lib

pytestmark = pytest.mark.gpu


def _x(shape, seed):
    return np.random.default_rng(seed).standard_normal(shape).astype(np.float32)


def _t(a):
    return T.Tensor.from_numpy(a)


def _softmax(a):
    e = np.exp(a - a.max(-1, keepdims=True))
    return e / e.sum(-1, keepdims=True)


# elementwise, flat groups of an odd width, a constant, movement, wave reductions, folds in segments (a scratch buffer between two
# kernels), column folds in segments, row-resident kernels with one and two reductions
FORMS = {
    "add": (lambda a, b: a.try_add(b), lambda a, b: a + b, (33, 64)),
    "odd": (lambda a, b: a.try_mul(b).try_add(a), lambda a, b: a * b + a, (32, 51)),
    "const": (lambda a, b: a.try_mul(2.5).maximum(b), lambda a, b: np.maximum(a * np.float32(2.5), b), (40, 64)),
    "transposed": (lambda a, b: a.try_permute([1, 0]).try_sub(b.try_permute([1, 0])).contiguous(), lambda a, b: a.T - b.T, (24, 40)),
    "sum": (lambda a, b: a.try_mul(b).sum([1]), lambda a, b: (a.astype(np.float64) * b).sum(1), (64, 512)),
    "segments": (lambda a, b: a.try_mul(b).sum([1]), lambda a, b: (a.astype(np.float64) * b).sum(1), (2, 1 << 17)),
    "columns": (lambda a, b: a.try_add(b).max([0]), lambda a, b: (a + b).max(0), (2048, 64)),
    "row": (lambda a, b: a.rms_norm(-1, 1e-6).try_mul(b), lambda a, b: a / np.sqrt((a.astype(np.float64) ** 2).mean(-1, keepdims=True) + 1e-6) * b, (200, 512)),
    "row2": (lambda a, b: a.try_add(b).log_softmax(-1), lambda a, b: np.log(_softmax((a + b).astype(np.float64))), (200, 256)),
}


@pytest.mark.parametrize("form", sorted(FORMS))
def test_kept_kernels_read_the_tensors_of_this_call(dev, form):
    build, ref, shape = FORMS[form]
    lib.mrk_hip_kernel_cache_clear()

    def check(a, b, same=False):
        ta = _t(a)
        y = build(ta, ta if same else _t(b)).realize()
        # sums of up to 2^17 products of order one in f32: 2^17 terms in chains of at most 2^12, far below 1e-4 of their scale
        want = ref(a, a if same else b)
        np.testing.assert_allclose(y.to_numpy(), want, rtol=1e-5, atol=1e-5 * max(1.0, np.abs(want).max()))
        return T.last_cached_count(), len(y.kernels())

    cached, n = check(_x(shape, 0), _x(shape, 1))
    assert cached == 0 and n >= 1
    assert check(_x(shape, 2), _x(shape, 3)) == (n, n)          # kept, other inputs
    check(_x(shape, 4), None, same=True)                        # one operand twice: a program of its own
    assert check(_x(shape, 5), _x(shape, 6)) == (n, n)
    other = (shape[0] + 8, shape[1])
    check(_x(other, 7), _x(other, 8))                           # another extent
    lib.mrk_hip_kernel_cache_clear()
    assert check(_x(shape, 9), _x(shape, 10)) == (0, n)         # nothing kept outlives the cache it refers to


def test_constants_and_side_outputs_are_part_of_the_structure(dev):
    a, w = _x((130, 512), 0), _x((512,), 1)
    for c in (0.5, 2.0, 0.5):
        y = _t(a).try_mul(c).realize().to_numpy()
        assert np.array_equal(y, a * np.float32(c))
    for i in range(3):  # the looked-up rows are written by the norm's kernel; the second reader finds them in memory
        table, ids = _x((50, 512), 10 + i), np.random.default_rng(i).integers(0, 50, 130).astype(np.int32)
        h = T.Tensor.from_numpy(table).embedding(T.Tensor.from_numpy(ids)).contiguous()
        y = h.rms_norm(-1, 1e-6).try_mul(_t(w)).contiguous().try_add(h).realize().to_numpy()
        rows = table[ids]
        want = rows / np.sqrt((rows.astype(np.float64) ** 2).mean(-1, keepdims=True) + 1e-6) * w + rows
        np.testing.assert_allclose(y, want, rtol=1e-5, atol=1e-5)
