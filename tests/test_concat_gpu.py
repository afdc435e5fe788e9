"""`cat` of tensors in memory, or of views of such, as one copy kernel whose extents are launch arguments: the bytes of numpy's."""
import numpy as np
import pytest

from morok_amd import tensor as T, uop

pytestmark = pytest.mark.gpu


def _of(shape, seed):
    return np.random.default_rng(seed).integers(0, 1 << 16, shape, dtype=np.uint16)  # (every bit pattern, NaNs among them)


def _t(x):
    return T.Tensor.from_numpy(x, uop.BF16)


# (shapes of the parts, axis): whole workgroups and remainders, one part shorter than a workgroup, outer axes that fold and that do
# not, four parts, an axis of extent 1, a one-row result
@pytest.mark.parametrize("shapes,axis", [([(2, 3, 37, 64), (2, 3, 1, 64)], 2), ([(2, 3, 256, 64), (2, 3, 5, 64)], 2), ([(5, 2048), (5, 8), (5, 1000), (5, 24)], 1),
                                         ([(300, 64), (1, 64)], 0), ([(1, 4, 1, 40, 128), (1, 4, 1, 7, 128)], 3), ([(70001, 8), (3, 8)], 0)])
def test_cat_of_tensors_in_memory(dev, shapes, axis):
    parts = [_of(s, i) for i, s in enumerate(shapes)]
    y = T.Tensor.cat([_t(p) for p in parts], axis).contiguous().realize()
    assert len(y.kernels()) == 1 and y.kernels()[0].startswith("concat_"), y.kernels()
    assert np.array_equal(y.to_numpy().view(np.uint16), np.concatenate(parts, axis))


def test_cat_of_a_cache_and_a_view(dev):
    """New rows read in place out of a packed token-major projection, as a decode step appends them."""
    past, packed = _of((3, 4, 50, 64), 0), _of((3, 3 * 4 * 64), 1)
    new = _t(packed).try_shrink([(0, 3), (256, 512)]).try_reshape([3, 1, 4, 64]).try_permute([0, 2, 1, 3])
    y = T.Tensor.cat([_t(past), new], 2).contiguous().realize()
    assert y.kernels()[0].startswith("concat_")
    want = np.concatenate([past, packed[:, 256:512].reshape(3, 1, 4, 64).transpose(0, 2, 1, 3)], 2)
    assert np.array_equal(y.to_numpy().view(np.uint16), want)
    # two new rows that lie apart
    two = _t(packed).try_reshape([3, 3, 4, 64]).try_permute([0, 2, 1, 3])
    y = T.Tensor.cat([two, _t(past)], 2).realize()
    assert y.kernels()[0].startswith("concat_")
    assert np.array_equal(y.to_numpy().view(np.uint16), np.concatenate([packed.reshape(3, 3, 4, 64).transpose(0, 2, 1, 3), past], 2))


def test_other_cats_stay_generated(dev):
    """Rows that are no whole 16-byte pieces, axes in reverse order, a computed part."""
    # (generated kernels pass through f32, which quiets a signalling NaN: finite values here)
    a, b = _of((40, 2047), 0) & 0x7EFF, _of((40, 3), 1) & 0x7EFF
    y = T.Tensor.cat([_t(a), _t(b)], 1).contiguous().realize()
    assert not y.kernels()[0].startswith("concat_")
    assert np.array_equal(y.to_numpy().view(np.uint16), np.concatenate([a, b], 1))
    f = np.random.default_rng(2).standard_normal((64, 512)).astype(np.float32)
    x = T.Tensor.from_numpy(f)
    y = T.Tensor.cat([x.try_permute([1, 0]), x.try_permute([1, 0])], 1).contiguous().realize()
    assert np.array_equal(y.to_numpy(), np.concatenate([f.T, f.T], 1))
    y = T.Tensor.cat([x, x.try_add(x)], 0).contiguous().realize()
    assert np.array_equal(y.to_numpy(), np.concatenate([f, f + f], 0))
