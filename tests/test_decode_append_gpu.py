"""The decode attention that grows its caches: the bytes of the copies, and the bits of the attention over caches that are in memory."""
import numpy as np
import pytest

from morok_amd import synth, tensor as T, uop

pytestmark = pytest.mark.gpu


def _t(x):
    return T.Tensor.from_numpy(np.ascontiguousarray(x), uop.BF16)


# (batch, heads, keys before the new one, head dim): the new key alone in a chunk of 32, last in one, and in between; one key range
# and many; fewer ranges than waves
@pytest.mark.parametrize("b,h,past,d", [(2, 3, 256, 64), (3, 4, 287, 128), (1, 2, 300, 256), (1, 1, 2047, 128), (2, 2, 4096, 64), (64, 16, 511, 128),
                                        (8, 32, 767, 64), (1, 8, 9000, 256)])
def test_append(dev, b, h, past, d):
    pk, pv = (synth.normal_bf16((b, h, past, d), 21, i) for i in range(2))
    packed = synth.normal_bf16((b, 3 * h * d), 22, 0)
    pk[0, 0, 7, :4] = pv[0, 0, past - 1, :4] = [0x7F81, 0x8000, 0x0001, 0xFFFF]  # (signalling and quiet NaNs, -0, a denormal)

    def part(i):  # a packed token-major projection, read in place
        t = _t(packed).try_shrink([(0, b), (i * h * d, (i + 1) * h * d)])
        return t.try_reshape([b, 1, h, d]).try_permute([0, 2, 1, 3])

    q, k1, v1 = (part(i) for i in range(3))
    k, v = (T.Tensor.cat([_t(p), n], 2).contiguous() for p, n in ((pk, k1), (pv, v1)))
    o = q.scaled_dot_product_attention(k, v).realize()
    names = o.kernels()
    assert len(names) == 1 and names[0].startswith("flash_fwd_bf16_append_"), names
    new = packed.reshape(b, 3, h, 1, d)
    want = [np.concatenate([p, new[:, i]], 2) for i, p in ((1, pk), (2, pv))]
    for got, w in zip((k, v), want):
        assert np.array_equal(got.to_numpy().view(np.uint16), w)
    ref = _t(new[:, 0]).scaled_dot_product_attention(_t(want[0]), _t(want[1])).realize()
    assert not any("append" in n or "concat" in n for n in ref.kernels())
    assert np.array_equal(o.to_numpy(), ref.to_numpy())


def test_what_does_not_append(dev):
    """Two new keys, a causal call and caches of another length keep the copies, with the same result."""
    b, h, past, d = 1, 2, 300, 64
    pk, pv, n = synth.normal_bf16((b, h, past, d), 23, 0), synth.normal_bf16((b, h, past, d), 23, 1), synth.normal_bf16((b, h, 2, d), 23, 2)
    for new, keys, causal in ((n, past, False), (n[:, :, :1], past, True), (n[:, :, :1], 100, False)):
        k, v = (T.Tensor.cat([_t(p[:, :, :keys]), _t(new)], 2).contiguous() for p in (pk, pv))
        o = _t(new[:, :, :1]).scaled_dot_product_attention(k, v, is_causal=causal).realize()
        assert not any("append" in s for s in o.kernels())
        ref = _t(new[:, :, :1]).scaled_dot_product_attention(*(_t(np.concatenate([p[:, :, :keys], new], 2)) for p in (pk, pv)), is_causal=causal)
        assert np.array_equal(o.to_numpy(), ref.to_numpy())
