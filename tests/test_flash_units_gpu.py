"""Causal attention with one query tile per workgroup (few of them) and with two (many): a head's result has the same bits either way."""
import numpy as np
import pytest

from morok_amd import synth, tensor as T, uop

pytestmark = pytest.mark.gpu


# (heads, queries, head dim): more query tiles than run at once, an odd and an even number of them per head, a ragged last one
@pytest.mark.parametrize("heads,s,d", [(256, 300, 64), (256, 512, 128), (129, 257, 256)])
@pytest.mark.parametrize("mask", [False, True])
def test_units_do_not_change_the_bits(dev, heads, s, d, mask):
    s += mask * (-s % 4)
    q, k, v = (synth.normal_bf16((1, heads, s, d), 9, i) for i in range(3))
    keep = (np.arange(s) < s - 5).reshape(1, 1, 1, s)

    def run(n):
        t = [T.Tensor.from_numpy(np.ascontiguousarray(x[:, :n]), uop.BF16) for x in (q, k, v)]
        m = T.Tensor.from_numpy(keep) if mask else None
        return t[0].scaled_dot_product_attention(t[1], t[2], is_causal=True, attn_mask=m).to_numpy()

    many, few = run(heads), run(3)
    assert np.array_equal(many[:, :3], few)
    # the last head against f64: weights and the result rounded to bf16
    qf, kf, vf = (synth.from_bf16(x[0, -1]).astype(np.float64) for x in (q, k, v))
    sc = qf @ kf.T / np.sqrt(d)
    sc[~(np.tril(np.ones((s, s), bool)) & (keep[0, 0] if mask else True))] = -np.inf
    p = np.exp(sc - sc.max(-1, keepdims=True))
    want = p @ vf / p.sum(-1, keepdims=True)
    assert np.abs(synth.from_bf16(many[0, -1]) - want).max() <= 2e-2 * np.abs(want).max()


# rows of 256: pairs and single tiles by how far the last round of pairs is filled; an even and an odd count of tiles, few and many rounds
@pytest.mark.parametrize("heads,s", [(160, 378), (200, 500), (88, 628), (144, 250), (416, 300)])
def test_units_of_rows_of_256(dev, heads, s):
    test_units_do_not_change_the_bits(dev, heads, s, 256, False)
    test_units_do_not_change_the_bits(dev, heads, s, 256, True)


# rows of 64 and 128: just above one workgroup to a compute unit, and above two
@pytest.mark.parametrize("heads,s,d", [(80, 790, 128), (90, 790, 128), (208, 615, 128), (224, 615, 64), (300, 140, 64)])
def test_units_of_rows_of_64_and_128(dev, heads, s, d):
    test_units_do_not_change_the_bits(dev, heads, s, d, False)
    test_units_do_not_change_the_bits(dev, heads, s, d, True)


# heads that are a multiple of the XCDs and that are not, with eight tiles a head; four tiles a head; even counts with little left for the last round
@pytest.mark.parametrize("heads,s,d", [(69, 986, 128), (144, 984, 128), (97, 1001, 256), (72, 930, 256), (168, 512, 64), (88, 728, 256), (56, 1190, 128)])
@pytest.mark.parametrize("mask", [False, True])
def test_units_of_even_counts(dev, heads, s, d, mask):
    test_units_do_not_change_the_bits(dev, heads, s, d, mask)
