"""Attention of a few queries under a Bool mask, whose bytes are copied chunk by chunk with the keys: against the same mask as additive zeros and
minus infinities, which every lane loads for itself.  The same bits."""
import numpy as np
import pytest

from morok_amd import synth
from morok_amd import tensor as T, uop

pytestmark = pytest.mark.gpu


# a last chunk of one to eight groups of four keys, one and several chunks a wave, one to 32 query slots (copies of eight slots each)
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("sq", [1, 7, 8, 9, 16, 17, 32])
@pytest.mark.parametrize("sk", [256, 260, 276, 284, 1052, 3000])
def test_bool_and_additive_masks_agree(dev, sk, sq, d):
    q, k, v = (T.Tensor.from_numpy(synth.normal_bf16(s, 41, i), uop.BF16) for i, s in enumerate([(2, 3, sq, d), (2, 3, sk, d), (2, 3, sk, d)]))
    keep = synth.randint((2, 3, sq, sk), 41, 5, 3) > 0
    keep[..., 0] = True
    keep[0, 0, :, 40:200] = False  # (chunks without a visible key)
    added = synth.to_bf16(np.where(keep, 0.0, -np.inf).astype(np.float32))
    got = q.scaled_dot_product_attention(k, v, attn_mask=T.Tensor.from_numpy(keep)).to_numpy()
    want = q.scaled_dot_product_attention(k, v, attn_mask=T.Tensor.from_numpy(added, uop.BF16)).to_numpy()
    assert np.all(np.isfinite(synth.from_bf16(want)))
    assert np.array_equal(got, want)
