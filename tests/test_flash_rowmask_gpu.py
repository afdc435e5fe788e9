"""Attention under a Bool mask that is one row of keys for every query (a key-padding mask): whole tiles of hidden keys at the
end, in the middle and at the front, rows of one visible key, with and without the causal rule, against the kernel for
masks of any shape (the same mask expanded over the queries in memory), and rows that see nothing come out as NaN."""
import numpy as np
import pytest

import morok_amd.tensor as T
from morok_amd import synth, uop

pytestmark = pytest.mark.gpu


def _attend(q, k, v, mask, causal):
    t = [T.Tensor.from_numpy(x, uop.BF16) for x in (q, k, v)]
    out = t[0].scaled_dot_product_attention(t[1], t[2], is_causal=causal, attn_mask=T.Tensor.from_numpy(mask))
    got = synth.from_bf16(out.to_numpy())
    # (more than 65536 keys: the general kernel for any mask)
    row = mask.shape[2] == 1 and k.shape[2] <= 65536
    assert out.kernels()[0].startswith("flash_fwd_bf16_ext_bool" + ("_row_" if row else "_")), out.kernels()
    assert row or "_row_" not in out.kernels()[0]
    return got


def _row(pattern, sk, rng):
    row = np.ones(sk, bool)
    if pattern == "end":
        row[rng.integers(1, sk):] = False
    elif pattern == "one":
        row[:] = False
        row[rng.integers(0, sk)] = True
    elif pattern == "front":
        row[:rng.integers(0, sk)] = False
    elif pattern == "middle" and sk > 150:
        row[64:140] = False
    elif pattern == "random":
        row = rng.random(sk) < 0.5
        row[rng.integers(0, sk)] = True
    elif pattern == "last":
        row[-1] = False
    return row


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("sq,sk", [(33, 4), (130, 64), (128, 68), (257, 192), (300, 1000), (40, 4160)])
def test_row_mask_matches_the_general_kernel(d, causal, sq, sk):
    if causal:
        sk = (sq + 3) // 4 * 4
        sq = sk
    rng = np.random.default_rng(sq * 31 + sk + d + causal)
    patterns = ["all", "end", "one", "front", "middle", "random", "last"]
    B, H = len(patterns), 2
    q, k, v = (synth.normal_bf16((B, H, s, d), 11, i) for i, s in enumerate((sq, sk, sk)))
    rows = np.stack([_row(p, sk, rng) for p in patterns])[:, None, None, :]
    if causal:
        rows[..., 0] = True   # (a query that sees nothing is NaN: below)
    got = _attend(q, k, v, np.ascontiguousarray(rows), causal)
    want = _attend(q, k, v, np.ascontiguousarray(np.broadcast_to(rows, (B, 1, sq, sk))), causal)
    # the two round probabilities to bf16 against reference points that may differ by up to 2^8, and the result once:
    # 2^-9 relative each on terms whose sum is at most max |v|
    assert np.all(np.isfinite(got)) and np.abs(got - want).max() <= 2.0 ** -8 * np.abs(synth.from_bf16(v)).max()


@pytest.mark.parametrize("sk", [65532, 65536, 65540])
@pytest.mark.parametrize("pattern", ["end", "one", "random", "last"])
def test_the_longest_rows(sk, pattern):
    """The last tile whose words fit the local memory, and one key group more, which the general kernel takes."""
    rng = np.random.default_rng(sk)
    q, k, v = (synth.normal_bf16((1, 2, s, 64), 13, i) for i, s in enumerate((40, sk, sk)))
    row = _row(pattern, sk, rng)[None, None, None, :]
    got = _attend(q, k, v, row, False)
    want = _attend(q, k, v, np.ascontiguousarray(np.broadcast_to(row, (1, 1, 40, sk))), False)
    assert np.all(np.isfinite(got)) and np.abs(got - want).max() <= 2.0 ** -8 * np.abs(synth.from_bf16(v)).max()


def test_rows_that_see_nothing_are_nan():
    q, k, v = (synth.normal_bf16((2, 2, s, 64), 12, i) for i, s in enumerate((100, 200, 200)))
    mask = np.ones((2, 1, 1, 200), bool)
    mask[1] = False
    got = _attend(q, k, v, mask, False)
    assert np.all(np.isfinite(got[0])) and np.all(np.isnan(got[1]))
