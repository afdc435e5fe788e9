"""Attention of a few queries in a prepared plan: the last workgroup of a pair folds the pair's key ranges.  Against the same graph realized, whose
ranges a second kernel folds in the same order: the same bits, on every execution and every replay."""
import numpy as np
import pytest

import morok_amd
from morok_amd import synth
from morok_amd import tensor as T, uop
from morok_amd._ffi import lib
from tests.test_flash_decode_gpu import _attn, _check, _inputs


def _build(B, H, group, Sq, Sk, d, mask, cap, seed):
    """group > 1: heads that share their keys."""
    q, k, v = (T.Tensor.from_numpy(synth.normal_bf16(s, seed, i), uop.BF16) for i, s in
               enumerate([(B, H, Sq, d), (B, 1 if group else H, Sk, d), (B, 1 if group else H, Sk, d)]))
    if group:
        k, v = k.try_expand([B, H, Sk, d]), v.try_expand([B, H, Sk, d])
    m = None
    if mask:
        keep = np.arange(Sk)[None, :] < np.maximum(1, synth.randint((B, 1), seed, 7, Sk))
        m = T.Tensor.from_numpy(np.ascontiguousarray(keep.reshape(B, 1, 1, Sk)))
    return lambda: q.scaled_dot_product_attention(k, v, attn_mask=m, softcap=cap)


# two ranges and the most there are; one, several and 32 query slots; more partial results than a workgroup's local memory holds (the
# second kernel folds those); heads that share their keys; masks that leave ranges empty
CASES = [(1, 32, False, 1, 4096, 128, False, None), (2, 3, False, 1, 1030, 64, False, None), (1, 1, False, 1, 70000, 128, False, None),
         (1, 4, False, 3, 5000, 256, False, None), (1, 2, False, 32, 16384, 128, False, None), (1, 1, False, 17, 2000, 64, False, None),
         (4, 8, True, 1, 9000, 128, False, None), (3, 12, True, 2, 3000, 256, False, None), (2, 4, True, 1, 5000, 256, False, None), (3, 4, False, 1, 4100, 128, True, None),
         (2, 4, False, 2, 2048, 64, True, 20.0), (40, 4, False, 1, 513, 128, False, None), (1, 2, False, 1, 300, 128, False, None),
         # (more partial results than are folded by counting, and just as many: many ranges of few slots, two blocks of slots, rows of 256)
         (2, 8, True, 1, 12000, 128, False, None), (1, 8, True, 1, 12000, 64, False, None), (2, 4, False, 24, 1500, 128, False, None), (1, 8, False, 8, 4096, 128, False, None),
         (16, 4, False, 3, 1500, 256, False, None), (2, 4, False, 4, 1500, 256, False, None), (1, 3, False, 1, 12000, 256, True, None)]


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(x) for x in c))
def test_a_plans_executions_match_a_realization(dev, case):
    B, H, group, Sq, Sk, d, mask, cap = case
    build = _build(B, H, group, Sq, Sk, d, mask, cap, seed=31)
    want = build().realize().to_numpy()
    root = build()
    plan = root.prepare()
    other = T.Tensor.from_numpy(np.ones((64, 512), np.float32))
    for i in range(4):
        root.buffer().copyin(np.full(want.shape, 0x7FC0, np.uint16))
        if i < 2:
            plan.execute()
        else:
            plan.execute_graph()
        got = root.buffer().copyout(np.uint16, want.shape)
        assert np.array_equal(got, want), i
        assert np.all(other.try_mul(float(i)).sum(1).to_numpy() == 512.0 * i)  # (work of others in between)


@pytest.mark.gpu
def test_executions_that_follow_each_other_without_a_wait(dev):
    build = _build(2, 4, False, 1, 6000, 128, False, None, seed=32)
    want = build().realize().to_numpy()
    roots = [build() for _ in range(3)]
    plans = [r.prepare() for r in roots]
    for _ in range(50):
        for p in plans:
            p.execute()
    for r in roots:
        assert np.array_equal(r.buffer().copyout(np.uint16, want.shape), want)


# Pairs, query slots, keys, head dim: ranges a pair.  Rows of 256 in as many workgroups as there are compute units, or one more pair than that; more
# ranges in a band of pairs above, its first and last count and the keys, by slots, from which there are two and three
RANGES = {(96, 1, 1231, 256): 2, (129, 1, 900, 256): 1, (257, 1, 1499, 256): 1, (257, 1, 1500, 256): 3, (320, 8, 1500, 256): 3, (320, 16, 2499, 256): 1, (320, 16, 2500, 256): 3, (321, 1, 1530, 256): 1,
          (260, 17, 1500, 128): 1, (257, 1, 1499, 128): 1, (257, 1, 1500, 128): 2, (320, 1, 1535, 128): 2, (257, 1, 1536, 128): 3, (288, 8, 2199, 128): 1, (288, 8, 2200, 128): 3, (320, 16, 2999, 128): 1, (320, 16, 3000, 128): 3,
          (321, 1, 1600, 128): 1, (256, 1, 1600, 128): 1, (257, 1, 1600, 64): 1}


def test_ranges_of_a_pair():
    for (pairs, slots, Sk, d), ranges in RANGES.items():
        slice_bytes = pairs * (16 if slots <= 16 else 32) * (d + 2) * 4
        got = lib.mrk_hip_flash_attn_workspace_bytes(1, pairs, slots, Sk, d, 0)
        # (the scratch also holds what runs of heads that share their keys would take: less than two ranges of all pairs)
        assert max(1, got // slice_bytes) == ranges, (pairs, slots, Sk, d)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(6, 16, 1, 1231, 256), (1, 129, 1, 900, 256), (1, 257, 1, 1500, 128), (10, 32, 1, 1501, 128), (1, 321, 1, 1500, 128),
                                   (1, 260, 16, 1530, 256), (1, 260, 17, 1500, 128),
                                   (1, 320, 1, 1535, 128), (1, 257, 1, 1536, 128), (2, 160, 2, 1601, 128), (1, 257, 8, 1500, 256)])
def test_ranges_that_follow_the_count_of_compute_units(dev, oracle, shape):
    B, H, Sq, Sk, d = shape
    q, k, v = _inputs(B, H, Sq, Sk, d, seed=33)
    want = oracle.sdpa_bf16(q, k, v, float(d) ** -0.5, causal=False)
    for mode in ("abi", "program", "program_ws"):
        _check(_attn(dev, q, k, v, float(d) ** -0.5, mode=mode), want)


@pytest.mark.gpu
def test_counters_come_with_a_workspace(dev):
    bits = int(np.float32(0.1).view(np.uint32))
    for params in ([8, 1, 2048, 128, 0, bits, 0, 1], [8, 1, 2048, 128, 0, bits, 1 << 20, 2]):
        with pytest.raises(morok_amd.MorokHipError):
            morok_amd.Program.builtin("flash_fwd_bf16", params, dev.device_id)
    ws = lib.mrk_hip_flash_attn_workspace_bytes(8, 1, 1, 2048, 128, 0)
    assert morok_amd.Program.builtin("flash_fwd_bf16", [8, 1, 2048, 128, 0, bits, ws, 1], dev.device_id).name.endswith("_splitkv")
