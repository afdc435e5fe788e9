"""16-bit products on every tile a shape can be sent to.  Which one that is follows from an estimate of the time, so each shape here states
its tile (rows, columns, ranges of K, stages of the small-tile kernel, 0: the kernels of large tiles), checked on the CPU: an estimate
fitted anew cannot leave a kernel without a test.  The checks themselves are those of the tests imported here."""
import ctypes as C

import pytest

from morok_amd._ffi import lib
from tests.test_gemm_bf16_gpu import (test_gemm_rotary_epilogue as _rotary, test_gemm_swiglu_epilogue_parity as _gated,
                                      test_gemm_transposed_second_operand as _transposed,
                                      test_gemm_transposed_second_operand_epilogues as _transposed_epilogues)
from tests.test_gemm_mid_gpu import test_small_tiles_exact as _exact

# (M, N, K): each tile with ragged rows and columns, whole and partial last steps of K, and K in ranges
PLAIN = {
    (1164, 2744, 64): (128, 128, 1, 2),
    (201, 8200, 3976): (128, 128, 3, 2),
    (676, 4872, 488): (128, 128, 1, 3),
    (452, 6632, 600): (128, 128, 1, 3),
    (415, 1848, 5944): (128, 128, 4, 3),
    (2131, 856, 9936): (128, 128, 2, 3),
    (2297, 688, 72): (128, 64, 1, 3),
    (900, 160, 9712): (128, 64, 8, 3),
    (100, 264, 4000): (64, 64, 8, 3),
    (972, 5592, 64): (128, 256, 1, 0),
    (1314, 4976, 72): (128, 256, 1, 0),
    (136, 4424, 6088): (128, 256, 7, 0),
    (2169, 4400, 64): (256, 256, 1, 0),
    (1322, 6672, 72): (256, 256, 1, 0),
    (2169, 4401, 136): (256, 256, 1, 0),
}
# (M, N = gate and up, K) and (M, N, K, rotated columns, positions)
GATED = {(2068, 5776, 128): (256, 256, 1, 0), (1040, 11056, 72): (256, 256, 1, 0), (67, 9248, 64): (128, 64, 1, 3), (664, 7456, 72): (128, 128, 1, 2),
         (1553, 7440, 136): (128, 128, 1, 3)}
ROTARY = {(2068, 5776, 128, 5632, 100): (256, 256, 1, 0), (1040, 11056, 192, 10752, 1040): (256, 256, 1, 0), (67, 9240, 64, 9216, 50): (128, 64, 1, 3),
          (664, 7456, 64, 7168, 64): (128, 128, 1, 2), (1553, 7440, 128, 7424, 512): (128, 128, 1, 2), (193, 8216, 128, 7936, 193): (128, 128, 1, 3)}


def _tile(m, n, k, nt=False, paired=False):
    out = (C.c_int64 * 4)()
    assert lib.mrk_hip_gemm_16bit_tile(m, n, k, 1, nt, paired, out) == 0
    return tuple(out)


def test_shapes_reach_the_tiles_they_stand_for():
    for nt in (False, True):
        for shape, tile in PLAIN.items():
            assert _tile(*shape, nt) == tile, shape
        for shape, tile in GATED.items():
            assert _tile(*shape, nt, True) == tile, shape
        for (m, n, k, _, _), tile in ROTARY.items():
            assert _tile(m, n, k, nt, 2) == tile, (m, n, k)
    assert _tile(300, 3001, 777) == (64, 64, 1, 2)            # rows that start on any element
    assert _tile(8, 4096, 4096, True)[0] == 0                  # streamed


@pytest.mark.parametrize("m,n,k", [(1 << 30, 16, 8), (1 << 30, 256, 8), (1 << 28, 264, 64)])
def test_tiles_stay_within_the_launch_limit(m, n, k):
    """A grid dimension holds fewer than 2^32 work-items: products of that many small tiles stay on tiles of 256 x 256."""
    for nt in (False, True):
        rows, cols, _, stages = _tile(m, n, k, nt, True)
        groups = -(-m // rows) * -(-(-(-n // 128) * 128) // cols)
        assert groups * (256 if stages else 512) < 1 << 32, (rows, cols)


@pytest.mark.gpu
@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("nt", [False, True])
@pytest.mark.parametrize("shape", list(PLAIN))
def test_plain_bias_and_residual_exact(dev, shape, nt, f16):
    _exact(dev, (*shape, 1), nt, f16)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [s for s in PLAIN if s[1] % 8 == 0 and s[2] < 1000])
def test_both_layouts_give_the_same_bits(dev, oracle, shape):
    _transposed(dev, oracle, shape)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", list(GATED))
def test_gated_epilogue(dev, oracle, shape):
    m, n, k = shape
    _gated(dev, oracle, (m, n // 2, k))
    _transposed_epilogues(dev, shape)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", list(ROTARY))
def test_rotary_epilogue(dev, oracle, shape):
    _rotary(dev, oracle, shape)
