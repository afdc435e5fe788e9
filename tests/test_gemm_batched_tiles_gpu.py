"""Batched 16-bit products long enough for the pipeline (more than four steps of K): which tile they run on, and exact results there.  Above 256
tiles of 128 x 256 that is the large tile: small ones are worth it there only where workgroups take them in turn, which those of a batch do not."""
import ctypes as C

import pytest

from morok_amd._ffi import lib
from tests.test_gemm_mid_gpu import test_small_tiles_exact as _exact

# (M, N, K, batch): rows, columns
SHAPES = {
    (640, 768, 320, 20): (256, 256),
    (1000, 3000, 384, 8): (256, 256),
    (268, 2832, 328, 8): (256, 256),
    (65, 2928, 448, 6): (128, 128),
    (500, 1208, 392, 6): (128, 128),
    (66, 2816, 328, 3): (128, 64),
    (93, 176, 392, 2): (64, 64),
}


def test_shapes_reach_the_tiles_they_stand_for():
    out = (C.c_int64 * 4)()
    for (m, n, k, batch), tile in SHAPES.items():
        for nt in (0, 1):
            assert lib.mrk_hip_gemm_16bit_tile(m, n, k, batch, nt, 0, out) == 0
            assert tuple(out[:3]) == (*tile, 1), (m, n, k, batch)


@pytest.mark.gpu
@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("nt", [False, True])
@pytest.mark.parametrize("shape", [s for s in SHAPES if s != (1000, 3000, 384, 8)])
def test_batched_products_exact(dev, shape, nt, f16):
    _exact(dev, shape, nt, f16)
