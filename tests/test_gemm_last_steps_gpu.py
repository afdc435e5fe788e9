"""The tiles of 256 and 128 rows over a partial last step of K and over odd columns: the steps that copy the last tile run a loop of their own,
so every count of steps around it, whole and partial; odd columns inside C and at its edge.  Small whole numbers, as in
test_gemm_any_shape_gpu.py: the result has to be the exactly rounded one."""
import numpy as np
import pytest

import morok_amd
from morok_amd import ops, synth
from tests.test_gemm_any_shape_gpu import GUARD, _bits, _guarded, _whole, test_any_shape_exact as _exact
from tests.test_gemm_routes_gpu import _tile

ODD = [(2300, 4001, 64 * steps) for steps in (1, 3, 4, 5, 6)] + [(2300, 4001, 200), (2049, 4105, 328)]  # (tiles inside C, at its right and at its lower edge)


def test_odd_columns_reach_the_large_tiles():
    assert all(_tile(*shape, True) == (256, 256, 1, 0) for shape in ODD)


@pytest.mark.gpu
@pytest.mark.parametrize("variant", [3, 4])
@pytest.mark.parametrize("left", [8, 40, 64])
@pytest.mark.parametrize("steps", range(1, 10))
def test_every_count_of_steps(dev, steps, left, variant):
    M, N, K = 300, 520, 64 * (steps - 1) + left
    a, b = _whole((M, K), 0), _whole((K, N), 1)
    ba, bb = _guarded(dev, _bits(a, False)), _guarded(dev, _bits(b, False))
    bc = morok_amd.Buffer.from_numpy(np.full(M * N + GUARD, 0x1234, np.uint16), dev.device_id)
    ops.gemm_bf16(ba, bb, bc, M, N, K, dev.device_id, variant)
    got = bc.copyout(np.uint16)
    assert np.array_equal(got[:M * N].reshape(M, N), synth.to_bf16((a.astype(np.float64) @ b).astype(np.float32)))
    assert np.all(got[M * N:] == 0x1234)


@pytest.mark.gpu
@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("shape", ODD)
def test_odd_columns_exact(dev, shape, f16):
    _exact(dev, shape, True, f16)
