"""f32 products whose rows are no whole groups of four: the last group of a row is read where it ends with the row.  Whole-number operands
(sums exact in f32, |sum| <= 9 K), NaNs right behind A and B, a pattern behind C."""
import numpy as np
import pytest

import morok_amd
from morok_amd import synth
from tests.test_gemm_f32_gpu import test_ragged_products_are_no_less_exact_than_64_partial_sums as ragged_accuracy

GUARD = 256


def _whole(shape, tid):
    return synth.randint(shape, 6, tid, 7).astype(np.float32) - 3.0


def _guarded(x):
    return morok_amd.Buffer.from_numpy(np.concatenate([x.reshape(-1), np.full(GUARD, np.nan, np.float32)]))


# one, two and three columns / k past a group, tiles of 64 whose last one has less than a group of columns, less than a step and odd
# numbers of steps; tiles of 32 and of 16
@pytest.mark.gpu
@pytest.mark.parametrize("nt", [False, True])
@pytest.mark.parametrize("shape", [(4200, 65, 67), (4200, 66, 129), (4200, 67, 190), (1300, 513, 258), (1300, 514, 131), (900, 961, 200), (700, 704, 77),
                                   (300, 257, 253), (481, 500, 258), (40, 33, 255), (17, 4101, 66), (129, 70, 1021)])
def test_rows_of_any_length_exact(dev, shape, nt):
    M, N, K = shape
    a, b, row = _whole((M, K), 0), _whole((K, N), 1), _whole((N,), 2)
    want = (a.astype(np.float64) @ b).astype(np.float32)
    ba, bb = _guarded(a), _guarded(np.ascontiguousarray(b.T) if nt else b)
    for kind, add in (("", None), ("_bias", row)):
        bc = morok_amd.Buffer.from_numpy(np.full(M * N + GUARD, 77.0, np.float32))
        more = [_guarded(add)] if add is not None else []
        morok_amd.Program.builtin("gemm_f32" + ("_nt" if nt else "") + kind, [M, N, K], dev.device_id).execute([bc, ba, bb, *more])
        got = bc.copyout(np.float32)
        assert np.array_equal(got[:M * N].reshape(M, N), want if add is None else want + add), kind
        assert np.all(got[M * N:] == 77.0)


# 257 to 384 tiles of 32 x 32 above K = 256, which run on tiles of 64 x 32 with sums of eight products: K and N in no groups of four, whole
# groups and whole tiles, whole groups and ragged rows, a partial last tile of columns; odd and even numbers of steps
TWO_ROUNDS = [(602, 640, 1031), (700, 500, 777), (576, 640, 704), (570, 636, 704), (481, 530, 260)]


def test_two_rounds_of_tiles_of_32():
    for m, n, k in TWO_ROUNDS:
        assert 256 < -(-m // 32) * -(-n // 32) <= 384 and k > 256


@pytest.mark.gpu
@pytest.mark.parametrize("nt", [False, True])
@pytest.mark.parametrize("shape", TWO_ROUNDS)
def test_tiles_of_64_by_32_exact(dev, shape, nt):
    test_rows_of_any_length_exact(dev, shape, nt)
    M, N, K = shape
    a, b, mat = _whole((M, K), 0), _whole((K, N), 1), _whole((M, N), 2)
    bc = morok_amd.Buffer.from_numpy(np.full(M * N + GUARD, 77.0, np.float32))
    kind = "gemm_f32" + ("_nt" if nt else "") + "_residual"
    morok_amd.Program.builtin(kind, [M, N, K], dev.device_id).execute([bc, _guarded(a), _guarded(np.ascontiguousarray(b.T) if nt else b), _guarded(mat)])
    got = bc.copyout(np.float32)
    assert np.array_equal(got[:M * N].reshape(M, N), (a.astype(np.float64) @ b).astype(np.float32) + mat)
    assert np.all(got[M * N:] == 77.0)


@pytest.mark.gpu
@pytest.mark.parametrize("nt", [False, True])
@pytest.mark.parametrize("shape", TWO_ROUNDS)
def test_tiles_of_64_by_32_are_no_less_exact_than_64_partial_sums(dev, shape, nt):
    ragged_accuracy(*shape, nt)


# Steps that end before K does run a loop of their own, two at a time, up to the three that meet the end of K: every count of whole steps around
# it, with a partial one behind and without.  Whole tiles of 64 x 64 (steps of 64), of 64 x 32 and of 128 x 128 (steps of 32), rows in no
# groups of four
@pytest.mark.gpu
@pytest.mark.parametrize("nt", [False, True])
@pytest.mark.parametrize("k", [64, 96, 100, 128, 132, 160, 192, 200, 256, 260, 320, 323, 384, 448, 516])
def test_steps_inside_of_k_exact(dev, k, nt):
    for M, N in ((640, 640), (512, 1024), (2048, 2048), (901, 963)):
        test_rows_of_any_length_exact(dev, (M, N, k), nt)
