"""f32 products on the f32 matrix instructions, through the tensor API: every tile size, each layout of the weight, rows that
are and are not whole 16-byte chunks, with a bias row, with a matrix, and over views, against float64.

The bound is the forward error of a sum of K products in any order, gamma_K * (|A| |B|) with gamma_K = K u / (1 - K u)
and u = 2^-24, plus one rounding for the addend."""
import numpy as np
import pytest

import morok_amd.tensor as T

pytestmark = pytest.mark.gpu
U24 = 2.0 ** -24

SHAPES = [
    (16, 256, 64), (17, 257, 65), (1, 4100, 68), (33, 130, 200), (4000, 3, 260), (64, 96, 784),  # tiles of 16, K in 4 and 16 runs
    (31, 33, 8192), (257, 300, 256), (480, 500, 257), (512, 512, 77),                            # tiles of 32
    (640, 704, 64), (641, 703, 65), (768, 768, 191), (777, 1000, 128), (1000, 1025, 63 + 64),    # tiles of 64, odd and even steps
    (2048, 2048, 64), (2047, 2044, 100), (2049, 2052, 96),                                       # tiles of 128
]


def _bound(a, b, add=None):
    k = a.shape[1]
    mag = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    g = k * U24 / (1 - k * U24)
    return g * mag + (0 if add is None else U24 * (mag + np.abs(add))) + 1e-30


def _check(got, a, b, add=None):
    ref = a.astype(np.float64) @ b.astype(np.float64) + (0 if add is None else add)
    assert got.dtype == np.float32 and np.all(np.abs(got - ref) <= _bound(a, b, add))


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_layouts_and_addends(m, n, k):
    rng = np.random.default_rng(m * 7 + n * 3 + k)
    a, b = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
    row, mat = rng.standard_normal(n, dtype=np.float32), rng.standard_normal((m, n), dtype=np.float32)
    x, w, wt = T.Tensor.from_numpy(a), T.Tensor.from_numpy(b), T.Tensor.from_numpy(np.ascontiguousarray(b.T))
    plain = x.matmul(w)
    _check(plain.to_numpy(), a, b)
    assert plain.kernels() == [f"r_{m}_{n}_{k}"] and T.last_kernel_sources() == [""]  # (a generated kernel of that name has a source)
    lin = x.linear(wt)
    _check(lin.to_numpy(), a, b)
    assert lin.kernels() == [f"gemm_f32_nt_{m}_{n}_{k}"]
    # an addend changes nothing but the last rounding: the bits of the product followed by the add
    biased = x.linear(wt, T.Tensor.from_numpy(row))
    got = biased.to_numpy()
    assert biased.kernels() == [f"gemm_f32_nt_bias_{m}_{n}_{k}"] and np.array_equal(got, lin.to_numpy() + row)
    res = T.Tensor.from_numpy(mat).try_add(x.matmul(w))
    got = res.to_numpy()
    assert res.kernels() == [f"gemm_f32_residual_{m}_{n}_{k}"] and np.array_equal(got, plain.to_numpy() + mat)


@pytest.mark.parametrize("m,n,k", [(40, 130, 96), (600, 640, 96)])
@pytest.mark.parametrize("shift", [1, 4])
def test_views(m, n, k, shift):
    """Operands that are views: a column slice and a transposed left operand are copied first; rows sliced off the
    top may start on any float."""
    rng = np.random.default_rng(shift)
    a, b = rng.standard_normal((m + shift, k + shift), dtype=np.float32), rng.standard_normal((k + shift, n), dtype=np.float32)
    x = T.Tensor.from_numpy(a).try_shrink([(shift, m + shift), (shift, k + shift)])
    w = T.Tensor.from_numpy(b).try_shrink([(shift, k + shift), (0, n)])
    _check(x.matmul(w).to_numpy(), a[shift:, shift:], b[shift:])
    _check(T.Tensor.from_numpy(np.ascontiguousarray(a[shift:, shift:].T)).try_permute([1, 0]).matmul(w).to_numpy(), a[shift:, shift:], b[shift:])


def test_infinities_and_nan_stay_in_their_rows_and_columns():
    a, b = np.ones((70, 130), np.float32), np.ones((130, 66), np.float32)
    a[3, 129], a[69, 0], b[7, 65] = np.inf, np.nan, -np.inf
    got = T.Tensor.from_numpy(a).matmul(T.Tensor.from_numpy(b)).to_numpy()
    with np.errstate(invalid="ignore"):
        ref = a.astype(np.float64) @ b.astype(np.float64)
    assert np.array_equal(got, ref.astype(np.float32), equal_nan=True)


def _sums_of_64(a, b):
    """Row by column products the way the generated reduction adds them: lane l of a wave takes k = l, l + 64, ... one rounded
    product and one addition after the other, and the 64 partial sums meet in a tree."""
    parts = []
    for lane in range(64):
        acc = np.zeros((a.shape[0], b.shape[1]), np.float32)
        for k in range(lane, a.shape[1], 64):
            acc = acc + a[:, k:k + 1] * b[k:k + 1]
        parts.append(acc)
    while len(parts) > 1:
        parts = [parts[i] + parts[i + 1] for i in range(0, len(parts), 2)]
    return parts[0]


@pytest.mark.parametrize("nt", [False, True])
@pytest.mark.parametrize("m,n,k", [(130, 200, 130), (130, 200, 1000), (481, 501, 257), (641, 703, 130), (641, 703, 192), (641, 704, 257),
                                   (1001, 640, 777), (2049, 2052, 200), (2049, 2052, 515 + 1)])
def test_ragged_products_are_no_less_exact_than_64_partial_sums(m, n, k, nt):
    """2-norm against float64 over all outputs, against the same figure for 64 partial sums over 32 rows of it (at least 6400
    outputs: the two figures are known to 1 %)."""
    rng = np.random.default_rng(m + n + k)
    a, b = (rng.uniform(-1, 1, s).astype(np.float32) for s in ((m, k), (k, n)))
    x = T.Tensor.from_numpy(a)
    got = (x.linear(T.Tensor.from_numpy(np.ascontiguousarray(b.T))) if nt else x.matmul(T.Tensor.from_numpy(b))).to_numpy()
    ref = a.astype(np.float64) @ b.astype(np.float64)
    off = lambda y, r: np.linalg.norm(y - r) / np.linalg.norm(r)  # noqa: E731
    assert off(got, ref) <= 1.02 * off(_sums_of_64(a[:32], b), ref[:32])


@pytest.mark.parametrize("m,n,k,nt,matrix", [(65536, 1, 200, True, False), (65536, 1, 200, False, False), (300, 3, 1024, False, False),
                                             (1, 8192, 1024, True, False), (64, 10, 784, False, False), (65536, 12, 200, True, True),
                                             (8192, 10, 784, False, True), (2, 65536, 200, False, True), (129, 64 * 65536 // 129, 64, False, True)])
def test_narrow_products(m, n, k, nt, matrix):
    """A side of a few: on the matrix kernels where tiles of 16 or 32 pay, a reduction where they do not; with a bias either way."""
    rng = np.random.default_rng(m + n + k)
    a, b, row = (rng.uniform(-1, 1, s).astype(np.float32) for s in ((m, k), (k, n), (n,)))
    x = T.Tensor.from_numpy(a)
    w = T.Tensor.from_numpy(np.ascontiguousarray(b.T) if nt else b)
    y = (x.linear(w) if nt else x.matmul(w)).realize()
    assert (y.kernels() == [f"gemm_f32_nt_{m}_{n}_{k}" if nt else f"r_{m}_{n}_{k}"]) == matrix, y.kernels()
    _check(y.to_numpy(), a, b)
    z = (x.linear(w, T.Tensor.from_numpy(row)) if nt else x.matmul(w).try_add(T.Tensor.from_numpy(row))).to_numpy()
    _check(z, a, b, row)


def test_an_error_left_by_an_earlier_call_is_not_the_products():
    """The last error of a thread stays until it is read; a call that HIP refuses (a device that does not exist) leaves one."""
    import ctypes

    a = np.ones((640, 704), np.float32)
    x, w = T.Tensor.from_numpy(a), T.Tensor.from_numpy(np.ones((704, 128), np.float32))
    plan = x.matmul(w).prepare()
    maps = open("/proc/self/maps").read().split()
    hip = ctypes.CDLL(next(p for p in maps if "libamdhip64.so" in p))
    assert hip.hipSetDevice(12345) != 0
    plan.execute()
    assert np.all(T.Tensor.from_numpy(a).matmul(w).to_numpy() == 704.0)
