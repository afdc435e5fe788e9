"""16-bit products whose N or K is no multiple of 8: padded operands, a partial last K step, rows of C that start on any
element.  Operands are small whole numbers, so every f32 sum is exact (|sum| <= 9 K < 2^24) whatever its order and the
result has to be the exactly rounded one, bit for bit; NaNs lie behind every operand and a pattern behind C."""
import numpy as np
import pytest

import morok_amd
from morok_amd import synth, tensor, uop

pytestmark = pytest.mark.gpu
GUARD = 512


def _whole(shape, tid):
    return synth.randint(shape, 6, tid, 7).astype(np.float32) - 3.0


def _bits(x, f16):
    return x.astype(np.float16).view(np.uint16) if f16 else synth.to_bf16(x)


def _guarded(dev, bits):
    return morok_amd.Buffer.from_numpy(np.concatenate([bits.reshape(-1), np.full(GUARD, 0x7FFF, np.uint16)]), dev.device_id)


# one row / column past and short of a tile and of a chunk, K of one element, a partial and a whole last K step, K in ranges
# (few tiles, long K), more than 256 rows
SHAPES = [(1, 1, 1), (2, 7, 9), (65, 9, 63), (129, 255, 65), (100, 257, 127), (257, 513, 64), (300, 1001, 320), (70, 129, 1003), (17, 999, 2050),
          (520, 3001, 72), (128, 256, 1023)]


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("nt", [False, True])
@pytest.mark.parametrize("shape", SHAPES)
def test_any_shape_exact(dev, shape, nt, f16):
    M, N, K = shape
    a, b, row, mat = _whole((M, K), 0), _whole((K, N), 1), _whole((N,), 2), _whole((M, N), 3)
    product = a.astype(np.float64) @ b
    ba, bb = _guarded(dev, _bits(a, f16)), _guarded(dev, _bits(b.T if nt else b, f16))
    base = "gemm_" + ("f16" if f16 else "bf16") + ("_nt" if nt else "")
    want = _bits(product.astype(np.float32), f16)
    rounded = want.view(np.float16).astype(np.float32) if f16 else synth.from_bf16(want)
    # the scratch the C entry point would take; enough for either layout
    pad = lambda r, c: -(-r * (-(-c // 8) * 8) * 2 // 256) * 256  # noqa: E731
    scratch = dev.buffer(pad(M, K) + max(pad(K, N), pad(N, K)) + 256 * 128 * 256 * 4)
    for kind, addend in (("", None), ("_bias", row), ("_residual", mat)):
        if addend is not None and not nt and N % 8 and K <= 128 and M * N < 1 << 19:
            continue  # small [K, N] products keep the kernel without padded operands, which has no epilogue
        bc = morok_amd.Buffer.from_numpy(np.full(M * N + GUARD, 0x1234, np.uint16), dev.device_id)
        bufs = [bc, ba, bb] + ([_guarded(dev, _bits(addend, f16))] if addend is not None else []) + [scratch]
        morok_amd.Program.builtin(base + kind, [M, N, K, 1, scratch.size], dev.device_id).execute(bufs)
        got = bc.copyout(np.uint16)
        expect = want if addend is None else _bits(rounded + addend, f16)
        assert np.array_equal(got[:M * N].reshape(M, N), expect), kind
        assert np.all(got[M * N:] == 0x1234), kind


# short and long K around the line between the kernel that reads odd rows as they are and the padded tiles, in the classes of
# rows the line is drawn for; wide weights; K in several ranges
@pytest.mark.parametrize("shape", [(3, 33, 393), (4, 50257, 200), (16, 4097, 421), (33, 7, 19), (256, 255, 129), (256, 255, 337), (256, 255, 345),
                                   (100, 513, 1001), (40, 257, 5003), (1030, 1001, 96)])
def test_the_bits_do_not_depend_on_the_kernel(dev, shape):
    M, N, K = shape
    a, b, row = synth.normal_bf16((M, K), 8, 0), synth.normal_bf16((K, N), 8, 1), synth.normal_bf16((N,), 8, 2)
    bufs = {nt: (_guarded(dev, a), _guarded(dev, np.ascontiguousarray(b.T) if nt else b)) for nt in (False, True)}
    scratch = dev.buffer((M + 8) * (K + 8) * 2 + max((K + 8) * (N + 15), (N + 8) * (K + 15)) * 2 + 256 * 128 * 256 * 4)

    def run(kind, nt, *more):
        bc = morok_amd.Buffer.from_numpy(np.full(M * N + GUARD, 0x1234, np.uint16), dev.device_id)
        morok_amd.Program.builtin(kind, [M, N, K, 1, scratch.size], dev.device_id).execute([bc, *bufs[nt], *more, scratch])
        got = bc.copyout(np.uint16)
        assert np.all(got[M * N:] == 0x1234), kind
        return got[:M * N]

    got = run("gemm_bf16", False)
    any_shape = dev.buffer(M * N * 2)
    morok_amd.ops.gemm_bf16(*bufs[False], any_shape, M, N, K, dev.device_id, variant=2)
    assert np.array_equal(got, any_shape.copyout(np.uint16, nbytes=M * N * 2))
    if M > 64 or K % 8:  # (up to 64 rows of whole chunks are streamed: another order)
        assert np.array_equal(run("gemm_bf16_nt", True), got)
        want = synth.to_bf16(synth.from_bf16(got).reshape(M, N) + synth.from_bf16(row)).reshape(-1)
        assert np.array_equal(run("gemm_bf16_nt_bias", True, _guarded(dev, row)), want)
        if K > 128:
            assert np.array_equal(run("gemm_bf16_bias", False, _guarded(dev, row)), want)


@pytest.mark.parametrize("f16", [False, True])
def test_odd_linear_through_the_tensor_api(dev, f16):
    """A projection onto an odd number of outputs, weight [out, in]: one program, no transposed copy; with a bias as well."""
    M, N, K = 130, 1003, 200
    tag = uop.F16 if f16 else uop.BF16
    x, w, bias = _whole((M, K), 4), _whole((N, K), 5), _whole((N,), 6)
    tx, tw, tb = (tensor.Tensor.from_numpy(_bits(t, f16), tag) for t in (x, w, bias))
    y = tx.linear(tw).realize()
    assert len(y.kernels()) == 1
    p = _bits((x.astype(np.float64) @ w.T).astype(np.float32), f16)
    assert np.array_equal(y.to_numpy().view(np.uint16), p)
    z = tx.linear(tw, tb).realize()
    assert len(z.kernels()) == 1
    p32 = p.view(np.float16).astype(np.float32) if f16 else synth.from_bf16(p)
    assert np.array_equal(z.to_numpy().view(np.uint16), _bits(p32 + bias, f16))
