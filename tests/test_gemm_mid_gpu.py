"""16-bit products on tiles of 64 and 128 (gemm_mid.hip): edges of the tiles, partial last K steps, K in ranges, batches, and bases that are
not aligned.  Operands are small whole numbers, so every f32 sum is exact (|sum| <= 9 K < 2^24) whatever its order and the result
has to be the exactly rounded one, bit for bit; NaNs lie behind every operand and a pattern behind C."""
import numpy as np
import pytest

import morok_amd
from morok_amd import ops, synth

pytestmark = pytest.mark.gpu
GUARD = 512


def _whole(shape, tid):
    return synth.randint(shape, 6, tid, 7).astype(np.float32) - 3.0


def _bits(x, f16):
    return x.astype(np.float16).view(np.uint16) if f16 else synth.to_bf16(x)


def _guarded(dev, bits):
    return morok_amd.Buffer.from_numpy(np.concatenate([bits.reshape(-1), np.full(GUARD, 0x7FFF, np.uint16)]), dev.device_id)


# one short of, at and past a tile of 64 in rows and columns; one K step, one chunk more, fewer steps than stages; several ranges of K with
# a partial last step; a batch (the other tiles: test_gemm_routes_gpu.py)
SHAPES = [(65, 64, 64, 1), (127, 72, 72, 1), (129, 136, 136, 1), (128, 248, 200, 1), (66, 1408, 512, 1), (100, 264, 4000, 1), (200, 1000, 1096, 1),
          (2106, 1024, 264, 1), (250, 4104, 1032, 1), (600, 3704, 1544, 1), (70, 72, 1000, 3), (130, 65, 129, 2)]


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("nt", [False, True])
@pytest.mark.parametrize("shape", SHAPES)
def test_small_tiles_exact(dev, shape, nt, f16):
    M, N, K, batch = shape
    a, b = _whole((batch, M, K), 0), _whole((batch, K, N), 1)
    product = np.matmul(a.astype(np.float64), b)
    want = _bits(product.astype(np.float32), f16)
    rounded = want.view(np.float16).astype(np.float32) if f16 else synth.from_bf16(want)
    ba, bb = _guarded(dev, _bits(a, f16)), _guarded(dev, np.ascontiguousarray(_bits(b.transpose(0, 2, 1) if nt else b, f16)))
    row, mat = _whole((N,), 2), _whole((batch, M, N), 3)
    pad = lambda r, c: -(-r * (-(-c // 8) * 8) * 2 // 256) * 256  # noqa: E731
    scratch = dev.buffer(batch * (pad(M, K) + max(pad(K, N), pad(N, K))) + (32 << 20))
    for kind, addend in (("", None), ("_bias", row), ("_residual", mat)):
        bc = morok_amd.Buffer.from_numpy(np.full(batch * M * N + GUARD, 0x1234, np.uint16), dev.device_id)
        more = [_guarded(dev, _bits(addend, f16))] if addend is not None else []
        base = "gemm_" + ("f16" if f16 else "bf16") + ("_nt" if nt else "")
        morok_amd.Program.builtin(base + kind, [M, N, K, batch, scratch.size], dev.device_id).execute([bc, ba, bb, *more, scratch])
        got = bc.copyout(np.uint16)
        expect = want if addend is None else _bits(rounded + addend, f16)
        assert np.array_equal(got[:batch * M * N], expect.reshape(-1)), kind
        assert np.all(got[batch * M * N:] == 0x1234), kind


@pytest.mark.parametrize("shape", [(70, 72, 136), (129, 65, 700), (100, 264, 4000), (300, 2056, 520)])
def test_bases_on_any_element_give_the_same_bits(dev, shape):
    """Operands and result one element behind a 16-byte boundary."""
    M, N, K = shape
    a, b = synth.normal_bf16((M, K), 8, 0), synth.normal_bf16((K, N), 8, 1)
    # (the sums in the ranges of K that the kernel without scratch takes as well)
    aligned = dev.buffer(M * N * 2)
    ops.gemm_bf16(morok_amd.Buffer.from_numpy(a), morok_amd.Buffer.from_numpy(b), aligned, M, N, K, dev.device_id)
    one = lambda x: np.concatenate([np.zeros(1, np.uint16), x.reshape(-1), np.full(GUARD, 0x7FFF, np.uint16)])  # noqa: E731
    ba, bb = morok_amd.Buffer.from_numpy(one(a)), morok_amd.Buffer.from_numpy(one(b))
    bc = morok_amd.Buffer.from_numpy(np.full(1 + M * N + GUARD, 0x1234, np.uint16))
    ops.gemm_bf16(ba.ptr + 2, bb.ptr + 2, bc.ptr + 2, M, N, K, dev.device_id)
    got = bc.copyout(np.uint16)
    assert np.array_equal(got[1:1 + M * N], aligned.copyout(np.uint16, nbytes=M * N * 2))
    assert got[0] == 0x1234 and np.all(got[1 + M * N:] == 0x1234)
