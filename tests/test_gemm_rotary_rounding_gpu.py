"""Rotary products: the tile a shape runs on, and the last bit of a rotated value.  x cos - y sin (x sin + y cos) is one rounded product and one
fused multiply-add; which product is rounded is a property of the tiles: the sine's on small ones, on tiles of 256 x 256 the sine's in rows
0..3 of every sixteen and the cosine's in the others.  A value's bits follow from that exactly."""
import numpy as np
import pytest

import morok_amd
from morok_amd import synth
from tests.test_gemm_bf16_gpu import _gemm
from tests.test_gemm_routes_gpu import _tile

ROTARY = 2
LARGE = (256, 256, 1, 0)
# (M, N, K, rotated columns, positions): more than 256 tiles of 128 x 256 in the first seven
SHAPES = {
    (2568, 6144, 2048, 4096, 642): (128, 128, 1, 3),   # taken in turn
    (5400, 3072, 1024, 2048, 2048): (128, 128, 1, 3),
    (2440, 3112, 384, 3072, 61): (128, 128, 1, 3),
    (4001, 4608, 256, 3072, 1000): (128, 128, 1, 2),   # too few steps of K for the pipeline
    (8000, 3072, 1024, 2048, 2000): LARGE,
    (2068, 5776, 128, 5632, 100): LARGE,
    (140, 40000, 384, 39936, 140): LARGE,              # up to 256 rows
    (2124, 2888, 384, 2816, 531): (128, 128, 1, 2),    # too few steps of K for tiles of 256 x 128
    (1708, 3072, 1024, 2048, 854): (128, 128, 1, 2),
    (815, 9216, 1600, 6144, 815): (128, 128, 1, 2),    # more tiles of 128 x 128 than compute units
    (1153, 4616, 1280, 4608, 384): (128, 128, 1, 2),   # the last count of steps, and the first they are worth it from
    (1153, 4616, 1344, 4608, 384): (256, 128, 1, 3),
    (706, 3216, 384, 3072, 100): (128, 128, 1, 3),
    (147, 5384, 384, 5120, 147): (128, 64, 1, 3),
    (67, 264, 384, 256, 50): (64, 64, 1, 3),
}


def test_shapes_reach_the_tiles_they_stand_for():
    for nt in (False, True):
        for (m, n, k, _, _), tile in SHAPES.items():
            assert _tile(m, n, k, nt, ROTARY) == tile, (m, n, k)


@pytest.mark.gpu
@pytest.mark.parametrize("nt", [False, True])
@pytest.mark.parametrize("shape", list(SHAPES))
def test_rotated_values_bit_for_bit(dev, shape, nt):
    m, n, k, split, seq = shape
    a, b = synth.normal_bf16((m, k), 37, 0), synth.normal_bf16((k, n), 37, 1, sigma=k ** -0.5)
    angle = synth.uniform((seq, 64), 37, 2).astype(np.float64) * 3.0
    cos, sin = np.cos(angle).astype(np.float32), np.sin(angle).astype(np.float32)
    plain = _gemm(dev, a, b)
    ba, bb = (morok_amd.Buffer.from_numpy(x, dev.device_id) for x in (a, np.ascontiguousarray(b.T) if nt else b))
    tables = [morok_amd.Buffer.from_numpy(t, dev.device_id) for t in (cos, sin)]
    rot, rest = dev.buffer(m * split * 2), dev.buffer(max(m * (n - split) * 2, 2))
    morok_amd.Program.builtin("gemm_bf16_nt_rope" if nt else "gemm_bf16_rope", [m, n, k, split, seq], dev.device_id).execute([rot, ba, bb, rest, *tables])
    assert np.array_equal(rest.copyout(np.uint16, (m, n - split)), plain[:, split:])
    x = synth.from_bf16(plain[:, :split]).reshape(m, split // 128, 2, 64)
    pos = np.arange(m) % seq
    c, s = cos[pos][:, None], sin[pos][:, None]

    def fused(p, q, rounded):  # p q + a product rounded to f32, one rounding (p q is exact in 64 bits, and so, all but always, the sum)
        return (p.astype(np.float64) * q + rounded).astype(np.float32)

    first, second = x[:, :, 0], x[:, :, 1]
    sine = np.stack([fused(first, c, second * -s), fused(second, c, first * s)], 2)
    want = sine
    if SHAPES[shape] == LARGE:
        cosine = np.stack([fused(second, -s, first * c), fused(first, s, second * c)], 2)
        want = np.where((np.arange(m) % 16 < 4)[:, None, None, None], sine, cosine)
    assert np.array_equal(rot.copyout(np.uint16, (m, split)), synth.to_bf16(want.reshape(m, split)))
