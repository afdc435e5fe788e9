"""16-bit products whose copies are made by waves of their own, in one range of K long enough for the pipeline (more than four steps; tiles
of 64 x 64 more than eight, and no more of them than compute units, with shapes on either side): every tile such a product can be sent to, with ragged rows and columns, whole and partial last steps of K.  As in test_gemm_routes_gpu.py each
shape states its tile, checked on the CPU; the checks themselves are those of the tests imported here."""
import numpy as np
import pytest

import morok_amd
from morok_amd import synth
from tests.test_gemm_bf16_gpu import (test_gemm_rotary_epilogue as _rotary, test_gemm_swiglu_epilogue_parity as _gated,
                                      test_gemm_transposed_second_operand as _transposed,
                                      test_gemm_transposed_second_operand_epilogues as _transposed_epilogues)
from tests.test_gemm_mid_gpu import test_small_tiles_exact as _exact
from tests.test_gemm_routes_gpu import _tile

PLAIN = {
    (65, 72, 328): (64, 64, 1, 3),        # one row and one chunk of columns past a tile
    (65, 72, 584): (64, 64, 1, 3),        # the same, ten steps: with such waves
    (256, 2048, 576): (64, 64, 1, 3),     # nine, the first with them
    (1024, 1024, 640): (64, 64, 1, 3),    # as many tiles as compute units
    (147, 9392, 1160): (64, 64, 1, 3),    # more
    (256, 2048, 512): (64, 64, 1, 3),     # whole tiles
    (129, 5592, 360): (128, 64, 1, 3),
    (384, 3072, 1024): (128, 64, 1, 3),
    (341, 5464, 328): (128, 128, 1, 3),
    (1541, 4968, 328): (128, 128, 1, 3),  # more than 256 tiles of 128 x 256
    (2492, 3144, 328): (256, 128, 1, 3),
}
GATED = {(68, 144, 392): (64, 64, 1, 3), (68, 144, 584): (64, 64, 1, 3), (147, 5456, 360): (128, 64, 1, 3), (2055, 912, 328): (128, 128, 1, 3), (2124, 2880, 704): (128, 128, 1, 2), (2124, 2880, 712): (256, 128, 1, 3)}
# More tiles than the 256 workgroups that take them in turn, two and three a workgroup: the copies run on into the next tile while the last is
# stored.  Ragged rows and columns, and counts of steps (K) with every remainder by the ring's three stages, with a partial last step and without
IN_TURN = {
    (769, 9376, 352): (128, 128, 1, 3),   # six steps
    (642, 11096, 280): (128, 128, 1, 3),  # five; 522 tiles
    (790, 9776, 448): (128, 128, 1, 3),   # seven; 539 tiles
    (1281, 10800, 520): (256, 128, 1, 3),  # nine
    (1540, 9264, 512): (256, 128, 1, 3),  # eight
    (4100, 5640, 448): (256, 128, 1, 3),  # seven; 765 tiles
}
IN_TURN_GATED = {(376, 22240, 376): (128, 128, 1, 3), (376, 22240, 440): (128, 128, 1, 3), (280, 20304, 2112): (128, 128, 1, 3), (1281, 10768, 376): (256, 128, 1, 3), (4096, 5632, 1024): (256, 128, 1, 3)}
ROTARY = {(67, 264, 384, 256, 50): (64, 64, 1, 3), (67, 264, 704, 256, 50): (64, 64, 1, 3), (147, 5384, 384, 5120, 147): (128, 64, 1, 3), (706, 3216, 384, 3072, 100): (128, 128, 1, 3),
          (2124, 2888, 1344, 2816, 531): (256, 128, 1, 3)}


def _in_turn(tile, m, n):
    return tile[0] * tile[1] >= 128 * 128 and tile[3] == 3 and -(-m // tile[0]) * -(-n // tile[1]) > 256


def test_shapes_reach_the_tiles_they_stand_for():
    for nt in (False, True):
        for shape, tile in PLAIN.items():
            assert _tile(*shape, nt) == tile, shape
        for shape, tile in GATED.items():
            assert _tile(*shape, nt, True) == tile, shape
        for (m, n, k, _, _), tile in ROTARY.items():
            assert _tile(m, n, k, nt, 2) == tile, (m, n, k)
        for k, tall in ((384, (128, 128)), (1344, (256, 128))):  # (of the last test)
            for m, tile in ((2440, (128, 128)), (1830, tall), (732, (128, 128)), (61, (64, 64))):
                assert _tile(m, 3112, k, nt, 2)[:2] == tile, m
        for shapes, paired in ((IN_TURN, 0), (IN_TURN_GATED, 1)):
            for (m, n, k), tile in shapes.items():
                assert _tile(m, n, k, nt, paired) == tile, (m, n, k)
                assert _in_turn(tile, m, n), (m, n, k)


@pytest.mark.gpu
@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("nt", [False, True])
@pytest.mark.parametrize("shape", list(PLAIN))
def test_plain_bias_and_residual_exact(dev, shape, nt, f16):
    _exact(dev, (*shape, 1), nt, f16)


@pytest.mark.gpu
@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("nt", [False, True])
@pytest.mark.parametrize("shape", list(IN_TURN))
def test_tiles_in_turn_exact(dev, shape, nt, f16):
    _exact(dev, (*shape, 1), nt, f16)


@pytest.mark.gpu
@pytest.mark.parametrize("nt", [False, True])
@pytest.mark.parametrize("shape", list(IN_TURN_GATED))
def test_gated_tiles_in_turn(dev, shape, nt):
    """Against the same rows in products of few enough tiles for a workgroup each: the same bits, whichever tile those run on."""
    m, n, k = shape
    a, w = synth.normal_bf16((m, k), 41, 0), synth.normal_bf16((k, n), 41, 1, sigma=k ** -0.5)
    ba = morok_amd.Buffer.from_numpy(a, dev.device_id)
    bw = morok_amd.Buffer.from_numpy(np.ascontiguousarray(w.T) if nt else w, dev.device_id)
    bc = morok_amd.Buffer.from_numpy(np.full(m * n // 2 + 64, 0x7FC0, np.uint16), dev.device_id)
    kind = "gemm_bf16_nt_swiglu" if nt else "gemm_bf16_swiglu"
    morok_amd.Program.builtin(kind, [m, n // 2, k], dev.device_id).execute([bc, ba, bw])
    got = bc.copyout(np.uint16)
    assert np.all(got[m * n // 2:] == 0x7FC0)
    got = got[:m * n // 2].reshape(m, n // 2)
    for first in range(0, m, 120):  # (more than the 64 rows that are streamed)
        rows = min(120, m - first)
        if rows < 65:
            first, rows = m - 65, 65
        assert not _in_turn(_tile(rows, n, k, nt, 1), rows, n)
        part = dev.buffer(rows * n)
        morok_amd.Program.builtin(kind, [rows, n // 2, k], dev.device_id).execute([part, ba.view(first * k * 2, rows * k * 2), bw])
        assert np.array_equal(part.copyout(np.uint16, (rows, n // 2)), got[first:first + rows]), first


@pytest.mark.gpu
@pytest.mark.parametrize("shape", list(PLAIN))
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


@pytest.mark.gpu
@pytest.mark.parametrize("nt", [False, True])
@pytest.mark.parametrize("k", [384, 1344])
def test_rotation_gives_the_same_bits_on_every_tile(dev, k, nt):
    """The same rows in products of each small tile and of more tiles than workgroups (2440 rows): all round the products of a rotation alike.
    (Tiles of 256 x 256 do not: test_gemm_rotary_rounding_gpu.py.)"""
    n, split, seq = 3112, 3072, 61
    rows = (2440, 1830, 732, 61)
    a, b = synth.normal_bf16((2440, k), 31, 0), synth.normal_bf16((k, n), 31, 1, sigma=k ** -0.5)
    angle = synth.uniform((seq, 64), 31, 2).astype(np.float64) * 3.0
    cos, sin = (morok_amd.Buffer.from_numpy(f(angle).astype(np.float32), dev.device_id) for f in (np.cos, np.sin))
    bb = morok_amd.Buffer.from_numpy(np.ascontiguousarray(b.T) if nt else b, dev.device_id)
    got = []
    for m in rows:
        ba = morok_amd.Buffer.from_numpy(np.ascontiguousarray(a[:m]), dev.device_id)
        rot, rest = dev.buffer(m * split * 2), dev.buffer(m * (n - split) * 2)
        morok_amd.Program.builtin("gemm_bf16_nt_rope" if nt else "gemm_bf16_rope", [m, n, k, split, seq], dev.device_id).execute([rot, ba, bb, rest, cos, sin])
        got.append((rot.copyout(np.uint16, (m, split)), rest.copyout(np.uint16, (m, n - split))))
    for rot, rest in got[1:]:
        assert np.array_equal(rot, got[0][0][:len(rot)]) and np.array_equal(rest, got[0][1][:len(rest)])
