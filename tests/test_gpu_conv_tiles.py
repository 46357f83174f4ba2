"""QLinearConv and ConvInteger at the edges of the convolution kernels' tiles, bit for bit
against the oracle: position tiles (16, 32 and 64), channel tiles, chunks of K, images of a
launch, unaligned outputs, more channels than travel in the arguments, and the kernel of a
lane per position.  test_conv_plans asserts the tiles that its sizes stand for."""
import numpy as np
import pytest

from oracle import qlinear as Q
from onnx_runtime_dart_amd import _lib, ops
from tests.conv_plan import plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,c,hw,m,ks,stride,group", [
    (1, 1, 1, 1, 1, 1, 1),          # one product
    (1, 3, 7, 16, 5, 2, 1),         # P = 16, ragged K
    (2, 5, 17, 65, 3, 1, 1),        # P = 289: bytes stored one by one; a channel past a tile
    (1, 256, 7, 40, 3, 1, 1),       # K = 2304: several chunks
    (3, 57, 40, 130, 3, 1, 1),      # all channels in one workgroup, ragged K of one chunk
    (2, 16, 100, 72, 1, 1, 1),      # K = 16, 72 channels
    (1, 8, 9, 300, 3, 1, 1),        # parameters by way of scratch
    (1, 40, 5, 1100, 2, 1, 1),      # ... copied there
    (2, 24, 11, 48, 3, 2, 24),      # depthwise
    (2, 130, 20, 260, 3, 1, 130),   # ... with parameters by way of scratch
    (1, 12, 13, 128, 1, 1, 1),      # a lane per position: K = 12, 13, 28, channels split
    (1, 13, 9, 3, 1, 1, 1),
    (3, 28, 10, 64, 1, 1, 1),
    (1, 29, 190, 9, 1, 1, 1),       # ... K = 29 and 64 with many positions
    (1, 64, 182, 3, 1, 1, 1),
    (1, 1, 740, 2, 1, 1, 1),        # ... several blocks of positions per wave
])
def test_conv_tiles(n, c, hw, m, ks, stride, group):
    check(n, c, hw, m, ks, stride, group)


@pytest.mark.parametrize("n,c,hw,m,ks,pt,cw,chunks,tiles", [
    (1, 120, 90, 20, 3, 32, 2, 2, 1),
    (1, 130, 91, 9, 3, 32, 1, 2, 1),     # an odd number of positions
    (1, 15, 81, 33, 9, 32, 4, 2, 1),
    (1, 257, 87, 100, 2, 32, 8, 2, 1),   # K = 1028
    (1, 60, 130, 20, 3, 64, 2, 2, 1),
    (1, 65, 113, 300, 3, 64, 16, 2, 2),  # no LDS reduction, two channel tiles
    (5, 230, 20, 270, 3, 16, 16, 2, 2),
])
def test_conv_plans(n, c, hw, m, ks, pt, cw, chunks, tiles):
    o, k = hw + 2 * (ks // 2) - ks + 1, c * ks * ks
    p = plan(o * o, k, m, n, _lib.default_context().info()["compute_units"])
    assert (p["taps"], p["pt"], p["cw"], p["gy"]) == (0, pt, cw, tiles)
    assert -(-(-(-k // 64) * 64) // (32768 // pt)) == chunks
    check(n, c, hw, m, ks, 1, 1)


def check(n, c, hw, m, ks, stride, group):
    ctx = _lib.default_context()
    rng = np.random.default_rng(n + 3 * c + 5 * hw + 7 * m)
    x = rng.integers(0, 256, (n, c, hw, hw)).astype(np.uint8)
    w = rng.integers(-128, 128, (m, c // group, ks, ks)).astype(np.int8)
    xz, wz = np.uint8(rng.integers(0, 256)), rng.integers(-128, 128, m).astype(np.int8)
    st, pads, dl = [stride] * 2, [ks // 2] * 4, [1, 1]
    geo = dict(strides=st, pads=pads, dilations=dl, group=group)
    y = ops.op_conv_integer(x, w, xz, wz, ctx=ctx, **geo)
    np.testing.assert_array_equal(y, Q.conv_integer(x, w, xz, wz, st, pads, dl, group))
    ws = rng.uniform(0.001, 0.01, m).astype(np.float32)
    bias = rng.integers(-3000, 3000, m).astype(np.int32)
    ys, yz = np.float32(0.05 * np.sqrt(c // group * ks * ks)), np.uint8(120)
    y = ops.op_qlinear_conv(x, np.float32(0.02), xz, w, ws, wz, ys, yz, bias, lo=0, hi=255,
                            ctx=ctx, **geo)
    want = Q.qlinear_conv(x, np.float32(0.02), xz, w, ws, wz, ys, yz, bias, st, pads, dl, group,
                          0, 255)
    np.testing.assert_array_equal(y, want)


def test_conv_of_an_image_beyond_16_bit_positions():
    rng = np.random.default_rng(3)
    x = rng.integers(0, 256, (1, 1, 70001, 2)).astype(np.uint8)
    w = rng.integers(-128, 128, (4, 1, 3, 1)).astype(np.int8)
    y = ops.op_conv_integer(x, w, np.uint8(9), np.int8(3), ctx=_lib.default_context(),
                            strides=[1, 1], pads=[66000, 0, 66000, 0], dilations=[66000, 1])
    want = Q.conv_integer(x, w, np.uint8(9), np.int8(3), [1, 1], [66000, 0, 66000, 0],
                          [66000, 1])
    np.testing.assert_array_equal(y, want)


@pytest.mark.parametrize("pad", [36, 37])
@pytest.mark.parametrize("side", [0, 1])
def test_conv_at_the_limit_of_16_bit_positions(pad, side):
    # taps from -pad to 65499 + pad: told apart modulo 2^16 up to a pad of 36
    rng = np.random.default_rng(pad)
    shape, kern, pads = [1, 1, 3, 3], [2, 1, 1, 1], [0] * 4
    shape[2 + side], kern[2 + side], pads[side], pads[2 + side] = 65500, 3, pad, pad
    x = rng.integers(0, 256, shape).astype(np.uint8)
    w = rng.integers(-128, 128, kern).astype(np.int8)
    y = ops.op_conv_integer(x, w, np.uint8(9), np.int8(3), ctx=_lib.default_context(),
                            strides=[1, 1], pads=pads, dilations=[1, 1])
    want = Q.conv_integer(x, w, np.uint8(9), np.int8(3), [1, 1], pads, [1, 1])
    np.testing.assert_array_equal(y, want)


def test_wide_image_of_many_taps():
    rng = np.random.default_rng(5)
    x = rng.integers(0, 256, (1, 65, 1, 70001)).astype(np.uint8)
    w = rng.integers(-128, 128, (4, 65, 1, 3)).astype(np.int8)
    y = ops.op_conv_integer(x, w, np.uint8(9), np.int8(3), ctx=_lib.default_context(),
                            strides=[1, 1], pads=[0, 1, 0, 1], dilations=[1, 1])
    want = Q.conv_integer(x, w, np.uint8(9), np.int8(3), [1, 1], [0, 1, 0, 1], [1, 1])
    np.testing.assert_array_equal(y, want)
