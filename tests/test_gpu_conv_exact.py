"""The learned preconditioner's convolution kernels, bit for bit against the
CPU restatement (oracle/convnet.py, pinned by direct sums and finite
differences in tests/test_convnet_oracle.py).

Inputs and weights are small integers, exact in BF16; every product and
every partial sum is an integer far below 2^24, so FP32 accumulation on the
MFMA units is exact in any order and the device's output must equal the
restatement's exactly.  A tap dropped or doubled at a tile seam, a transposed
channel block or a misplaced halo changes some output by at least 1.

The grids span the kernels' tile seams: 151 x 131 pixels is three 64-pixel
tile columns (the last partial) and a partial last tile row of the tiled
forward kernel; the 3D grids cover the tiled kernel's tile lengths along
the lines and partial 4-line tiles.
"""
import numpy as np
import pytest

from oracle import convnet as cn

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import pansfem2_amd as pa
    c = pa.Context(0)
    yield c
    c.close()


def ints(rng, shape, lo, hi):
    return rng.integers(lo, hi + 1, size=shape).astype(np.float32)


# the (cin, cout) pairs the network launches (64-channel layers: 62-88 KB of LDS)
SHAPES_2D = [(16, 16), (16, 32), (32, 16), (32, 32), (32, 64), (64, 32)]


@pytest.mark.parametrize("cin,cout", SHAPES_2D)
def test_conv2d_forward_exact(ctx, cin, cout):
    rng = np.random.default_rng(100 + cin + cout)
    H, W = 151, 131
    x = ints(rng, (H, W, cin), -3, 3)
    w = ints(rng, (9, cout, cin), -3, 3)
    y = ctx.conv_raw(x, w)
    ref = cn.conv(x.astype(np.float64), w.astype(np.float64))
    assert np.max(np.abs(ref)) < 2 ** 20
    assert np.array_equal(y.astype(np.float64), ref), float(np.max(np.abs(y - ref)))


@pytest.mark.parametrize("cin,cout", SHAPES_2D)
def test_conv2d_weight_gradient_exact(ctx, cin, cout):
    rng = np.random.default_rng(200 + cin + cout)
    H, W = 151, 131
    x = ints(rng, (H, W, cin), -2, 2)
    dz = ints(rng, (H, W, cout), -2, 2)
    g = ctx.conv_wgrad_raw(x, dz)
    _, ref = cn.conv_grads(x.astype(np.float64), dz.astype(np.float64), np.zeros((9, cout, cin)))
    assert np.sum(np.abs(x)) * 2 < 2 ** 24
    assert np.array_equal(g.astype(np.float64), ref), float(np.max(np.abs(g - ref)))


@pytest.mark.parametrize("H,W,D", [(9, 7, 70), (5, 9, 100), (6, 5, 40)])
@pytest.mark.parametrize("cin,cout", [(16, 16), (16, 32), (32, 16), (32, 32), (32, 64), (64, 32)])
def test_conv3d_forward_and_weight_gradient_exact(ctx, cin, cout, H, W, D):
    """Up to 32 channels run the LDS-tiled kernel, whose tile along the
    lines is 16 ceil(D / 16) nodes up to 80 (64 with 32 input channels), else
    64: lines of 40 nodes one 48-node tile, of 70 one 80-node tile (two 64-node
    tiles with 32 input channels), of 100 a 64-node tile and a partial one;
    9 lines two full 4-line tiles and a partial one.  64-channel layers run
    one line per workgroup."""
    rng = np.random.default_rng(300 + cin + cout + D)
    x = ints(rng, (H, W, D, cin), -2, 2)
    w = ints(rng, (27, cout, cin), -2, 2)
    y = ctx.conv_raw(x, w)
    ref = cn.conv(x.astype(np.float64), w.astype(np.float64))
    assert np.array_equal(y.astype(np.float64), ref), float(np.max(np.abs(y - ref)))
    dz = ints(rng, (H, W, D, cout), -2, 2)
    g = ctx.conv_wgrad_raw(x, dz)
    _, gref = cn.conv_grads(x.astype(np.float64), dz.astype(np.float64), np.zeros((27, cout, cin)))
    assert np.array_equal(g.astype(np.float64), gref), float(np.max(np.abs(g - gref)))


def test_conv_raw_rejects_unsupported_channels(ctx):
    import pansfem2_amd as pa
    with pytest.raises(pa.PfError):
        ctx.conv_raw(np.zeros((4, 4, 8), np.float32), np.zeros((9, 16, 8), np.float32))


@pytest.mark.parametrize("shape", [(1, 1), (40, 3), (1, 5000), (4097, 1), (300, 17), (1, 1, 37), (30, 2, 3), (3, 40, 1),
                                   (20, 20, 20)])
@pytest.mark.parametrize("cin,cout", [(16, 16), (16, 32), (32, 16), (32, 32), (64, 32)])
def test_conv_weight_gradient_line_edges_exact(ctx, cin, cout, shape):
    """Lines shorter than a 16-pixel chunk (a lane's pixel crosses several
    lines, in 3D several planes, from one chunk to the next), one line of more
    than a block of 4096 pixels, and blocks that end inside a chunk."""
    rng = np.random.default_rng(400 + cin + cout + shape[0])
    x = ints(rng, shape + (cin,), -2, 2)
    dz = ints(rng, shape + (cout,), -2, 2)
    g = ctx.conv_wgrad_raw(x, dz)
    _, ref = cn.conv_grads(x.astype(np.float64), dz.astype(np.float64), np.zeros((3 ** len(shape), cout, cin)))
    assert np.sum(np.abs(x)) * 2 < 2 ** 24
    assert np.array_equal(g.astype(np.float64), ref), float(np.max(np.abs(g - ref)))
