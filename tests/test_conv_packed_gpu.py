"""Convolutions on operands packed to fp16 (conv_packed.hip) at the edges of
their tiles, against the oracle: pixel counts around the 64-, 128- and 256-pixel
tiles and the 64-pixel dW slices, channel and filter counts around the 32- and
64-channel blocks, strides that leave residues without taps, padding beyond the
kernel, and infinities, which must not leave the outputs they belong to."""
import zlib

import numpy as np
import pytest

import oracle
from ml_framework_amd import capi
from oracle import fp16r
from tests.helpers import _dev, _out, assert_parity, hip_conv_bwd, hip_conv_fwd, hip_convT_bwd, hip_convT_fwd, out_hw

pytestmark = pytest.mark.gpu
S = oracle.seera_cpp
# fp32 sums of the same fp16 products in another order. Each addition rounds the
# partial sum by 0.41 * 2^-24 of it (root mean square); over a chain of n terms of
# random sign the partial sums grow with the square root of their length, so the
# result is off by about 0.41 * 2^-24 * sqrt(n / 2): 3.9e-6 at the 50 thousand
# terms of the longest dW here. The oracle's chain may be off as much: 5.5e-6
# together, stated with less than a factor of two. (A term lost or read twice
# shows in test_exact.)
STRICT = 1e-5


@pytest.fixture(autouse=True, scope="module")
def _gpu():
    assert capi.gpu_available(), "no HIP device visible"


# name, N, C, H, W, F, KH, KW, stride, pad
CASES = [
    ("one_pixel", 1, 33, 1, 1, 5, 1, 1, 1, 0),
    ("px63", 7, 32, 3, 3, 64, 3, 3, 1, 1),       # 63 pixels
    ("px64_c64", 1, 64, 8, 8, 65, 3, 3, 1, 1),   # one tile, one filter past 64
    ("px65", 13, 65, 5, 1, 33, 3, 3, 1, 1),
    ("px257", 1, 40, 257, 1, 130, 3, 1, 1, 1),
    ("image_below_slice", 70, 31, 2, 3, 96, 3, 3, 1, 1),  # 11 images per 64-pixel slice
    ("c96", 3, 96, 7, 9, 96, 3, 3, 1, 1),        # 32-channel blocks, 3 of them
    ("c128_f192", 2, 128, 14, 14, 192, 3, 3, 1, 1),
    ("s2_odd", 3, 64, 13, 11, 72, 3, 3, 2, 1),
    ("s2_1x1", 2, 64, 14, 14, 128, 1, 1, 2, 0),  # residues without taps: zero dX
    ("s3_2x2", 2, 34, 11, 10, 40, 2, 2, 3, 0),   # stride beyond the kernel
    ("s3_3x3", 1, 16, 16, 17, 20, 3, 3, 3, 2),
    ("pad_beyond", 2, 24, 6, 5, 24, 2, 2, 1, 3), # windows wholly in the padding
    ("k5", 2, 20, 9, 10, 24, 5, 5, 1, 2),
    ("k8", 1, 8, 12, 13, 9, 8, 8, 1, 3),         # 64 taps, the most it takes
    # first layers in space-to-depth form: odd images and paddings, 1 to 4
    # channels, kernels of odd and even size, filters around 64
    ("stem_odd", 2, 3, 31, 29, 33, 7, 7, 2, 3),
    ("stem_c1", 3, 1, 24, 28, 64, 7, 7, 2, 3),
    ("stem_c4_k8", 2, 4, 22, 25, 65, 8, 8, 2, 3),
    ("stem_nopad", 1, 2, 20, 23, 8, 7, 7, 2, 0),
    ("stem_5x7", 2, 3, 17, 20, 40, 5, 7, 2, 2),
    ("stem_tiles", 6, 3, 112, 112, 64, 7, 7, 2, 3),
    ("rows_1xk", 2, 36, 4, 30, 36, 1, 7, 1, 3),
    ("tiles_128", 20, 32, 30, 30, 128, 3, 3, 1, 1),   # 64 x 128 tiles in 32-deep slices
    ("tiles_256", 25, 32, 31, 31, 200, 3, 3, 1, 1),   # 256 x 128 tiles in 32-deep slices
    ("dw_splits", 40, 64, 30, 30, 64, 3, 3, 1, 1),    # 128 x 64 tiles; 64 x 128 dW tiles, many splits
]

# Every tile (pixels x channels) in 64- and 32-deep slices, forward and dX, with
# pixels and channels that are no multiple of it.
TILE_CASES = [
    ("bk64_64x128", 8, 190, 29, 31, 190, 3, 3, 1, 1),
    ("bk64_128x128", 17, 190, 29, 31, 190, 3, 3, 1, 1),
    ("bk64_256x128", 34, 190, 29, 31, 190, 2, 2, 1, 1),
    ("bk32_64x128", 8, 150, 29, 31, 150, 3, 3, 1, 1),
    ("bk32_128x128", 17, 150, 29, 31, 150, 3, 3, 1, 1),
    ("bk32_256x128", 34, 150, 29, 31, 150, 2, 2, 1, 1),
    ("s2_256x128", 33, 130, 29, 31, 64, 3, 3, 2, 1),   # dX in four residues of 15 x 16 to 14 x 15
    ("bk64_128x64", 37, 60, 29, 31, 62, 3, 3, 1, 1),
    ("bk32_128x64", 37, 30, 29, 31, 28, 3, 3, 1, 1),
]


def _data(name, N, C, H, W, F, KH, KW, s, p):
    r = np.random.default_rng(zlib.crc32(name.encode()))
    x = r.standard_normal((N, C, H, W)).astype(np.float32)
    w = (r.standard_normal((F, C, KH, KW)) / np.sqrt(C * KH * KW)).astype(np.float32)
    OH, OW = out_hw(H, W, KH, KW, s, p)
    return x, w, r.standard_normal((N, F, OH, OW)).astype(np.float32)


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_conv2d(case):
    name, *shape = case
    x, w, dy = _data(name, *shape)
    s, p = shape[-2:]
    assert_parity(hip_conv_fwd(x, w, s, p), S.conv2d_forward(fp16r(x), fp16r(w), s, s, p, p), name, STRICT)
    dx, dw = hip_conv_bwd(dy, x, w, s, p)
    rdx, rdw = S.conv2d_backward(fp16r(dy), fp16r(x), fp16r(w), s, s, p, p)
    assert_parity(dx, rdx, name + " dX", STRICT)
    assert_parity(dw, rdw, name + " dW", STRICT, mabs=2e-2 * max(1.0, float(np.abs(rdw).max()) / 100))


@pytest.mark.parametrize("case", CASES + TILE_CASES, ids=[c[0] for c in CASES + TILE_CASES])
def test_exact(case):
    """Small whole numbers: every product and partial sum (below 2^24) is exact
    in fp16 and fp32, so the results are the oracle's bits."""
    name, N, C, H, W, F, KH, KW, s, p = case
    r = np.random.default_rng(zlib.crc32(name.encode()))
    OH, OW = out_hw(H, W, KH, KW, s, p)
    x, w, dy, b = (r.integers(-2, 3, sh).astype(np.float32) for sh in ((N, C, H, W), (F, C, KH, KW), (N, F, OH, OW), (F,)))
    y = S.conv2d_forward(x, w, s, s, p, p)
    np.testing.assert_array_equal(hip_conv_fwd(x, w, s, p), y)
    rdx, rdw = S.conv2d_backward(dy, x, w, s, s, p, p)
    with _dev(x) as px, _dev(w) as pw, _dev(b) as pb, _dev(dy) as pdy, _out(dy.shape) as py, _out(dy.shape) as pm, \
            _out(x.shape) as pdx, _out(w.shape) as pdw, _out((F,)) as pdb:
        capi.call("seera_hip_conv2d_fwd_bias_act", px.ptr, pw.ptr, pb.ptr, py.ptr, pm.ptr, N, C, H, W, F, KH, KW,
                  p, p, s, s, capi.SEERA_ACT_RELU)
        capi.call("seera_hip_conv2d_bwd_bias", pw.ptr, px.ptr, pdy.ptr, pdx.ptr, pdw.ptr, pdb.ptr, N, C, H, W, F,
                  KH, KW, s, s, p, p)
        y += b[None, :, None, None]
        np.testing.assert_array_equal(py.to_array(y.shape), np.maximum(y, 0))
        np.testing.assert_array_equal(pm.to_array(y.shape), (y > 0).astype(np.float32))
        np.testing.assert_array_equal(pdx.to_array(x.shape), rdx)
        np.testing.assert_array_equal(pdw.to_array(w.shape), rdw)
        np.testing.assert_array_equal(pdb.to_array((F,)), dy.sum((0, 2, 3)))


@pytest.mark.parametrize("case", [c for c in CASES if c[0] in ("px65", "c96", "s2_odd", "tiles_256", "one_pixel", "stem_odd", "stem_c4_k8")],
                         ids=lambda c: c[0])
def test_conv2d_bias_relu_and_bias_grad(case):
    name, N, C, H, W, F, KH, KW, s, p = case
    x, w, dy = _data(*case)
    b = np.random.default_rng(3).standard_normal(F).astype(np.float32)
    with _dev(x) as px, _dev(w) as pw, _dev(b) as pb, _dev(dy) as pdy, _out(dy.shape) as py, _out(dy.shape) as pm, \
            _out(x.shape) as pdx, _out(w.shape) as pdw, _out((F,)) as pdb:
        capi.call("seera_hip_conv2d_fwd_bias_act", px.ptr, pw.ptr, pb.ptr, py.ptr, pm.ptr, N, C, H, W, F, KH, KW,
                  p, p, s, s, capi.SEERA_ACT_RELU)
        capi.call("seera_hip_conv2d_bwd_bias", pw.ptr, px.ptr, pdy.ptr, pdx.ptr, pdw.ptr, pdb.ptr, N, C, H, W, F,
                  KH, KW, s, s, p, p)
        y, m, dx, dw, db = (q.to_array(sh) for q, sh in ((py, dy.shape), (pm, dy.shape), (pdx, x.shape),
                                                        (pdw, w.shape), (pdb, (F,))))
    # the unfused calls' bits
    pre = hip_conv_fwd(x, w, s, p) + b[None, :, None, None]
    np.testing.assert_array_equal(y, np.where(pre > 0, pre, 0))
    np.testing.assert_array_equal(m, (pre > 0).astype(np.float32))
    dx0, dw0 = hip_conv_bwd(dy, x, w, s, p)
    np.testing.assert_array_equal(dx, dx0)
    np.testing.assert_array_equal(dw, dw0)
    assert_parity(db, dy.astype(np.float64).sum((0, 2, 3)), name + " db", STRICT)


@pytest.mark.parametrize("shape", [(3, 40, 5, 7, 24, 4, 4, 2, 1), (2, 64, 9, 8, 33, 3, 3, 2, 1), (5, 100, 1, 1, 64, 4, 4, 1, 0),
                                   (2, 48, 6, 6, 32, 2, 2, 2, 0), (2, 33, 5, 5, 40, 3, 3, 1, 1), (1, 16, 4, 5, 16, 3, 3, 3, 0)],
                         ids=str)
def test_conv_transpose(shape):
    N, Cin, H, W, Cout, KH, KW, s, p = shape
    r = np.random.default_rng(11)
    x = r.standard_normal((N, Cin, H, W)).astype(np.float32)
    w = (r.standard_normal((Cin, Cout, KH, KW)) / np.sqrt(Cin * KH * KW)).astype(np.float32)
    y = hip_convT_fwd(x, w, s, p)
    assert_parity(y, S.conv_transpose2d_forward(fp16r(x), fp16r(w), s, s, p, p), "convT", STRICT)
    dy = r.standard_normal(y.shape).astype(np.float32)
    dx, dw = hip_convT_bwd(dy, x, w, s, p)
    rdx, rdw = S.conv_transpose2d_backward(fp16r(dy), fp16r(x), fp16r(w), s, s, p, p)
    assert_parity(dx, rdx, "convT dX", STRICT)
    assert_parity(dw, rdw, "convT dW", STRICT)


def test_infinities_stay_where_they_belong():
    """An infinite input or gradient reaches exactly the outputs that it is a
    term of: no zero-weighted or padding term touches it."""
    N, C, H, W, F = 2, 40, 7, 9, 48
    x, w, dy = _data("inf", N, C, H, W, F, 3, 3, 1, 1)
    x[0, 3, 0, 8] = np.inf
    dy[1, 7, 6, 0] = np.inf
    y = hip_conv_fwd(x, w, 1, 1)
    hit = np.zeros(y.shape, bool)
    hit[0, :, 0:2, 7:9] = True
    np.testing.assert_array_equal(np.isfinite(y), ~hit)
    dx, dw = hip_conv_bwd(dy, x, w, 1, 1)
    hit = np.zeros(dx.shape, bool)
    hit[1, :, 5:7, 0:2] = True
    np.testing.assert_array_equal(np.isfinite(dx), ~hit)
    # dW: channel 3 through the infinite pixel's taps, filter 7 through dY's
    hit = np.zeros(dw.shape, bool)
    hit[:, 3, 0:2, 1:3] = True
    hit[7] = True
    assert np.all(np.isfinite(dw[~hit]))


@pytest.mark.parametrize("N,C,H,W,F,KH,KW,p", [(2, 3, 31, 29, 33, 7, 7, 3), (1, 4, 22, 24, 130, 7, 7, 2), (3, 1, 18, 26, 70, 5, 7, 2),
                                               (2, 2, 24, 28, 64, 8, 8, 3), (20, 3, 64, 62, 40, 7, 7, 3)], ids=str)
def test_first_layer_infinities_stay_where_they_belong(N, C, H, W, F, KH, KW, p):
    """The space-to-depth form multiplies real values by the zero weights of the
    taps that it adds: an infinite one must reach the outputs that it is a term
    of and leave the others, rows and columns beside them included, as they are."""
    x, w, dy = _data(f"stem{N}{F}", N, C, H, W, F, KH, KW, 2, p)
    b = np.random.default_rng(7).standard_normal(F).astype(np.float32)
    OH, OW = dy.shape[2:]
    spots = [(0, 0, 0, 0), (N - 1, C - 1, H - 1, W - 1), (0, C - 1, H // 2, W // 2 + 1)]
    hit = np.zeros(dy.shape, bool)
    for n, c, h, v in spots:
        x[n, c, h, v] = np.inf
        for r in range(KH):
            for q in range(KW):
                i, j = h + p - r, v + p - q
                if i % 2 == 0 and j % 2 == 0 and 0 <= i // 2 < OH and 0 <= j // 2 < OW:
                    hit[n, :, i // 2, j // 2] = True
    with _dev(x) as px, _dev(w) as pw, _dev(b) as pb, _out(dy.shape) as py:
        capi.call("seera_hip_conv2d_fwd_bias_act", px.ptr, pw.ptr, pb.ptr, py.ptr, 0, N, C, H, W, F, KH, KW, p, p, 2, 2, 0)
        y = py.to_array(dy.shape)
    np.testing.assert_array_equal(np.isfinite(y), ~hit)
    x[~np.isfinite(x)] = 0
    want = S.conv2d_forward(fp16r(x), fp16r(w), 2, 2, p, p) + b[None, :, None, None]
    assert_parity(y[~hit], want[~hit], "fwd", STRICT)

    hit = np.zeros(x.shape, bool)
    for n, f, i, j in [(0, 1, 0, 0), (N - 1, F - 1, OH - 1, OW - 1), (0, F // 2, OH // 2, OW // 2)]:
        dy[n, f, i, j] = -np.inf
        for r in range(KH):
            for q in range(KW):
                h, v = 2 * i - p + r, 2 * j - p + q
                if 0 <= h < H and 0 <= v < W:
                    hit[n, :, h, v] = True
    dx, dw = hip_conv_bwd(dy, x, w, 2, p)
    np.testing.assert_array_equal(np.isfinite(dx), ~hit)
    bad = ~np.isfinite(dy).all((0, 2, 3))
    assert np.isfinite(dw[~bad]).all()
    dy[~np.isfinite(dy)] = 0
    rdx, rdw = S.conv2d_backward(fp16r(dy), fp16r(x), fp16r(w), 2, 2, p, p)
    assert_parity(dx[~hit], rdx[~hit], "dX", STRICT)
    assert_parity(dw[~bad], rdw[~bad], "dW", STRICT)
