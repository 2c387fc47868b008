"""1x1 stride-1 convolutions in one pass over memory (conv_pointwise.hip): image
sizes around the 128-pixel tiles, channels and filters around their 64s and 32s,
every channel count class of the backward, more tiles than blocks. The operands
are small whole numbers, so every product and partial sum is exact in fp16 and
fp32 and the results must equal the integer ones."""
import numpy as np
import pytest

from ml_framework_amd import capi
from tests.helpers import _dev, _out, hip_conv_bwd, hip_conv_fwd

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True, scope="module")
def _gpu():
    assert capi.gpu_available(), "no HIP device visible"


# N, C, H, W, F
CASES = [
    (1, 1, 2, 2, 1),
    (3, 64, 1, 4, 64),
    (2, 33, 4, 31, 31),       # 124 pixels
    (2, 64, 8, 16, 32),       # one tile an image
    (3, 63, 12, 11, 33),      # 132 pixels: a tile of four
    (2, 65, 16, 24, 64),      # two slices, three tiles
    (600, 40, 8, 8, 24),      # more images than blocks
    (40, 128, 28, 28, 57),    # two slices, 280 tiles
    (120, 130, 28, 28, 64),   # three slices, 840 tiles
    (210, 256, 20, 21, 48),   # four
    (810, 257, 8, 12, 40),    # five
    (410, 384, 12, 12, 16),   # six
    (810, 448, 8, 8, 8),      # seven
    (205, 505, 20, 20, 64),   # eight
    (110, 192, 28, 28, 80),   # four filter tiles forward
    (50, 64, 56, 56, 128),
]


def _ints(r, shape):
    return r.integers(-2, 3, shape).astype(np.float32)  # sums of 2^22 products stay below 2^24


@pytest.mark.parametrize("N,C,H,W,F", CASES)
def test_exact(N, C, H, W, F):
    r = np.random.default_rng(N + C + F)
    x, dy, w = _ints(r, (N, C, H * W)), _ints(r, (N, F, H * W)), _ints(r, (F, C))
    y = np.matmul(w, x)  # exact in fp32 as well
    np.testing.assert_array_equal(hip_conv_fwd(x.reshape(N, C, H, W), w.reshape(F, C, 1, 1), 1, 0).reshape(y.shape), y)
    dx, dw = hip_conv_bwd(dy.reshape(N, F, H, W), x.reshape(N, C, H, W), w.reshape(F, C, 1, 1), 1, 0)
    np.testing.assert_array_equal(dx.reshape(x.shape), np.matmul(w.T, dy))
    want = np.matmul(dy, x.transpose(0, 2, 1)).sum(0)
    np.testing.assert_array_equal(dw.reshape(F, C), want)

    b = _ints(r, (F,))
    with _dev(x) as px, _dev(w) as pw, _dev(b) as pb, _dev(dy) as pdy, _out(dy.shape) as py, _out(dy.shape) as pm, \
            _out(x.shape) as pdx, _out(w.shape) as pdw, _out((F,)) as pdb:
        capi.call("seera_hip_conv2d_fwd_bias_act", px.ptr, pw.ptr, pb.ptr, py.ptr, pm.ptr, N, C, H, W, F, 1, 1, 0, 0, 1,
                  1, capi.SEERA_ACT_RELU)
        pre = y + b[:, None]
        np.testing.assert_array_equal(py.to_array(y.shape), np.maximum(pre, 0))
        np.testing.assert_array_equal(pm.to_array(y.shape), (pre > 0).astype(np.float32))
        capi.call("seera_hip_conv2d_bwd_bias", pw.ptr, px.ptr, pdy.ptr, pdx.ptr, pdw.ptr, pdb.ptr, N, C, H, W, F, 1, 1,
                  1, 1, 0, 0)
        np.testing.assert_array_equal(pdw.to_array((F, C)), want)
        np.testing.assert_array_equal(pdb.to_array((F,)), dy.sum((0, 2)))


def test_not_finite():
    """Infinities and NaN stay in the outputs that use them."""
    r = np.random.default_rng(3)
    N, C, H, W, F = 2, 40, 6, 22, 24
    x, dy, w = (_ints(r, s) + 3 for s in ((N, C, H * W), (N, F, H * W), (F, C)))
    x[1, -1, -1], dy[0, -1, -1] = np.inf, np.nan
    y = hip_conv_fwd(x.reshape(N, C, H, W), w.reshape(F, C, 1, 1), 1, 0).reshape(N, F, H * W)
    want = np.zeros(y.shape, bool)
    want[1, :, -1] = True
    np.testing.assert_array_equal(~np.isfinite(y), want)
    dx, dw = hip_conv_bwd(dy.reshape(N, F, H, W), x.reshape(N, C, H, W), w.reshape(F, C, 1, 1), 1, 0)
    want = np.zeros((N, C, H * W), bool)
    want[0, :, -1] = True
    np.testing.assert_array_equal(~np.isfinite(dx.reshape(want.shape)), want)
    want = np.zeros((F, C), bool)
    want[-1], want[:, -1] = True, True
    np.testing.assert_array_equal(~np.isfinite(dw.reshape(F, C)), want)
