"""Layers at the sizes from which the dispatch leaves packed operands for the
kernels that read fp32 rows (conv_routes.h): channel slices on many full rows, few
filters over an input that fills the cache. Whole-number operands, so every
product and partial sum (below 2^24) is exact and the results are the oracle's bits."""
import numpy as np
import pytest

import oracle
from ml_framework_amd import capi
from tests.helpers import _dev, _out, hip_conv_bwd, out_hw

pytestmark = pytest.mark.gpu
S = oracle.seera_cpp


@pytest.fixture(autouse=True, scope="module")
def _gpu():
    assert capi.gpu_available(), "no HIP device visible"


@pytest.mark.parametrize("N,C,H,W,F,K,s,p,backward", [
    (32, 128, 56, 56, 24, 3, 1, 1, False),    # two slices, one filter tile
    (13, 192, 56, 224, 10, 3, 1, 1, False),   # three slices, column tiles
    (62, 256, 56, 56, 8, 3, 1, 1, False),     # four
    (64, 128, 56, 56, 128, 3, 1, 1, False),   # two slices x two filter tiles
    (32, 128, 56, 56, 128, 3, 1, 1, True),    # and the two-pass backward
    (60, 64, 112, 112, 16, 3, 2, 1, False),   # 3x3, 2x2 and 1x1 at stride 2
    (13, 64, 224, 224, 12, 2, 2, 0, False),
    (50, 64, 112, 112, 20, 1, 2, 0, False),
    (8, 3, 224, 224, 16, 3, 2, 1, False),     # few channels
    (6, 24, 56, 56, 96, 4, 2, 1, True),       # 4x4 at stride 2, few rows of 48 and more
    (8, 256, 56, 56, 32, 3, 1, 1, True),      # few pixels of many channels: the backward on rows
], ids=str)
def test_exact(N, C, H, W, F, K, s, p, backward):
    r = np.random.default_rng(N + F)
    OH, OW = out_hw(H, W, K, K, s, p)
    x, w, b, dy = (r.integers(-2, 3, sh, dtype=np.int8).astype(np.float32)
                   for sh in ((N, C, H, W), (F, C, K, K), (F,), (N, F, OH, OW)))
    if backward:
        dx, dw = hip_conv_bwd(dy, x, w, s, p)
        rdx, rdw = S.conv2d_backward(dy, x, w, s, s, p, p)
        np.testing.assert_array_equal(dx, rdx)
        np.testing.assert_array_equal(dw, rdw)
        return
    pre = S.conv2d_forward(x, w, s, s, p, p) + b[None, :, None, None]
    with _dev(x) as px, _dev(w) as pw, _dev(b) as pb, _out(dy.shape) as py, _out(dy.shape) as pm:
        capi.call("seera_hip_conv2d_fwd_bias_act", px.ptr, pw.ptr, pb.ptr, py.ptr, pm.ptr, N, C, H, W, F, K, K, p, p, s, s,
                  capi.SEERA_ACT_RELU)
        np.testing.assert_array_equal(py.to_array(dy.shape), np.maximum(pre, 0))
        np.testing.assert_array_equal(pm.to_array(dy.shape), (pre > 0).astype(np.float32))
