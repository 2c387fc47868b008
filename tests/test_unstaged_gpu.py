"""Calls whose operands would be packed to fp16 or widened, on a stream that has
no memory for the copies: captured before any call of their size, so the staging
buffer cannot grow, they run on the kernels that read the caller's tensors
(gather GEMMs and, on aligned rows, the band and channel-slice kernels for
convolutions; scalar-load tiles for products). Each graph is
replayed with other work between the replays, and every replay is compared with
the oracle; a call made outside capture afterwards takes the copies and must
agree within the order of its sums."""
import ctypes

import numpy as np
import pytest

import oracle
from ml_framework_amd import capi
from ml_framework_amd.capi import DeviceBuffer
from oracle import fp16r
from tests.helpers import assert_parity, convT_hw, hip_conv_bwd, hip_conv_fwd, out_hw

pytestmark = pytest.mark.gpu
S = oracle.seera_cpp
# fp32 sums of at most 2304 of the same fp16 products in two orders:
# 2 * 0.41 * 2^-24 * sqrt(2304 / 2) = 1.7e-6 of the result (see test_conv_packed_gpu.py)
STRICT = 5e-6


@pytest.fixture(scope="module")
def lib():
    assert capi.gpu_available(), "no HIP device visible"
    return capi.load()


def _held(lib):
    held = ctypes.c_size_t()
    capi.check(lib.seera_hip_workspace_stats(ctypes.byref(held), None))
    return held.value


def _unstaged(lib, calls, outputs):
    """calls: [(entry point, arguments without the stream)]; outputs: [(buffer,
    shape, expected)]. Captures the calls on a fresh stream whose workspace, but
    not its staging buffer, has grown, and checks three replays and a call
    outside capture."""
    st, g = ctypes.c_void_p(), ctypes.c_void_p()
    capi.check(lib.seera_hip_stream_create(ctypes.byref(st)))
    r = np.random.default_rng(1)
    m, k = 256, 8192  # a split product: several MB of partial sums
    warm = [DeviceBuffer.from_array(r.uniform(-1, 1, s).astype(np.float32)) for s in ((m, k), (k, m))]
    scratch = DeviceBuffer(m * m * 4)

    def check(what):
        for i, (buf, shape, want) in enumerate(outputs):
            got = buf.to_array(shape)
            assert_parity(got, want, f"{what}, output {i}", STRICT, 1e-2 * max(1.0, float(np.abs(want).max())))
            buf.fill(0x7F)

    try:
        capi.check(lib.seera_hip_matmul_async(warm[0].ptr, warm[1].ptr, scratch.ptr, m, m, k, 1, st.value))
        capi.check(lib.seera_hip_stream_synchronize(st.value))
        held = _held(lib)
        capi.check(lib.seera_hip_graph_capture_begin(st.value))
        status = [getattr(lib, name)(*args, st.value) for name, args in calls]
        capi.check(lib.seera_hip_graph_capture_end(st.value, ctypes.byref(g)))
        for s in status:
            capi.check(s)
        assert _held(lib) == held, "memory was allocated under capture"
        for rep in range(3):
            capi.check(lib.seera_hip_graph_launch(g.value, st.value))
            capi.check(lib.seera_hip_stream_synchronize(st.value))
            check(f"replay {rep}")
            capi.check(lib.seera_hip_matmul_async(warm[0].ptr, warm[1].ptr, scratch.ptr, m, m, k, 1, st.value))
            capi.check(lib.seera_hip_synchronize())
        for name, args in calls:
            capi.check(getattr(lib, name)(*args, st.value))
        capi.check(lib.seera_hip_stream_synchronize(st.value))
        assert _held(lib) > held, "the call outside capture takes no copies: this test has lost its subject"
        check("outside capture")
    finally:
        if g.value:
            capi.check(lib.seera_hip_graph_destroy(g.value))
        lib.seera_hip_stream_destroy(st.value)


def _dev(a):
    return DeviceBuffer.from_array(np.ascontiguousarray(a, np.float32))


@pytest.mark.parametrize("N,C,H,W,F,K,s,p", [
    (2, 24, 11, 13, 40, 3, 1, 1),    # rows that are not whole float4s
    (3, 64, 7, 7, 96, 3, 1, 1),
    (2, 16, 13, 15, 70, 3, 2, 1),    # stride 2
    (2, 20, 9, 10, 24, 5, 1, 2),     # 25 taps
    (2, 3, 30, 26, 33, 7, 2, 3),     # a first layer
    (2, 128, 12, 16, 64, 3, 1, 1),   # two 64-channel slices, the epilogue on their total
    (1, 192, 6, 60, 64, 3, 1, 1),    # three, column tiles
    (1, 256, 5, 20, 64, 3, 1, 1),    # four
    (1, 128, 6, 60, 96, 3, 1, 1),    # two slices x two filter tiles (the second partial)
    (1, 128, 4, 64, 128, 3, 1, 1),
    (2, 96, 10, 12, 40, 3, 2, 1),    # band kernels, aligned: stride 2
], ids=str)
def test_conv2d(lib, N, C, H, W, F, K, s, p):
    r = np.random.default_rng(N + C + H)
    OH, OW = out_hw(H, W, K, K, s, p)
    x, b, dy = (r.standard_normal(sh).astype(np.float32) for sh in ((N, C, H, W), (F,), (N, F, OH, OW)))
    w = (r.standard_normal((F, C, K, K)) / np.sqrt(C * K * K)).astype(np.float32)
    pre = S.conv2d_forward(fp16r(x), fp16r(w), s, s, p, p) + b[None, :, None, None]
    dx, dw = S.conv2d_backward(fp16r(dy), fp16r(x), fp16r(w), s, s, p, p)
    px, pw, pb, pdy = (_dev(a) for a in (x, w, b, dy))
    py, pdx, pdw, pdb = (DeviceBuffer(a.size * 4) for a in (dy, x, w, b))
    _unstaged(lib, [("seera_hip_conv2d_fwd_bias_act_async", (px.ptr, pw.ptr, pb.ptr, py.ptr, 0, N, C, H, W, F, K, K, p, p, s, s,
                                                              capi.SEERA_ACT_RELU)),
                    ("seera_hip_conv2d_bwd_bias_async", (pw.ptr, px.ptr, pdy.ptr, pdx.ptr, pdw.ptr, pdb.ptr, N, C, H, W, F, K, K,
                                                         s, s, p, p))],
              [(py, dy.shape, np.maximum(pre, 0)), (pdx, x.shape, dx), (pdw, w.shape, dw),
               (pdb, (F,), dy.astype(np.float64).sum((0, 2, 3)))])


@pytest.mark.parametrize("N,Ci,H,W,Co,K,s,p", [(2, 48, 7, 9, 24, 4, 2, 1), (3, 33, 5, 6, 40, 3, 1, 1)], ids=str)
def test_conv_transpose(lib, N, Ci, H, W, Co, K, s, p):
    r = np.random.default_rng(N + Ci)
    OH, OW = convT_hw(H, W, K, K, s, p)
    x, dy = (r.standard_normal(sh).astype(np.float32) for sh in ((N, Ci, H, W), (N, Co, OH, OW)))
    w = (r.standard_normal((Ci, Co, K, K)) / np.sqrt(Ci * K * K)).astype(np.float32)
    y = S.conv_transpose2d_forward(fp16r(x), fp16r(w), s, s, p, p)
    dx, dw = S.conv_transpose2d_backward(fp16r(dy), fp16r(x), fp16r(w), s, s, p, p)
    px, pw, pdy = (_dev(a) for a in (x, w, dy))
    py, pdx, pdw = (DeviceBuffer(a.size * 4) for a in (dy, x, w))
    _unstaged(lib, [("seera_hip_conv2DTranpose_fwd_async", (px.ptr, pw.ptr, py.ptr, N, Ci, H, W, Co, K, K, s, s, p, p)),
                    ("seera_hip_conv2DTranspose_bwd_async", (pw.ptr, px.ptr, pdy.ptr, pdx.ptr, pdw.ptr, N, Ci, H, W, Co, K, K,
                                                             s, s, p, p))],
              [(py, dy.shape, y), (pdx, x.shape, dx), (pdw, w.shape, dw)])


@pytest.mark.parametrize("M,K,N", [(333, 515, 257), (1300, 1300, 1300)])
def test_matmul(lib, M, K, N):
    r = np.random.default_rng(M)
    a, b, dc = (r.uniform(-1, 1, s).astype(np.float32) for s in ((M, K), (K, N), (M, N)))
    c = S.matmul_batched(fp16r(a)[None], fp16r(b))[0]
    da, db = S.matmul_bwd(fp16r(a)[None], fp16r(b), fp16r(dc)[None])
    pa, pb, pdc = (_dev(v) for v in (a, b, dc))
    pc, pda, pdb = (DeviceBuffer(v.size * 4) for v in (dc, a, b))
    _unstaged(lib, [("seera_hip_matmul_async", (pa.ptr, pb.ptr, pc.ptr, M, N, K, 1)),
                    ("seera_hip_matmul_bwd_async", (pa.ptr, pb.ptr, pdc.ptr, pda.ptr, pdb.ptr, M, N, K, 1))],
              [(pc, (M, N), c), (pda, (M, K), da[0]), (pdb, (K, N), db)])


@pytest.mark.parametrize("N,C,H,W,F,K,s,p", [
    (2, 24, 22, 30, 40, 3, 4, 1),    # 16 stride residues, rows widened to float4s for the forward and dW
    (1, 16, 33, 41, 24, 5, 5, 2),    # 25 of them
    (2, 6, 14, 15, 10, 9, 1, 4),     # 81 taps
    (1, 12, 15, 20, 18, 9, 2, 4),
], ids=str)
def test_beyond_packed_sizes(lib, N, C, H, W, F, K, s, p):
    """Strides and kernels that the packed convolutions do not hold (more than 9
    residues, more than 64 taps)."""
    r = np.random.default_rng(N + C + H)
    x = r.standard_normal((N, C, H, W)).astype(np.float32)
    w = (r.standard_normal((F, C, K, K)) / np.sqrt(C * K * K)).astype(np.float32)
    y = S.conv2d_forward(fp16r(x), fp16r(w), s, s, p, p)
    assert_parity(hip_conv_fwd(x, w, s, p), y, "fwd", STRICT)
    dy = r.standard_normal(y.shape).astype(np.float32)
    dx, dw = hip_conv_bwd(dy, x, w, s, p)
    rdx, rdw = S.conv2d_backward(fp16r(dy), fp16r(x), fp16r(w), s, s, p, p)
    assert_parity(dx, rdx, "dX", STRICT)
    assert_parity(dw, rdw, "dW", STRICT)
