"""GEMMs with few tiles and a long contraction on 128x128 tiles split over K
(plan.h): tile and split remainders, the bias gradient's column sums, and the
plan's fallback where the scratch is not to be had, against the oracle."""
import ctypes

import numpy as np
import pytest

import oracle
from ml_framework_amd import capi
from ml_framework_amd.capi import DeviceBuffer
from oracle import fp16r
from tests.helpers import _dev, _out, assert_parity, hip_matmul, hip_matmul_bwd

pytestmark = pytest.mark.gpu
S = oracle.seera_cpp
STRICT = 1e-5  # fp32 sums of the same fp16 products in another order


@pytest.fixture(autouse=True, scope="module")
def _gpu():
    assert capi.gpu_available(), "no HIP device visible"


# (M, K, N, Nbatch): the forward splits at K 4096, dB where Nbatch * M is long
@pytest.mark.parametrize("M,K,N,nb", [(512, 4096, 512, 1), (500, 4160, 388, 1), (512, 512, 512, 16),
                                      (4096, 388, 516, 1), (1024, 1024, 1024, 8)])
def test_parity(M, K, N, nb):
    r = np.random.default_rng(M + K)
    a = r.uniform(-1, 1, (nb, M, K)).astype(np.float32)
    b = r.uniform(-1, 1, (K, N)).astype(np.float32)
    dc = r.uniform(-1, 1, (nb, M, N)).astype(np.float32)
    big = 2e-2 * max(1.0, nb * M / 1000)  # the entries of dB grow with the rows
    assert_parity(hip_matmul(a, b), S.matmul_batched(fp16r(a), fp16r(b)), "C", STRICT, big)
    da, db = hip_matmul_bwd(a, b, dc)
    rda, rdb = S.matmul_bwd(fp16r(a), fp16r(b), fp16r(dc))
    assert_parity(da, rda, "dA", STRICT, big)
    assert_parity(db, rdb, "dB", STRICT, big)


def test_column_sums_and_epilogue():
    M, K, N = 8192, 384, 448
    r = np.random.default_rng(4)
    a = r.uniform(-1, 1, (M, K)).astype(np.float32)
    b = r.uniform(-1, 1, (K, N)).astype(np.float32)
    dc = r.uniform(-1, 1, (M, N)).astype(np.float32)
    with _dev(a) as pa, _dev(b) as pb, _dev(dc) as pdc, _out(a.shape) as pda, _out(b.shape) as pdb, _out((N,)) as ps:
        capi.call("seera_hip_matmul_bwd_bias", pa.ptr, pb.ptr, pdc.ptr, pda.ptr, pdb.ptr, ps.ptr, M, N, K, 1)
        db, s = pdb.to_array(b.shape), ps.to_array((N,))
    assert_parity(s, dc.astype(np.float64).sum(0), "db", STRICT)
    np.testing.assert_array_equal(db, hip_matmul_bwd(a, b, dc)[1])
    M, K, N = 512, 4096, 500
    a = r.uniform(-1, 1, (M, K)).astype(np.float32)
    b = r.uniform(-1, 1, (K, N)).astype(np.float32)
    bias = r.uniform(-1, 1, N).astype(np.float32)
    with _dev(a) as pa, _dev(b) as pb, _dev(bias) as pbias, _out((M, N)) as pc, _out((M, N)) as pm:
        capi.call("seera_hip_matmul_bias_act", pa.ptr, pb.ptr, pbias.ptr, pc.ptr, pm.ptr, M, N, K, 1,
                  capi.SEERA_ACT_RELU)
        c, m = pc.to_array((M, N)), pm.to_array((M, N))
    pre = hip_matmul(a, b) + bias
    np.testing.assert_array_equal(c, np.where(pre > 0, pre, 0))
    np.testing.assert_array_equal(m, (pre > 0).astype(np.float32))


def test_captured_without_a_call_before():
    """A capture on a fresh stream has no scratch to split with: the call takes
    the unsplit plan."""
    lib = capi.load()
    M, K, N = 512, 4096, 512
    r = np.random.default_rng(9)
    a = r.uniform(-1, 1, (M, K)).astype(np.float32)
    b = r.uniform(-1, 1, (K, N)).astype(np.float32)
    st, g = ctypes.c_void_p(), ctypes.c_void_p()
    capi.check(lib.seera_hip_stream_create(ctypes.byref(st)))
    try:
        with _dev(a) as pa, _dev(b) as pb, DeviceBuffer(M * N * 4) as pc:
            capi.check(lib.seera_hip_graph_capture_begin(st.value))
            status = lib.seera_hip_matmul_async(pa.ptr, pb.ptr, pc.ptr, M, N, K, 1, st.value)
            capi.check(lib.seera_hip_graph_capture_end(st.value, ctypes.byref(g)))
            capi.check(status)
            for _ in range(3):
                pc.fill(0x7F)
                capi.check(lib.seera_hip_synchronize())
                capi.check(lib.seera_hip_graph_launch(g.value, st.value))
                capi.check(lib.seera_hip_stream_synchronize(st.value))
                got = pc.to_array((M, N))
                assert_parity(got, S.matmul_batched(fp16r(a)[None], fp16r(b))[0], "C", STRICT, 2e-1)
            capi.check(lib.seera_hip_graph_destroy(g.value))
    finally:
        lib.seera_hip_stream_destroy(st.value)
