"""Matrix products over operands packed to fp16 (gemm_packed.hip): every tile
and split of its plan at remainders of tiles, slices and rows. The operands
are small whole numbers, so every product and every partial sum is exact in
fp16 and fp32 and the results must equal the integer product."""
import numpy as np
import pytest

from ml_framework_amd import capi
from ml_framework_amd.capi import DeviceBuffer
from oracle import fp16r
from tests.helpers import _dev, _out, hip_matmul, hip_matmul_bwd

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True, scope="module")
def _gpu():
    assert capi.gpu_available(), "no HIP device visible"


def _ints(r, shape):
    return r.integers(-3, 4, shape).astype(np.float32)  # sums of 2^20 products stay below 2^24


def _mm(a, b):
    return (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32)


# (M, K, N, Nbatch); the tiles (and splits) of C, dA and dB
SHAPES = [
    (512, 250, 257, 1),    # 64, 64, 64
    (85, 511, 513, 3),     # 64, 64, 64 over a batch
    (1030, 66, 515, 1),    # 64 with one slice and two columns more
    (70, 4099, 130, 1),    # 64 in 16 parts, 64, 64
    (1025, 8191, 333, 1),  # 128 in 8 parts, 64, 64
    (2305, 1001, 3333, 1), # 64, 128, 128
    (3329, 129, 2817, 1),  # 64, 64 in 4, 64 in 4
    (300, 2561, 2561, 1),  # 64 in 2, 64 in 2, 256
    (1500, 1500, 1500, 1), # whole float4s, ragged slices
    (2304, 2560, 2560, 1), # whole slices: tiles that leave compute units idle
    (3001, 1501, 2047, 1), # 256, 256, 128
]


@pytest.mark.parametrize("M,K,N,nb", SHAPES)
def test_exact(M, K, N, nb):
    r = np.random.default_rng(M + K)
    a, b, dc = _ints(r, (nb, M, K)), _ints(r, (K, N)), _ints(r, (nb, M, N))
    np.testing.assert_array_equal(hip_matmul(a, b), _mm(a, b))
    da, db = hip_matmul_bwd(a, b, dc)
    np.testing.assert_array_equal(da, _mm(dc, b.T))
    np.testing.assert_array_equal(db, _mm(a.reshape(-1, K).T, dc.reshape(-1, N)))


@pytest.mark.parametrize("M,K,N,nb", SHAPES[:8] + SHAPES[-1:])
def test_epilogues(M, K, N, nb):
    r = np.random.default_rng(N)
    a, b, dc = _ints(r, (nb, M, K)), _ints(r, (K, N)), _ints(r, (nb, M, N))
    bias, gate = _ints(r, (N,)), (r.random((nb, M, K)) < 0.5).astype(np.float32)
    pre = _mm(a, b) + bias
    want_da, want_db = _mm(dc, b.T), _mm(a.reshape(-1, K).T, dc.reshape(-1, N))
    with _dev(a) as pa, _dev(b) as pb, _dev(dc) as pdc, _dev(bias) as pbias, _dev(gate) as pg, \
            _out(dc.shape) as pc, _out(dc.shape) as pm, _out(a.shape) as pda, _out(b.shape) as pdb, _out((N,)) as ps:
        capi.call("seera_hip_matmul_bias_act", pa.ptr, pb.ptr, pbias.ptr, pc.ptr, pm.ptr, M, N, K, nb,
                  capi.SEERA_ACT_RELU)
        np.testing.assert_array_equal(pc.to_array(dc.shape), np.maximum(pre, 0))
        np.testing.assert_array_equal(pm.to_array(dc.shape), (pre > 0).astype(np.float32))
        capi.call("seera_hip_matmul_bwd_relu", pa.ptr, pb.ptr, pdc.ptr, pg.ptr, pda.ptr, pdb.ptr, M, N, K, nb)
        np.testing.assert_array_equal(pda.to_array(a.shape), np.where(gate > 0, want_da, 0))
        np.testing.assert_array_equal(pdb.to_array(b.shape), want_db)
        capi.call("seera_hip_matmul_bwd_bias", pa.ptr, pb.ptr, pdc.ptr, pda.ptr, pdb.ptr, ps.ptr, M, N, K, nb)
        np.testing.assert_array_equal(pda.to_array(a.shape), want_da)
        np.testing.assert_array_equal(pdb.to_array(b.shape), want_db)
        np.testing.assert_array_equal(ps.to_array((N,)), dc.reshape(-1, N).sum(0))


def test_rounding():
    """Sums of K products in fp32, in any order: within (K + 2) 2^-24 of the
    sum of their magnitudes."""
    r = np.random.default_rng(1)
    for M, K, N in [(515, 1027, 333), (2305, 2049, 2051)]:
        a, b = (r.standard_normal(s).astype(np.float32) for s in ((M, K), (K, N)))
        ra, rb = fp16r(a).astype(np.float64), fp16r(b).astype(np.float64)
        err = np.abs(hip_matmul(a[None], b)[0] - ra @ rb)
        assert (err <= (K + 2) * 2.0 ** -24 * (np.abs(ra) @ np.abs(rb))).all()


def test_not_finite():
    """Infinities and NaN reach the entries that use them and no others; a
    value past fp16's range becomes an infinity."""
    r = np.random.default_rng(2)
    M, K, N = 513, 515, 259
    a, b = _ints(r, (1, M, K)) + 4, _ints(r, (K, N)) + 4
    a[0, -1, -1], a[0, 3, 0], b[-1, 5] = np.inf, 1e6, np.nan
    c = hip_matmul(a, b)[0]
    nan, inf = np.zeros((M, N), bool), np.zeros((M, N), bool)
    inf[-1], inf[3], nan[:, 5] = True, True, True
    np.testing.assert_array_equal(np.isnan(c), nan)
    np.testing.assert_array_equal(np.isposinf(c), inf & ~nan)


@pytest.mark.parametrize("shift", [(1, 0, 0), (0, 3, 0), (0, 0, 2)])
def test_operands_off_16_bytes(shift):
    """Whole float4 rows at addresses that are only 4-byte aligned."""
    M, K, N = 384, 512, 320
    r = np.random.default_rng(5)
    a, b, dc = _ints(r, (M, K)), _ints(r, (K, N)), _ints(r, (M, N))
    pad = [np.concatenate([np.full(s, np.nan, np.float32), x.ravel()]) for s, x in zip(shift, (a, b, dc))]
    with _dev(pad[0]) as pa, _dev(pad[1]) as pb, _dev(pad[2]) as pdc, DeviceBuffer(M * N * 4) as pc, \
            DeviceBuffer(M * K * 4) as pda, DeviceBuffer(K * N * 4) as pdb:
        qa, qb, qdc = (p.ptr + 4 * s for p, s in zip((pa, pb, pdc), shift))
        capi.call("seera_hip_matmul", qa, qb, pc.ptr, M, N, K, 1)
        capi.call("seera_hip_matmul_bwd", qa, qb, qdc, pda.ptr, pdb.ptr, M, N, K, 1)
        np.testing.assert_array_equal(pc.to_array((M, N)), _mm(a, b))
        np.testing.assert_array_equal(pda.to_array((M, K)), _mm(dc, b.T))
        np.testing.assert_array_equal(pdb.to_array((K, N)), _mm(a.T, dc))
