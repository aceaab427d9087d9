"""INT4 weights with explicit zero points under INT8 activations on the INT8
matrix instructions (prefill_kernel.h, BITS 4): every workgroup shape, block
counts around a four-block stage, partial row pairs and column groups, and
legacy zero points outside 0..15.  Equal bits to the oracle."""
import numpy as np
import pytest

from conftest import bits_equal, rng_weights

pytestmark = pytest.mark.gpu

SHAPES = ["4:17", "4:16", "4:13", "4:12", "4:9", "4:8", "4:5", "4:4", "2:16", "2:8", "2:4", "1:16", "1:8"]


def _force(monkeypatch, shape):
    rp, ct = shape.split(":")
    monkeypatch.setenv("BREEZE_HIP_PF_I8", "1")
    monkeypatch.setenv("BREEZE_HIP_PREFILL_RP", rp)
    monkeypatch.setenv("BREEZE_HIP_PREFILL_CT", ct)
    monkeypatch.setenv("BREEZE_HIP_DEC_ROWS", "8")


@pytest.mark.parametrize("K", [32, 96, 160, 512, 1056])
@pytest.mark.parametrize("shape", SHAPES)
def test_shapes_and_block_counts(gpu, hb, orc, hi_prec, monkeypatch, shape, K):
    N = 304
    _force(monkeypatch, shape)
    rng = np.random.default_rng(K)
    qw, sc, qz = rng_weights(rng, N, K, 4, np.float32, True)
    h = hb.prepack(qw, sc, qz, K, N, bits=4)
    hb.set_hi_prec(False)
    try:
        for M in (9, 33, 70, 130):
            p = hb.plan(4, M, K, N, zeros=True, hi=False)
            assert p["pf_i8"] == 1 and f"{p['pf_rp']}:{p['pf_ct']}" == shape
            A = rng.normal(size=(M, K)).astype(np.float32)
            A[rng.random(A.shape) < 0.02] *= 20.0
            got = hb.matmul(h, gpu.from_numpy(A).cuda(), N)
            gpu.cuda.synchronize()
            assert bits_equal(got.cpu().numpy(), orc.matmul(qw, sc, qz, N, K, 4, A, False)), M
    finally:
        hb.free(h)


@pytest.mark.parametrize("zp_lo,zp_hi", [(-112, 16), (100, 128)])
def test_legacy_zero_points(gpu, hb, orc, hi_prec, monkeypatch, zp_lo, zp_hi):
    """Signed legacy zero points: nibble - zp must not borrow across bytes."""
    N, K = 64, 1056
    nblk = K // 32
    _force(monkeypatch, "4:4")
    rng = np.random.default_rng(zp_lo + 1000)
    B = rng.integers(0, 256, (N // 16, nblk, 8, 32), dtype=np.uint8)
    scale = rng.uniform(0.001, 0.02, (N // 16, nblk, 16)).astype(np.float32)
    zp = rng.integers(zp_lo, zp_hi, (N // 16, nblk, 16)).astype(np.int8)
    _, _, full = orc.unpack_legacy(B, scale, zp, np.zeros_like(scale, dtype=np.int32), N, K, 4)
    corr = np.ascontiguousarray(full.reshape(N // 16, 16, nblk).transpose(0, 2, 1)).astype(np.int32)
    h = hb._lib.i4_prepack(hb._p(B), hb._p(scale), hb._p(zp), hb._p(corr), N, K, nblk, 4)
    assert h, hb.last_error()
    hb.set_hi_prec(False)
    try:
        for M in (33, 130):
            A = rng.normal(size=(M, K)).astype(np.float32)
            got = hb.matmul(h, gpu.from_numpy(A).cuda(), N)
            gpu.cuda.synchronize()
            assert bits_equal(got.cpu().numpy(), orc.matmul_legacy(B, scale, zp, corr, N, K, 4, A, False)), M
    finally:
        hb.free(h)
