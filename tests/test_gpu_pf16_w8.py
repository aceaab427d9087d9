"""The INT8 GEMM of independent 16-row waves (pf16_w8_kernel.h) where it can go
wrong: block counts around its ring of four two-block chunks (odd counts end in
half a chunk), partial row tiles, the three scale layouts.  Equal bits to the
oracle, and to the workgroup GEMM."""
import numpy as np
import pytest

from conftest import bits_equal, rng_weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scales", ["channel", "group", "block"])
@pytest.mark.parametrize("K", [32, 64, 224, 256, 288, 544, 1056])
def test_block_counts_and_scales(gpu, hb, orc, hi_prec, monkeypatch, scales, K):
    N = 304
    nblk = K // 32
    rng = np.random.default_rng(K)
    qw, sc, _ = rng_weights(rng, N, K, 8)
    if scales != "block":
        every = nblk if scales == "channel" else 4
        sc = np.ascontiguousarray(np.repeat(sc[:, ::every], every, axis=1)[:, :nblk])
    monkeypatch.setenv("BREEZE_HIP_DEC_ROWS", "8")
    h = hb.prepack(qw, sc, None, K, N, bits=8)
    try:
        for M in (9, 16, 33, 70):
            A = rng.normal(size=(M, K)).astype(np.float32)
            A[rng.random(A.shape) < 0.02] *= 20.0
            for hp in (True, False):
                hb.set_hi_prec(hp)
                got = []
                for mode in ("1", "0"):
                    monkeypatch.setenv("BREEZE_HIP_PF16", mode)
                    c = hb.matmul(h, gpu.from_numpy(A).cuda(), N)
                    gpu.cuda.synchronize()
                    got.append(c.cpu().numpy())
                want = orc.matmul(qw, sc, None, N, K, 8, A, hp)
                assert bits_equal(got[0], want), (M, hp)
                assert bits_equal(got[1], want), (M, hp)
    finally:
        hb.free(h)
