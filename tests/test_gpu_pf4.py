"""The INT4 prefill kernels on the FP6 matrix instructions (pf4_kernel.h,
pf16_kernel.h) where they can go wrong: block counts around a stage of four,
partial column groups and row tiles, per-block scales and zero points, and the
block integers' extremes (the exactness of the FP32 sums).  Equal bits to the
oracle."""
import numpy as np
import pytest

from conftest import bits_equal, rng_weights

pytestmark = pytest.mark.gpu


def _run(gpu, hb, orc, monkeypatch, kernel, qw, sc, qz, A, N, K, hp):
    monkeypatch.setenv("BREEZE_HIP_DEC_ROWS", "8")
    monkeypatch.setenv("BREEZE_HIP_PF16", kernel)
    h = hb.prepack(qw, sc, qz, K, N, bits=4)
    hb.set_hi_prec(hp)
    try:
        got = hb.matmul(h, gpu.from_numpy(A).cuda(), N)
        gpu.cuda.synchronize()
        got = got.cpu().numpy()
    finally:
        hb.free(h)
    assert bits_equal(got, orc.matmul(qw, sc, qz, N, K, 4, A, hp))


@pytest.mark.parametrize("kernel", ["0", "1"])
@pytest.mark.parametrize("zeros", [False, True])
@pytest.mark.parametrize("K", [32, 96, 128, 160, 512, 736, 1056])
def test_block_counts_and_partial_tiles(gpu, hb, orc, hi_prec, monkeypatch, kernel, zeros, K):
    """One to 33 blocks (none to eight whole stages, every remainder; the
    independent waves' unrolled stages and their tail), 19 column tiles, and
    rows around the 16- and 32-row tiles."""
    N = 304
    rng = np.random.default_rng(K + zeros)
    qw, sc, qz = rng_weights(rng, N, K, 4, np.float32, zeros)
    for M in (9, 33, 47, 130):
        A = rng.normal(size=(M, K)).astype(np.float32)
        for hp in (True, False):
            _run(gpu, hb, orc, monkeypatch, kernel, qw, sc, qz, A, N, K, hp)


@pytest.mark.parametrize("kernel", ["0", "1"])
@pytest.mark.parametrize("zp", [None, 0, 15])
@pytest.mark.parametrize("nibble", [0, 15, None])
def test_extreme_block_integers(gpu, hb, orc, hi_prec, monkeypatch, kernel, zp, nibble):
    """Every |q| at 32767 with one sign, alternating signs or at multiples of
    4096 (the top digit alone), against weights of 0, 15 or both: the largest
    partial sums, which the FP32 accumulation must hold exactly."""
    N, K, M = 64, 256, 40
    rng = np.random.default_rng(3)
    n = rng.choice([0, 15], (N, K)).astype(np.uint8) if nibble is None else np.full((N, K), nibble, np.uint8)
    qw = np.ascontiguousarray((n[:, 0::2] | n[:, 1::2] << 4).reshape(N, K // 32, 16))
    sc = rng.uniform(0.001, 0.02, (N, K // 32)).astype(np.float32)
    qz = None if zp is None else np.full((N, (K // 32 + 1) // 2), zp * 17, np.uint8)
    A = np.ones((M, K), np.float32)
    A[1::4] = -1.0
    A[2::4] = rng.choice([-1.0, 1.0], (len(A[2::4]), K))
    q = rng.integers(-7, 8, (len(A[3::4]), K)) * 4096.0
    q[:, ::32] = 32767.0
    A[3::4] = q / 32767.0
    _run(gpu, hb, orc, monkeypatch, kernel, qw, sc, qz, A, N, K, True)
