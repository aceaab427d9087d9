"""The INT4 prefill kernels on the FP6 matrix instructions (pf4_kernel.h,
pf16_kernel.h) where they can go wrong: block counts around a stage of four,
partial column groups and row tiles, every workgroup shape, both depths of the
independent waves' prefetch, per-block and group scales, zero points, and the
block integers' extremes (the exactness of the FP32 sums).  Kernels without
zero points run where none are given, whatever the scales.  Equal bits to the
oracle."""
import numpy as np
import pytest

from conftest import bits_equal, rng_weights

pytestmark = pytest.mark.gpu


# "0" and "1": workgroups of the rule's shape, independent waves; "1:2" and
# "1:4": these with two and four weight chunks in flight; "s4:17": workgroups of
# four row pairs by 17 column tiles.
def _force(monkeypatch, kernel):
    monkeypatch.setenv("BREEZE_HIP_PF_I8", "0")
    if kernel[0] == "s":
        rp, ct = kernel[1:].split(":")
        monkeypatch.setenv("BREEZE_HIP_PREFILL_RP", rp)
        monkeypatch.setenv("BREEZE_HIP_PREFILL_CT", ct)
        return
    monkeypatch.setenv("BREEZE_HIP_PF16", kernel[0])
    if len(kernel) > 1:
        monkeypatch.setenv("BREEZE_HIP_PF16_AHEAD", kernel[2])


def _run(gpu, hb, orc, monkeypatch, kernel, qw, sc, qz, A, N, K, hp):
    monkeypatch.setenv("BREEZE_HIP_DEC_ROWS", "8")
    _force(monkeypatch, kernel)
    p = hb.plan(4, len(A), K, N, zeros=qz is not None, hi=hp)
    assert p["pf_zp"] == (qz is not None and not (qz == 0x88).all())
    if kernel in ("1:4", "1:2"):
        assert (p["pf_rp"], p["pf_ahead"]) == (0, int(kernel[2]))
    elif kernel not in ("0", "1"):
        assert f"{p['pf_rp']}:{p['pf_ct']}" == kernel[1:]
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


# Odd column tiles leave half a group empty, 17 and 13 and 9 have slots of a
# remainder and parts of different widths, 5 and 4 only a remainder.
SHAPES = ["s4:17", "s4:16", "s4:13", "s4:12", "s4:9", "s4:8", "s4:5", "s4:4", "s2:16", "s2:8", "s2:4", "s1:16", "s1:8"]


@pytest.mark.parametrize("scales", ["group", "zeros"])
@pytest.mark.parametrize("kernel", SHAPES + ["1:2", "1:4"])
def test_every_shape_and_depth(gpu, hb, orc, hi_prec, monkeypatch, kernel, scales):
    """Block counts of no, one and several stages with every remainder (1, 3,
    4, 5, 8, 9, 23, 33), 41 column tiles (every shape has a partial last
    workgroup), rows that leave a row pair partial or without rows."""
    N = 656
    for nblk in (1, 3, 4, 5, 8, 9, 23, 33):
        K = 32 * nblk
        rng = np.random.default_rng(nblk)
        qw, sc, qz = rng_weights(rng, N, K, 4, np.float32, scales == "zeros")
        if scales == "group":
            sc = np.ascontiguousarray(np.repeat(sc[:, ::4], 4, axis=1)[:, :nblk])
        M = (70, 33, 130, 47, 9, 100, 150, 64)[nblk % 8]
        A = rng.normal(size=(M, K)).astype(np.float32)
        for hp in (True, False):
            _run(gpu, hb, orc, monkeypatch, kernel, qw, sc, qz, A, N, K, hp)


@pytest.mark.parametrize("kernel", ["s4:17", "s4:5", "1:2"])
@pytest.mark.parametrize("zp", [None, 0, 15])
def test_extreme_block_integers_with_group_scales(gpu, hb, orc, hi_prec, monkeypatch, kernel, zp):
    """The extremes again where a model's group scales and an odd shape are:
    the accumulator starts at -8 sum(q) without zero points."""
    N, K, M = 288, 256, 70
    rng = np.random.default_rng(7)
    n = rng.choice([0, 15], (N, K)).astype(np.uint8)
    n[::3], n[1::3] = 0, 15
    qw = np.ascontiguousarray((n[:, 0::2] | n[:, 1::2] << 4).reshape(N, K // 32, 16))
    sc = np.ascontiguousarray(np.repeat(rng.uniform(0.001, 0.02, (N, 2)).astype(np.float32), 4, axis=1))
    qz = None if zp is None else np.full((N, K // 64), zp * 17, np.uint8)
    A = np.ones((M, K), np.float32)
    A[1::5] = -1.0
    A[2::5] = rng.choice([-1.0, 1.0], (len(A[2::5]), K))
    q = rng.integers(-8, 8, (len(A[3::5]), K)) * 4096.0 + rng.choice([0, 4095], (len(A[3::5]), K))
    q = np.clip(q, -32767, 32767)
    q[:, ::32] = 32767.0
    A[3::5] = q / 32767.0
    A[4::5] = -(np.arange(K) % 2) * 28673.0 / 32767.0
    A[4::5, ::32] = -1.0
    for hp in (True, False):
        _run(gpu, hb, orc, monkeypatch, kernel, qw, sc, qz, A, N, K, hp)
