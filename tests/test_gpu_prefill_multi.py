"""Several projections of one activation, and the gate/up pair, past the decode
rows: one INT4 prefill launch over all their column tiles.  Segment ends fall
inside a column group, a workgroup and a wave's tile slots (3, 1 and 19 tiles).
Equal bits to the projections one by one."""
import numpy as np
import pytest

from conftest import bits_equal, rng_weights

pytestmark = pytest.mark.gpu


def _pack(hb, rng, K, Ns, zeros):
    hs = []
    for n in Ns:
        qw, sc, qz = rng_weights(rng, n, K, 4, np.float32, zeros)
        hs.append(hb.prepack(qw, sc, qz, K, n, bits=4))
    return hs


@pytest.mark.parametrize("kernel", ["0", "1"])
@pytest.mark.parametrize("zeros", [False, True])
@pytest.mark.parametrize("K", [160, 1056])
def test_multi_is_the_projections(gpu, hb, hi_prec, monkeypatch, kernel, zeros, K):
    Ns = [304, 48, 16, 272]
    rng = np.random.default_rng(K)
    hs = _pack(hb, rng, K, Ns, zeros)
    monkeypatch.setenv("BREEZE_HIP_PF16", kernel)
    try:
        for M in (33, 70, 129):
            A = gpu.from_numpy(rng.normal(size=(M, K)).astype(np.float32)).cuda()
            for hp in (True, False):
                hb.set_hi_prec(hp)
                got = hb.matmul_multi(hs, A, Ns)
                for h, n, c in zip(hs, Ns, got):
                    assert bits_equal(c.cpu().numpy(), hb.matmul(h, A, n).cpu().numpy()), (M, hp, n)
    finally:
        for h in hs:
            hb.free(h)


@pytest.mark.parametrize("kernel", ["0", "1"])
@pytest.mark.parametrize("zeros", [False, True])
def test_gate_up_is_two_products_and_silu(gpu, hb, hi_prec, monkeypatch, kernel, zeros):
    K, N = 544, 304
    rng = np.random.default_rng(8)
    gate, up = _pack(hb, rng, K, [N, N], zeros)
    monkeypatch.setenv("BREEZE_HIP_PF16", kernel)
    try:
        for M in (33, 130):
            A = gpu.from_numpy(rng.normal(size=(M, K)).astype(np.float32)).cuda()
            for hp in (True, False):
                hb.set_hi_prec(hp)
                got = hb.matmul_silu_mul(gate, up, A, N).cpu().numpy()
                want = hb.silu_mul(hb.matmul(gate, A, N), hb.matmul(up, A, N)).cpu().numpy()
                assert bits_equal(got, want), (M, hp)
    finally:
        hb.free(gate)
        hb.free(up)


def test_mixed_layouts_still_run_one_by_one(gpu, hb, hi_prec):
    """Zero points on one of two projections: no shared launch."""
    K, N, M = 320, 64, 40
    rng = np.random.default_rng(9)
    a, = _pack(hb, rng, K, [N], False)
    b, = _pack(hb, rng, K, [N], True)
    hb.set_hi_prec(True)
    try:
        A = gpu.from_numpy(rng.normal(size=(M, K)).astype(np.float32)).cuda()
        for h, c in zip((a, b), hb.matmul_multi([a, b], A, [N, N])):
            assert bits_equal(c.cpu().numpy(), hb.matmul(h, A, N).cpu().numpy())
    finally:
        hb.free(a)
        hb.free(b)


@pytest.mark.parametrize("kernel", ["0", "1"])
def test_zero_points_on_one_projection(gpu, hb, orc, hi_prec, monkeypatch, kernel):
    """Per-block scales on both and explicit zero points on one: one device
    layout, so one launch, which reads the zero points of both (8 on the one
    without).  Equal bits to the oracle, in either order."""
    K, N, M = 416, 80, 70
    rng = np.random.default_rng(4)
    w = [rng_weights(rng, N, K, 4, np.float32, z) for z in (False, True)]
    hs = [hb.prepack(qw, sc, qz, K, N, bits=4) for qw, sc, qz in w]
    monkeypatch.setenv("BREEZE_HIP_PF16", kernel)
    A = rng.normal(size=(M, K)).astype(np.float32)
    d = gpu.from_numpy(A).cuda()
    try:
        for hp in (True, False):
            hb.set_hi_prec(hp)
            want = [orc.matmul(qw, sc, qz, N, K, 4, A, hp) for qw, sc, qz in w]
            for o in ((0, 1), (1, 0)):
                got = hb.matmul_multi([hs[i] for i in o], d, [N, N])
                for i, c in zip(o, got):
                    assert bits_equal(c.cpu().numpy(), want[i]), (hp, o, i)
    finally:
        for h in hs:
            hb.free(h)
