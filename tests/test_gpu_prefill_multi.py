"""Several projections of one activation, and the gate/up pair, past the decode
rows: one INT4 prefill launch over all their column tiles.  Segments of 19, 3,
1 and 17 tiles: on the workgroup shapes forced below their ends fall inside a
column group, between the tile slots of a wave, and inside the remainder slot.
Equal bits to the projections one by one, and to the oracle."""
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


def test_zero_points_on_one_of_two(gpu, hb, hi_prec):
    """Per-block scales on both projections and zero points on one: one device
    layout, so one launch (independent waves by the rule)."""
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


def _weights(rng, N, K, zeros, group):
    qw, sc, qz = rng_weights(rng, N, K, 4, np.float32, zeros)
    if group:
        sc = np.ascontiguousarray(np.repeat(sc[:, ::4], 4, axis=1)[:, :K // 32])
    return qw, sc, qz


# 40 tiles: three workgroups of 17 tiles, two of them with a segment's end.
SHAPES = ["4:17", "4:13", "4:9", "4:5", "2:16", "1:16"]


def _shape(monkeypatch, shape):
    rp, ct = shape.split(":")
    monkeypatch.setenv("BREEZE_HIP_PREFILL_RP", rp)
    monkeypatch.setenv("BREEZE_HIP_PREFILL_CT", ct)


@pytest.mark.parametrize("form", ["group", "zeros"])
@pytest.mark.parametrize("shape", SHAPES)
def test_segments_on_a_shape(gpu, hb, orc, hi_prec, monkeypatch, shape, form):
    """Group scales without zero points (the kernels that start from
    -8 sum(q)), and explicit zero points, against the oracle."""
    Ns, K = [304, 48, 16, 272], 544
    rng = np.random.default_rng(17)
    w = [_weights(rng, n, K, form == "zeros", form == "group") for n in Ns]
    hs = [hb.prepack(qw, sc, qz, K, n, bits=4) for n, (qw, sc, qz) in zip(Ns, w)]
    _shape(monkeypatch, shape)
    try:
        for M in (33, 150):
            for hp in (True, False):
                p = hb.plan(4, M, K, sum(Ns), multi=True, zeros=form == "zeros", hi=hp)
                assert f"{p['pf_rp']}:{p['pf_ct']}" == shape and p["pf_zp"] == (form == "zeros")
                A = rng.normal(size=(M, K)).astype(np.float32)
                hb.set_hi_prec(hp)
                got = hb.matmul_multi(hs, gpu.from_numpy(A).cuda(), Ns)
                gpu.cuda.synchronize()
                for n, (qw, sc, qz), c in zip(Ns, w, got):
                    assert bits_equal(c.cpu().numpy(), orc.matmul(qw, sc, qz, n, K, 4, A, hp)), (M, hp, n)
    finally:
        for h in hs:
            hb.free(h)


@pytest.mark.parametrize("form", ["group", "zeros"])
@pytest.mark.parametrize("shape", SHAPES)
def test_gate_up_on_a_shape(gpu, hb, orc, hi_prec, monkeypatch, shape, form):
    """Two segments of 19 tiles; SiLU(gate) * up of the oracle's products."""
    N, K, M = 304, 416, 70
    rng = np.random.default_rng(18)
    w = [_weights(rng, N, K, form == "zeros", form == "group") for _ in range(2)]
    gate, up = (hb.prepack(qw, sc, qz, K, N, bits=4) for qw, sc, qz in w)
    _shape(monkeypatch, shape)
    A = rng.normal(size=(M, K)).astype(np.float32)
    try:
        for hp in (True, False):
            hb.set_hi_prec(hp)
            got = hb.matmul_silu_mul(gate, up, gpu.from_numpy(A).cuda(), N)
            gpu.cuda.synchronize()
            g, u = (orc.matmul(qw, sc, qz, N, K, 4, A, hp) for qw, sc, qz in w)
            want = hb.silu_mul(gpu.from_numpy(g).cuda(), gpu.from_numpy(u).cuda()).cpu().numpy()
            assert bits_equal(got.cpu().numpy(), want), hp
    finally:
        hb.free(gate)
        hb.free(up)


def test_mixed_scale_layouts_run_one_by_one(gpu, hb, orc, hi_prec):
    """Group scales on one projection and per-block scales on the other: two
    device layouts, no shared launch, the same bits."""
    K, N, M = 320, 64, 40
    rng = np.random.default_rng(9)
    w = [_weights(rng, N, K, False, group) for group in (True, False)]
    hs = [hb.prepack(qw, sc, qz, K, N, bits=4) for qw, sc, qz in w]
    assert [hb.handle_info(h)["scale_group"] for h in hs] == [4, 1]
    A = rng.normal(size=(M, K)).astype(np.float32)
    hb.set_hi_prec(True)
    try:
        for (qw, sc, qz), c in zip(w, hb.matmul_multi(hs, gpu.from_numpy(A).cuda(), [N, N])):
            assert bits_equal(c.cpu().numpy(), orc.matmul(qw, sc, qz, N, K, 4, A, True))
    finally:
        for h in hs:
            hb.free(h)
