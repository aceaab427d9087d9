"""The GPU path inside a captured HIP graph: the per-layer sequence of the
decoder's MLP (qwen35_decoder.cpp:405-409: gate and up projections, SiLU
times up, down projection) and the LM head's argmax, captured once after one
uncaptured call per shape on the capturing stream (which sizes that
stream's device scratch) and replayed.  Every replay is checked bit for bit
against the same sequence run eagerly on the same inputs, with eager work and
synchronisations between the replays."""
import numpy as np
import pytest

from conftest import bits_equal, rng_weights

pytestmark = pytest.mark.gpu


def _mlp(hb, torch, hg, hu, hd, x, inter, H):
    g = hb.matmul(hg, x, inter)
    u = hb.matmul(hu, x, inter)
    return hb.matmul(hd, torch.nn.functional.silu(g) * u, H)


# Hidden sizes past 4096 put the gate and up projections on the stand-alone
# quantizer and the eight-row groups (8 rows: one group, W4 with zero points;
# 16 rows: two, W8).
@pytest.mark.parametrize("rows,bits,H,inter", [(1, 4, 512, 1024), (4, 4, 512, 1024), (64, 8, 512, 1024),
                                               (8, 4, 5120, 1024), (16, 8, 4640, 2048)])
def test_captured_mlp_block_replays_bit_exact(gpu, hb, hi_prec, rows, bits, H, inter):
    torch = gpu
    rng = np.random.default_rng(rows + bits)
    hs = []
    for K, N in ((H, inter), (H, inter), (inter, H)):
        qw, sc, qz = rng_weights(rng, N, K, bits, np.float32, bits == 4)
        hs.append(hb.prepack(qw, sc, qz, K, N, bits=bits))
    try:
        hb.set_hi_prec(True)
        inputs = [torch.from_numpy(rng.normal(size=(rows, H)).astype(np.float32)).cuda() for _ in range(4)]
        cap = torch.cuda.Stream()
        cap.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(cap):
            want = [_mlp(hb, torch, *hs, x, inter, H) for x in inputs]  # also the uncaptured first calls
        torch.cuda.synchronize()

        x_static = inputs[0].clone()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=cap):
            y_static = _mlp(hb, torch, *hs, x_static, inter, H)
        for i, x in enumerate(inputs):
            x_static.copy_(x)
            graph.replay()
            torch.cuda.synchronize()
            assert bits_equal(y_static.cpu().numpy(), want[i].cpu().numpy()), (rows, bits, i)
            # Eager work between replays.
            again = _mlp(hb, torch, *hs, inputs[(i + 1) % len(inputs)], inter, H)
            torch.cuda.synchronize()
            assert bits_equal(again.cpu().numpy(), want[(i + 1) % len(inputs)].cpu().numpy())
    finally:
        for h in hs:
            hb.free(h)


def test_captured_argmax_replays_exact(gpu, hb, hi_prec):
    torch = gpu
    K, N = 1024, 16 * 600
    rng = np.random.default_rng(5)
    qw, sc, _ = rng_weights(rng, N, K, 8)
    h = hb.prepack(qw, sc, None, K, N, bits=8)
    try:
        hb.set_hi_prec(True)
        inputs = [torch.from_numpy(rng.normal(size=(1, K)).astype(np.float32)).cuda() for _ in range(3)]
        cap = torch.cuda.Stream()
        cap.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(cap):
            want = [hb.matmul_argmax(h, x, N) for x in inputs]
        torch.cuda.synchronize()
        x_static = inputs[0].clone()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=cap):
            logits, idx = hb.matmul_argmax(h, x_static, N)
        for i, x in enumerate(inputs):
            x_static.copy_(x)
            graph.replay()
            torch.cuda.synchronize()
            assert bits_equal(logits.cpu().numpy(), want[i][0].cpu().numpy()), i
            assert idx.cpu().tolist() == want[i][1].cpu().tolist(), i
            _ = hb.matmul_argmax(h, inputs[(i + 2) % len(inputs)], N)  # eager call between replays
            torch.cuda.synchronize()
    finally:
        hb.free(h)


@pytest.mark.parametrize("first,then", [
    ((8, 256), (8, 240)),   # workgroups, then independent waves (larger records a row)
    ((8, 128), (4, 128)),   # INT8 weights, then INT4 (FP6 records)
    ((4, 128), (8, 128)),
])
def test_capture_after_a_call_of_as_many_rows(gpu, hb, orc, hi_prec, monkeypatch, first, then):
    """A stream's room for the prefill's records depends on the rows and K
    alone, so after one call a call of no more rows is captured without an
    allocation, whatever its launch and weights; replays are bit-exact with
    eager work between them."""
    torch = gpu
    K, N = 1024, 3536
    rng = np.random.default_rng(first[1])
    handles, weights = {}, {}
    for bits in (4, 8):
        qw, sc, _ = rng_weights(rng, N, K, bits)
        sc = np.ascontiguousarray(np.repeat(sc[:, :1], K // 32, axis=1))
        weights[bits] = (qw, sc)
        handles[bits] = hb.prepack(qw, sc, None, K, N, bits=bits)
    hb.set_hi_prec(True)
    waves = first[0] == then[0] == 8

    def launch(which):
        if waves:
            monkeypatch.setenv("BREEZE_HIP_PF16", "01"[which == then])
            assert (hb.plan(8, which[1], K, N)["pf_rp"] == 0) == (which == then)

    try:
        cap = torch.cuda.Stream()
        a0 = torch.from_numpy(rng.normal(size=(first[1], K)).astype(np.float32)).cuda()
        A = [rng.normal(size=(then[1], K)).astype(np.float32) for _ in range(3)]
        x = torch.from_numpy(A[0]).cuda()
        torch.cuda.synchronize()
        launch(first)
        with torch.cuda.stream(cap):
            hb.matmul(handles[first[0]], a0, N)
        torch.cuda.synchronize()
        launch(then)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=cap):
            y = hb.matmul(handles[then[0]], x, N)
        for a in A:
            x.copy_(torch.from_numpy(a))
            graph.replay()
            torch.cuda.synchronize()
            assert bits_equal(y.cpu().numpy(), orc.matmul(*weights[then[0]], None, N, K, then[0], a, True))
            with torch.cuda.stream(cap):
                hb.matmul(handles[first[0]], a0, N)
            torch.cuda.synchronize()
    finally:
        for h in handles.values():
            hb.free(h)
