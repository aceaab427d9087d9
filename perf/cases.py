"""The calls a program makes of the quantized linear path, as timed cases.

Each case is one call of a public entry point of ``breeze_amd.hip_backend`` on
GPU tensors, with the weights prepacked beforehand as a model loader does:

- ``matmul``: one projection;
- ``argmax``: the LM head, logits and the greedy token;
- ``gate_up``: a decoder MLP's gate and up projections with SiLU(gate) * up;
- ``norm_multi``: RMSNorm and the projections that read it, in one call.

``bits`` is the weight width, ``group`` the 32-blocks that share one scale (0:
one scale a column), ``hi`` the activation mode (two-pass INT16, or INT8),
``zeros`` explicit INT4 zero points, ``half`` scales stored as fp16.
"""
import os
import sys
import weakref

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "breeze-engine_amd"))
from breeze_amd import hip_backend as hb  # noqa: E402

EPS = 1e-6


def _case(name, call, bits, M, K, Ns, group, hi=True, zeros=False, half=False, outliers=False):
    c = dict(call=call, bits=bits, M=M, K=K, N=",".join(map(str, Ns)), group=group, hi=hi, zeros=zeros, half=half,
             outliers=outliers)
    return dict(c, name=name) if name else c


def _ns(case):
    return [int(n) for n in case["N"].split(",")]


def listed():
    return [
        # Single-token decode, the smallest projection: launches and latency count.
        _case("w8_gemv", "matmul", 8, 1, 4096, [4096], 0),
        # Single-token decode, a wide W4 projection (the benchmark's headline shape).
        _case("w4_gemv", "matmul", 4, 1, 4096, [12288], 4),
        # A few tokens at once (speculative or small-batch decode), activations with outliers.
        _case("w4_decode_4", "matmul", 4, 4, 12288, [4096], 4, outliers=True),
        # The linear-attention block's norm and its four projections, single-token decode.
        _case("norm_qkvz", "norm_multi", 4, 1, 5120, [10240, 6144, 48, 48], 4),
        # The MLP's first half, single-token decode.
        _case("gate_up_1", "gate_up", 4, 1, 5120, [17408], 4),
        # The LM head with greedy sampling.
        _case("lm_head", "argmax", 8, 1, 5120, [151936], 0),
        # Batched decode of ragged size through the MLP's down projection.
        _case("w4_down_23", "matmul", 4, 23, 17408, [5120], 4),
        # A short prompt of odd length, fp16 scales and explicit zero points, INT8
        # activations (the mode a process starts in).
        _case("w4_zp_short_77", "matmul", 4, 77, 5120, [5120], 4, hi=False, zeros=True, half=True),
        # A medium batch or short prompt, INT8 weights.
        _case("w8_batch_64", "matmul", 8, 64, 5120, [5120], 0),
        # The MLP's first half for a prompt of ragged length.
        _case("gate_up_200", "gate_up", 4, 200, 5120, [17408], 4),
        # Prompt prefill, INT8 weights.
        _case("w8_prefill", "matmul", 8, 512, 5120, [17408], 0),
        # Prompt prefill, INT4 weights.
        _case("w4_prefill", "matmul", 4, 512, 5120, [17408], 4),
    ]


def _log(rng, lo, hi, step):
    """A multiple of `step` in [lo, hi], spread over the logarithm."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random() / step)) * step))


def draw(rng):
    call = rng.choice(["matmul", "matmul", "matmul", "argmax", "gate_up", "norm_multi"])
    bits = 8 if call == "argmax" or (call == "matmul" and rng.random() < 0.4) else 4
    K = _log(rng, 1024, 17408, 32)
    hi = rng.random() < 0.8
    zeros = bits == 4 and call == "matmul" and rng.random() < 0.2
    half = rng.random() < 0.3
    group = 0 if bits == 8 else rng.choice([1, 4, 4, 4])
    if K // 32 % 4:
        group = min(group, 1)
    M = _log(rng, 1, 512, 1)
    if call == "argmax":
        M, Ns = min(M, 8), [_log(rng, 16384, 151936, 16)]
    elif call == "norm_multi":
        Ns = [_log(rng, 1024, 12288, 16), _log(rng, 1024, 6144, 16), 48, 48][:rng.choice([2, 3, 4])]
    else:
        Ns = [_log(rng, 1024, 17408, 16)]
    pair = 2 if call == "gate_up" else 1
    # No more multiply-adds than the largest listed product.
    M = max(1, min(M, 512 * 5120 * 17408 // (pair * K * sum(Ns))))
    # No more weight bytes than the LM head.
    while pair * K * sum(Ns) * bits // 8 > 5120 * 151936:
        Ns = [max(16, n // 32 * 16) for n in Ns]
    return _case(None, call, bits, M, K, Ns, group, hi, zeros, half, outliers=rng.random() < 0.3)


def _weights(gen, case, N):
    """MatMulNBits arrays on the GPU: bytes [N, nblk, 4*bits], distinct scales
    [N, groups], packed zero points [N, ceil(nblk/2)] or None."""
    bits, nblk = case["bits"], case["K"] // 32
    dev = "cuda"
    ng = nblk // case["group"] if case["group"] else 1
    std = 0.02 / (127 if bits == 8 else 7)
    scales = (torch.randn((N, ng), generator=gen, device=dev).abs() * std).clamp_min(1e-6)
    scales = scales.to(torch.float16 if case["half"] else torch.float32)
    # INT8 weights span [-127, 127] around 128.
    lo = 1 if bits == 8 else 0
    qw = torch.randint(lo, 256, (N, nblk, 4 * bits), generator=gen, device=dev, dtype=torch.uint8)
    qz = None
    if case["zeros"]:
        lo4, hi4 = (torch.randint(5, 12, (N, (nblk + 1) // 2), generator=gen, device=dev, dtype=torch.uint8)
                    for _ in range(2))
        qz = lo4 | (hi4 << 4)
    return qw, scales, qz


def _inputs(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed * 1000003 + case["K"] * 31 + case["M"])
    ns = _ns(case) * (2 if case["call"] == "gate_up" else 1)
    weights = [_weights(gen, case, n) for n in ns]
    A = torch.randn((case["M"], case["K"]), generator=gen, device="cuda")
    if case["outliers"]:
        A *= torch.where(torch.rand(A.shape, generator=gen, device="cuda") < 0.01, 20.0, 1.0)
    w = 1 + 0.1 * torch.randn((case["K"],), generator=gen, device="cuda") if case["call"] == "norm_multi" else None
    return ns, weights, A, w


class _State:
    pass


def _release(handles):
    for h in handles:
        hb.free(h)


def prepare(case, seed):
    ns, weights, A, w = _inputs(case, seed)
    s = _State()
    s.case, s.A, s.w, s.ns = case, A, w, ns
    s.handles = []
    weakref.finalize(s, _release, s.handles)
    nblk = case["K"] // 32
    for n, (qw, sc, qz) in zip(ns, weights):
        sc = sc.cpu().numpy()
        sc = np.ascontiguousarray(np.repeat(sc, nblk // sc.shape[1], axis=1))
        qz = None if qz is None else qz.cpu().numpy()
        s.handles.append(hb.prepack(qw.cpu().numpy(), sc, qz, case["K"], n, bits=case["bits"]))
    return s


def run(s):
    c = s.case
    hb.set_hi_prec(c["hi"])
    if c["call"] == "matmul":
        return hb.matmul(s.handles[0], s.A, s.ns[0])
    if c["call"] == "argmax":
        return hb.matmul_argmax(s.handles[0], s.A, s.ns[0])
    if c["call"] == "gate_up":
        return hb.matmul_silu_mul(s.handles[0], s.handles[1], s.A, s.ns[0])
    return hb.rmsnorm_matmul_multi(s.A, s.w, EPS, s.handles, s.ns)


def work(case):
    """Packed weights, one fp32 (or fp16) per distinct scale, zero points and
    fp32 activations in, fp32 outputs out; a multiply-add per weight and row."""
    M, K, ns = case["M"], case["K"], _ns(case)
    pair = 2 if case["call"] == "gate_up" else 1
    N, nblk = sum(ns), K // 32
    b = pair * (N * K * case["bits"] // 8 + (2 if case["half"] else 4) * N * (nblk // case["group"] if case["group"] else 1))
    b += N * ((nblk + 1) // 2) if case["zeros"] else 0
    b += 4 * M * K + 4 * M * N + (4 * K if case["call"] == "norm_multi" else 0) + (8 * M if case["call"] == "argmax" else 0)
    return {"bytes": b, "flops": 2 * pair * M * N * K}


def tolerance(case):
    """fp32 sums of K/32 exact block products: summed in another order, rows of
    up to 544 blocks differ by 2e-7 to 5e-7 (2-norm), single values by up to 3e-6
    of the root mean square.  RMSNorm may also move an activation's INT16 (or
    INT8) step to its neighbour, as may the sums inside SiLU(gate) * up."""
    if case["call"] == "norm_multi":
        return {"rel": 4e-5 if case["hi"] else 2e-3, "max": 4e-4 if case["hi"] else 2e-2}
    if case["call"] == "argmax":
        return {"rel": 2e-6, "max": 2e-5, "differ": 0.0}
    return {"rel": 2e-6, "max": 2e-5}


def _dense(case, weights, n):
    """fp64 weights [n, K] of one handle."""
    qw, sc, qz = weights
    nblk = case["K"] // 32
    if case["bits"] == 8:
        w = qw.to(torch.float64) - 128.0
    else:
        w = torch.stack((qw & 15, qw >> 4), dim=-1).reshape(n, nblk, 32).to(torch.float64)
        if qz is None:
            w -= 8.0
        else:
            z = torch.stack((qz & 15, qz >> 4), dim=-1).reshape(n, -1)[:, :nblk]
            w -= z.to(torch.float64)[:, :, None]
    w *= sc.to(torch.float64).repeat_interleave(nblk // sc.shape[1], dim=1)[:, :, None]
    return w.reshape(n, case["K"])


def exact(case, seed):
    """The products with the activations as given, not quantized."""
    ns, weights, A, w = _inputs(case, seed)
    a = A.to(torch.float64)
    if w is not None:
        a = a / torch.sqrt((a * a).mean(dim=1, keepdim=True) + EPS) * w.to(torch.float64)
    outs = [a @ _dense(case, x, n).t() for n, x in zip(ns, weights)]
    if case["call"] == "gate_up":
        return outs[0] / (1 + torch.exp(-outs[0])) * outs[1]
    if case["call"] == "argmax":
        return outs[0], None
    return outs if case["call"] == "norm_multi" else outs[0]
