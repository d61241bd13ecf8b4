"""The workloads this library is timed on, as a program that uses it would run them.

Three kinds of call, all through the public entry points:

  matmul   C[M,N] int32 = A[M,K] int8 x W[K,N] ternary (ternix_hip_mul_mat_ternary, or the host-array
           form ternary_matmul)
  linear   one quantised linear layer: per-row activation quantisation of fp32 rows, then the matmul
           with the dequantisation in its output (ternix_hip_quantize_activations +
           ternix_hip_mul_mat_ternary_dequant, or the _tile64_dequant form on pre-permuted weights)
  ffn      one feed-forward block: RMSNorm, gate/up projection, SwiGLU, down projection
           (ternix_hip_ffn_forward, or the _tile64 form)

Decode-sized calls are launch-bound one by one, so a serving program captures its decode step in a
graph and replays it: those cases (`graph`) hold `layers` independent layers, each with weights, inputs
and outputs of its own, captured once (what runs between the layers, attention for one, is not this
library's).  The others are single calls made from Python as they are.

Sizes are those of the library's own configurations (ternixengine_amd/configs.py) and of its benchmark's
feed-forward block; `draw` spreads over the same ranges, ragged sizes included.
"""
import math

import numpy as np
import torch

import ternixengine_amd as tx
from ternixengine_amd import _lib

EPS = 1e-5


def listed():
    return [
        # The smallest call: one token's projection, one eager call; the latency of a single launch.
        dict(name="matmul_m1", kind="matmul", M=1, K=2560, N=6912, layers=1, graph=False, tile64=False, host=False),
        # The Python module's drop-in call on numpy arrays: upload, product, download.
        dict(name="matmul_host_m16", kind="matmul", M=16, K=2560, N=6912, layers=1, graph=False, tile64=False, host=True),
        # Sixteen sequences decoded together, a stack of up projections.
        dict(name="matmul_m16", kind="matmul", M=16, K=4096, N=11008, layers=8, graph=True, tile64=False, host=False),
        # Sixty-four sequences decoded together, a stack of down projections (long K).
        dict(name="matmul_m64", kind="matmul", M=64, K=11008, N=4096, layers=8, graph=True, tile64=False, host=False),
        # A short prompt on a matrix whose sizes fit no tile.
        dict(name="matmul_ragged_m129", kind="matmul", M=129, K=8191, N=2052, layers=1, graph=False, tile64=False, host=False),
        # A mid-sized prompt chunk against a very long K.
        dict(name="matmul_m256_longk", kind="matmul", M=256, K=16384, N=4096, layers=1, graph=False, tile64=False, host=False),
        # Prefill: a long prompt, compute-bound; the largest case.
        dict(name="matmul_m2048", kind="matmul", M=2048, K=4096, N=14336, layers=1, graph=False, tile64=False, host=False),
        # A quantised linear layer for eight sequences decoded together.
        dict(name="linear_m8", kind="linear", M=8, K=4096, N=4096, layers=8, graph=True, tile64=False, host=False),
        # A quantised linear layer of a prompt, on weights laid out once at load time.
        dict(name="linear_m512_tile64", kind="linear", M=512, K=4096, N=11008, layers=1, graph=False, tile64=True, host=False),
        # The decode step of one sequence: a stack of feed-forward blocks.
        dict(name="ffn_m1", kind="ffn", M=1, K=2560, N=6912, layers=8, graph=True, tile64=False, host=False),
        # The decode step of thirty-two sequences.
        dict(name="ffn_m32", kind="ffn", M=32, K=2560, N=6912, layers=4, graph=True, tile64=False, host=False),
        # A prompt through one feed-forward block.
        dict(name="ffn_m1024", kind="ffn", M=1024, K=2560, N=6912, layers=1, graph=False, tile64=False, host=False),
    ]


# The cost of the largest listed case, which no drawn one exceeds.
_MAX_FLOPS = 2.0 * 2048 * 4096 * 14336


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges: rows from one to a long prompt, K and N from small to large,
    whole tiles or ragged, every kind and option."""
    while True:
        kind = rng.choice(("matmul", "matmul", "linear", "ffn"))
        host = kind == "matmul" and rng.random() < 0.15
        tile64 = kind != "matmul" and rng.random() < 0.3
        ragged = not tile64 and rng.random() < 0.35
        M = _log(rng, 1, 2048)
        K, N = _log(rng, 512, 16384), _log(rng, 512, 16384)
        if ragged:  # any K (a feed-forward block's hidden size is the width of two packed matrices)
            K = K // 4 * 4 if kind == "ffn" else K
            N = N // 4 * 4
        else:
            step = 256 if tile64 else rng.choice((64, 128, 256))
            K, N = max(step, K // step * step), max(256, N // 256 * 256)
        graph = not host and M <= 64
        layers = rng.choice((2, 4, 8)) if graph else 1
        case = dict(kind=kind, M=M, K=K, N=N, layers=layers, graph=graph, tile64=tile64, host=host)
        if work(case)["flops"] <= _MAX_FLOPS and (not host or M * N <= 1 << 22):
            return case


def _packed(K, N, gen):
    """Packed random ternary weights (30 % -1, 30 % +1) and nothing outside the format's codes."""
    r = torch.randint(0, 10, (4, K, N // 4), generator=gen, device="cuda", dtype=torch.uint8)
    code = (r < 3).to(torch.uint8) + 3 * (r > 6).to(torch.uint8)
    return code[0] | code[1] << 2 | code[2] << 4 | code[3] << 6


def _unpacked(packed):
    """(K, N/4) packed weights -> (K, N) float64."""
    w = torch.stack([(packed >> s) & 3 for s in (0, 2, 4, 6)], dim=-1).reshape(packed.shape[0], -1)
    return (w == 1).double() - (w == 3).double()


def _inputs(case, seed):
    """Per layer, everything the case's data consists of, from the seed alone."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    M, K, N = case["M"], case["K"], case["N"]

    def normal(*shape):
        return torch.randn(*shape, generator=gen, device="cuda")

    out = []
    for _ in range(case["layers"]):
        if case["kind"] == "matmul":  # int8 activations of a layer's width, as a quantiser leaves them
            a = (normal(M, K) * 32).round().clamp(-127, 127).to(torch.int8)
            out.append(dict(a=a, w=_packed(K, N, gen)))
        elif case["kind"] == "linear":
            out.append(dict(x=normal(M, K), w=_packed(K, N, gen), ws=1.0 / math.sqrt(0.6 * K)))
        else:
            out.append(dict(x=normal(M, K), g=1.0 + 0.1 * normal(K), wgu=_packed(K, 2 * N, gen), wd=_packed(N, K, gen),
                            ws_gu=1.0 / math.sqrt(0.6 * K), ws_d=1.0 / math.sqrt(0.6 * N)))
    return out


def _check(status):
    if status != 0:
        raise RuntimeError(f"HIP error: {tx.ternix_error(status)}")


def _tile64(packed, K, N, stream):
    out = torch.empty_like(packed)
    _check(tx.interleave_tile64_device(out.data_ptr(), packed.data_ptr(), K, N, stream))
    return out


def _calls(case, layers, stream):
    """Per layer: the calls it makes (function and arguments, addresses as numbers), its output tensor
    and the tensors that must stay alive."""
    lib = _lib.load()
    M, K, N = case["M"], case["K"], case["N"]
    dev = dict(device="cuda")
    calls, outs, keep = [], [], []
    for d in layers:
        if case["kind"] == "matmul":
            c = torch.empty(M, N, dtype=torch.int32, **dev)
            calls.append((tx.mul_mat_ternary, (d["a"].data_ptr(), d["w"].data_ptr(), c.data_ptr(), M, K, N, stream)))
            keep.append(d)
            outs.append(c)
        elif case["kind"] == "linear":
            q, rs = torch.empty(M, K, dtype=torch.int8, **dev), torch.empty(M, **dev)
            y = torch.empty(M, N, **dev)
            w = _tile64(d["w"], K, N, stream) if case["tile64"] else d["w"]
            mul = lib.ternix_hip_mul_mat_ternary_tile64_dequant if case["tile64"] else lib.ternix_hip_mul_mat_ternary_dequant
            calls.append((lib.ternix_hip_quantize_activations, (d["x"].data_ptr(), q.data_ptr(), rs.data_ptr(), M, K, stream)))
            calls.append((mul, (q.data_ptr(), w.data_ptr(), y.data_ptr(), M, K, N, rs.data_ptr(), d["ws"], stream)))
            keep.append((d, w, q, rs))
            outs.append(y)
        else:
            wgu, wd = d["wgu"], d["wd"]
            if case["tile64"]:
                wgu, wd = _tile64(wgu, K, 2 * N, stream), _tile64(wd, N, K, stream)
            nws = lib.ternix_hip_ffn_workspace_size(M, K, N)
            ws, y = torch.empty(max(nws, 256), dtype=torch.uint8, **dev), torch.empty(M, K, **dev)
            fn = lib.ternix_hip_ffn_forward_tile64 if case["tile64"] else lib.ternix_hip_ffn_forward
            calls.append((fn, (y.data_ptr(), d["x"].data_ptr(), d["g"].data_ptr(), EPS, wgu.data_ptr(), d["ws_gu"],
                               wd.data_ptr(), d["ws_d"], M, K, N, ws.data_ptr(), nws, stream)))
            keep.append((d, wgu, wd, ws))
            outs.append(y)
    return calls, outs, keep


def prepare(case, seed):
    layers = _inputs(case, seed)
    if case["host"]:
        d = layers[0]
        return dict(host=(np.ascontiguousarray(d["a"].cpu().numpy()), np.ascontiguousarray(d["w"].cpu().numpy())))
    if not case["graph"]:
        stream = torch.cuda.current_stream().cuda_stream or None
        calls, outs, keep = _calls(case, layers, stream)
        return dict(calls=calls, outs=outs, keep=keep)
    # A stream of the program's own; one eager pass (the library sizes its scratch), then the capture.
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        calls, outs, keep = _calls(case, layers, s.cuda_stream)
        for fn, args in calls:
            _check(fn(*args))
    s.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        for fn, args in calls:
            _check(fn(*args))
    return dict(graph=graph, stream=s, outs=outs, keep=keep)


def run(state):
    if "host" in state:
        return tx.ternary_matmul(*state["host"])
    if "graph" in state:
        with torch.cuda.stream(state["stream"]):
            state["graph"].replay()
        return state["outs"]
    for fn, args in state["calls"]:
        status = fn(*args)
        if status != 0:
            _check(status)
    return state["outs"]


def work(case):
    M, K, N, L = case["M"], case["K"], case["N"], case["layers"]
    if case["kind"] == "matmul":
        nbytes, flops = M * K + K * N // 4 + 4 * M * N, 2 * M * N * K
    elif case["kind"] == "linear":
        nbytes, flops = 4 * M * K + K * N // 4 + 4 * M * N, 2 * M * N * K
    else:
        nbytes, flops = 4 * M * K + 4 * K + 3 * K * N // 4 + 4 * M * K, 6 * M * N * K
    return dict(bytes=float(L * nbytes), flops=float(L * flops))


def tolerance(case):
    if case["kind"] == "matmul":
        return "exact"
    # The int8 codes of the activations: a value at a rounding boundary moves by one code under another
    # order of the same fp32 operations.  Measured against `exact`: up to 1.5e-4 for a linear layer and
    # 5.5e-4 for a block (two quantisations); on the smallest calls one code more or less in M x K of
    # them is already 1 / (30 sqrt(M K)), twice that is allowed (three times for a block).
    if case["kind"] == "linear":
        return {"rel": 6e-4 + 0.06 / math.sqrt(case["M"] * case["K"])}
    return {"rel": 2e-3 + 0.1 / math.sqrt(case["M"] * min(case["K"], case["N"]))}


def exact(case, seed):
    layers = _inputs(case, seed)

    def quantised(x):
        a = x.abs().amax(dim=1, keepdim=True).clamp(min=1e-5)
        return (x * (127.0 / a)).round().clamp(-128, 127), a / 127.0

    outs = []
    for d in layers:
        if case["kind"] == "matmul":
            outs.append((d["a"].double() @ _unpacked(d["w"])).round().to(torch.int32))
        elif case["kind"] == "linear":
            q, s = quantised(d["x"].double())
            outs.append((q @ _unpacked(d["w"])) * (s * d["ws"]))
        else:
            x = d["x"].double()
            n = x / torch.sqrt((x * x).mean(dim=1, keepdim=True) + EPS) * d["g"].double()
            q, s = quantised(n)
            y = (q @ _unpacked(d["wgu"])) * (s * d["ws_gu"])
            gate, up = y[:, 0::2], y[:, 1::2]
            q, s = quantised(gate / (1.0 + torch.exp(-gate)) * up)
            outs.append((q @ _unpacked(d["wd"])) * (s * d["ws_d"]))
    return outs[0].cpu().numpy() if case["host"] else outs
