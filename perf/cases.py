"""The workloads whose speed counts: what programs built on this library have it do, from one
small layer's matvec to a prompt's worth of rows, through the entry points they call.

Kinds of a case
  call    BCQWeight.matvec: m activation rows against one packed weight, the drop-in of
          lutGEMM::matmul(output, input, nqW, m)
  cols    BCQWeight.matvec_cols: the column-major overload of the same
  stack   MatvecSequence, one launch per entry: `layers` weights of one shape, one token through each
  block   MatvecSequence, one launch per entry: the four projections of a decoder block of width
          `hidden` (QKV, attention output, FFN up, FFN down), m rows
  many    MatvecSequence, sharing launches: `layers` independent weights of one shape (Q, K and V
          as weights of their own), m rows each
  layer   LutLinear's forward with its bias: what a torch model calls, few rows or many (many rows
          go through the dequantised weight)
  load    a LutLinear made from host arrays (pack, upload) and expanded to its dense fp16 weight

All weights use the launch plans a handle has without tuning calls.  Data: random sign planes,
|N(0, 0.02)| scales, N(0, 0.01) offsets, N(0, 1) fp16 activations, the distributions of
lutgemm.synth, drawn on the GPU.
"""
import math
import os
import sys

import torch

_PACKAGE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lut-gemm_amd")
# the package of the tree that the program runs in, wherever this file itself lies
_HERE = os.path.join(os.getcwd(), "lut-gemm_amd")
sys.path.insert(0, _HERE if os.path.isdir(_HERE) else _PACKAGE)

import lutgemm  # noqa: E402
from lutgemm import torch_ops  # noqa: E402

MAX_WEIGHT_BYTES = 350 << 20      # packed bytes of the largest listed weight
MAX_PASS_BYTES = 512 << 20        # packed bytes of all weights of a pass
MAX_FLOPS = 2 * 1024 * 7168 * 28672


def listed():
    return [
        # one token through one projection of a small model, called from torch: launch and host latency
        dict(name="layer 768 m1", kind="layer", k=768, n=768, q=4, g=128, offset=True, m=1),
        # one token, one mid-sized projection, called through the binding: the shape of the CPU reference's configuration
        dict(name="call 4096 q3 m1", kind="call", k=4096, n=4096, q=3, g=128, offset=False, m=1),
        # one token through the headline projection, weights of several layers one after the other
        dict(name="stack 12288 q3 m1", kind="stack", k=12288, n=12288, q=3, g=128, offset=False, m=1, layers=5),
        # one token through an FFN up-projection whose uniform 4-bit codes are written as planes plus an offset
        dict(name="call ffn q4 offset m1", kind="call", k=12288, n=49152, q=4, g=128, offset=True, m=1),
        # Q, K and V of one token as three independent weights in one call
        dict(name="many 3x4096 q3 m1", kind="many", k=4096, n=4096, q=3, g=128, offset=False, m=1, layers=3),
        # two sequences, fine scale groups (the bit/group sweep's shape)
        dict(name="call 7168 q3 g32 m2", kind="call", k=7168, n=7168, q=3, g=32, offset=False, m=2),
        # eight sequences through a decoder block
        dict(name="block 12288 q2 m8", kind="block", hidden=12288, q=2, g=128, offset=False, m=8),
        # a small batch in the column-major form, the shape of the reference's own test
        dict(name="cols 7168x28672 q3 m12", kind="cols", k=7168, n=28672, q=3, g=128, offset=False, m=12),
        # many sequences decoded together, called from torch
        dict(name="layer 12288 q3 m48", kind="layer", k=12288, n=12288, q=3, g=128, offset=False, m=48),
        # a short prompt through the binding
        dict(name="call 7168 q3 m256", kind="call", k=7168, n=7168, q=3, g=128, offset=False, m=256),
        # a long prompt through a torch model's FFN
        dict(name="layer 7168x28672 q4 m1024", kind="layer", k=7168, n=28672, q=4, g=128, offset=True, m=1024),
        # a layer of a checkpoint brought onto the GPU and expanded
        dict(name="load 4096x16384 q4", kind="load", k=4096, n=16384, q=4, g=128, offset=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _shapes(case):
    """(k, n) of every weight of the case."""
    if case["kind"] == "block":
        h = case["hidden"]
        return [(h, 3 * h), (h, h), (h, 4 * h), (4 * h, h)]
    return [(case["k"], case["n"])] * case.get("layers", 1)


def _weight_bytes(case, k, n):
    groups = k // case["g"] if case["g"] else 1
    return k * n * case["q"] // 8 + groups * n * 2 * (case["q"] + int(case["offset"]))


def draw(rng):
    while True:
        kind = rng.choice(["call", "call", "cols", "stack", "block", "many", "layer", "layer", "layer", "load"])
        q = rng.choice([1, 2, 2, 3, 3, 4, 4, 5, 6, 8])
        g = rng.choice([32, 64, 128, 128, 128, 256, 0])            # 0: one group per row
        case = dict(kind=kind, q=q, g=g, offset=rng.random() < 0.4)
        if kind == "block":
            # (0: a group spans all of k, which differs between the four weights)
            case["hidden"] = max(1, _log(rng, 768, 12288) // 256) * 256
            case["g"] = g or 128
        else:
            step = g or 32
            case["k"] = max(1, _log(rng, 512, 49152) // step) * step
            case["n"] = _log(rng, 100, 49152)
            if rng.random() < 0.6:
                case["n"] = max(8, case["n"] // 32 * 32)             # a model's width; the rest stay ragged
        if kind in ("stack", "many"):
            case["layers"] = rng.randint(2, 8)
        if kind == "layer":
            case["m"] = rng.choice([1, 2, _log(rng, 3, 16), _log(rng, 17, 128), _log(rng, 129, 1024)])
        elif kind == "call":
            case["m"] = rng.choice([1, 2, _log(rng, 3, 16), _log(rng, 17, 256)])
        elif kind == "cols":
            case["m"] = _log(rng, 2, 64)
        elif kind != "load":
            case["m"] = rng.choice([1, 1, 2, _log(rng, 3, 16)])
        shapes = _shapes(case)
        sizes = [_weight_bytes(case, k, n) for k, n in shapes]
        flops = sum(2 * case.get("m", 1) * k * n for k, n in shapes)
        if max(sizes) > MAX_WEIGHT_BYTES or sum(sizes) > MAX_PASS_BYTES or flops > MAX_FLOPS:
            continue
        if kind == "load" and sizes[0] > (64 << 20):
            continue
        if kind in ("call", "cols") and flops > MAX_FLOPS // 8:     # passes of 16 rows: keeps a pass within milliseconds
            continue
        return case


def _container(case, k, n, gen):
    """Host arrays of one weight as quantize.to_container returns them, drawn on the GPU."""
    q, groups = case["q"], (k // case["g"] if case["g"] else 1)
    dev = gen.device
    bits = torch.randint(0, 256, (k // 32, q, n, 4), dtype=torch.uint8, device=dev, generator=gen)
    alpha = (torch.randn(groups, q, n, device=dev, generator=gen) * 0.02).abs().half().float()
    q_bias = None
    if case["offset"]:
        q_bias = (torch.randn(groups, n, device=dev, generator=gen) * 0.01).half().float().cpu().numpy()
    return dict(bW=bits.cpu().numpy().view("<u4")[..., 0], alpha=alpha.cpu().numpy(), q_bias=q_bias, k=k, n=n, q=q,
                num_groups=groups)


def _weight(case, k, n, gen):
    c = _container(case, k, n, gen)
    return lutgemm.BCQWeight(c["bW"], c["alpha"], k, n, c["q"], c["num_groups"], c["q_bias"])


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    kind, m = case["kind"], case.get("m", 1)
    if kind == "load":
        return dict(kind=kind, container=_container(case, case["k"], case["n"], gen))

    def activations(*shape):
        return torch.randn(*shape, device=dev, generator=gen).half()

    if kind == "layer":
        bias = (torch.randn(case["n"], device=dev, generator=gen) * 0.1).half()
        layer = torch_ops.LutLinear(_container(case, case["k"], case["n"], gen), bias=bias)
        return dict(kind=kind, layer=layer, x=activations(m, case["k"]))
    if kind in ("call", "cols"):
        k, n = case["k"], case["n"]
        xy = ((m, k), (m, n)) if kind == "call" else ((k, m), (n, m))
        return dict(kind=kind, m=m, weight=_weight(case, k, n, gen), x=activations(*xy[0]),
                    y=torch.zeros(*xy[1], dtype=torch.float16, device=dev))
    # lists: the weights of a stack or a fused call hold the same numbers in memory of their own
    weights = []
    for i, (k, n) in enumerate(_shapes(case)):
        weights.append(weights[0].clone() if kind != "block" and i else _weight(case, k, n, gen))
    xs = [activations(m, k) for k, _ in _shapes(case)]
    ys = [torch.zeros(m, n, dtype=torch.float16, device=dev) for _, n in _shapes(case)]
    sequence = lutgemm.MatvecSequence([(w, x.data_ptr(), y.data_ptr(), m) for w, x, y in zip(weights, xs, ys)])
    return dict(kind=kind, sequence=sequence, xs=xs, ys=ys)


def run(state):
    kind = state["kind"]
    if kind == "layer":
        return state["layer"](state["x"])
    if kind == "load":
        return torch_ops.LutLinear(state["container"], keep_dense=True).dense_weight()
    stream = torch.cuda.current_stream().cuda_stream
    if kind in ("call", "cols"):
        call = state["weight"].matvec if kind == "call" else state["weight"].matvec_cols
        call(state["x"].data_ptr(), state["y"].data_ptr(), state["m"], stream)
        return state["y"]
    state["sequence"].launch(stream, fused=kind == "many")
    return state["ys"]


def work(case):
    m = case.get("m", 0)
    total, flops = 0, 0
    for k, n in _shapes(case):
        packed = _weight_bytes(case, k, n)
        if case["kind"] == "load":
            # signs and fp32 scales from the host, the tiles written and read, the dense weight written
            groups = k // case["g"] if case["g"] else 1
            total += k * n * case["q"] // 8 + groups * n * 4 * (case["q"] + int(case["offset"])) + 2 * packed + 2 * k * n
            continue
        total += packed + 2 * m * (k + n) + (2 * n if case["kind"] == "layer" else 0)
        flops += 2 * m * k * n
    return {"bytes": total, "flops": flops}


def tolerance(case):
    if case["kind"] == "load":
        return "exact"      # the fp32 sum in plane order, rounded once, is part of what the call promises
    # measured against 64-bit sums over the same fp16 inputs: packed weight 2.1e-4 (the fp16 result's rounding; 3.0e-4 with
    # the bias added in fp16), dense weight rounded to fp16 as well 3.6e-4; largest single difference 4.9e-4 / 1.2e-3 / 2e-3
    if case["kind"] == "layer":
        return {"rel": 1.5e-3, "max": 8e-3}
    return {"rel": 8e-4, "max": 2e-3}


def _dense64(container, device):
    """The weight of host arrays [k/32][q][n], in 64 bits: W [k][n]."""
    bits = torch.from_numpy(container["bW"].view("<i4").copy()).to(device)
    alpha = torch.from_numpy(container["alpha"]).to(device).double()
    k, n, groups = container["k"], container["n"], container["num_groups"]
    shifts = torch.arange(32, device=device, dtype=torch.int32).view(1, 32, 1)
    W = torch.zeros(groups, k // groups, n, dtype=torch.float64, device=device)
    for b in range(container["q"]):
        signs = ((bits[:, b, None, :] >> shifts) & 1).view(groups, k // groups, n)
        W += alpha[:, b, None, :] * (2 * signs - 1)
        del signs
    if container["q_bias"] is not None:
        W += torch.from_numpy(container["q_bias"]).to(device).double()[:, None, :]
    return W.view(k, n)


def exact(case, seed):
    """What run returns for the inputs of prepare(case, seed), in 64 bits and plain torch."""
    dev = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    kind, m, shapes = case["kind"], case.get("m", 1), _shapes(case)

    def activations(rows, k):
        return torch.randn(rows, k, device=dev, generator=gen).half().double()

    if kind == "load":
        return _dense64(_container(case, case["k"], case["n"], gen), dev).t()
    if kind == "layer":
        bias = (torch.randn(case["n"], device=dev, generator=gen) * 0.1).half().double()
        W = _dense64(_container(case, case["k"], case["n"], gen), dev)
        return activations(m, case["k"]) @ W + bias
    if kind == "call":
        W = _dense64(_container(case, case["k"], case["n"], gen), dev)
        return activations(m, case["k"]) @ W
    if kind == "cols":
        W = _dense64(_container(case, case["k"], case["n"], gen), dev)
        x = torch.randn(case["k"], m, device=dev, generator=gen).half().double()
        return W.t() @ x
    containers = [_container(case, k, n, gen) for k, n in (shapes if kind == "block" else shapes[:1])]
    xs = [activations(m, k) for k, _ in shapes]
    return [x @ _dense64(containers[i if kind == "block" else 0], dev) for i, x in enumerate(xs)]
