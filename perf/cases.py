"""The work a user of this library has it do, as measurable cases: one sparse product (SpMM) or one sparse
convolution per pass, through the operator classes of the package.

A weight is pruned and laid out once and serves many calls, so `prepare` holds it on the device together with the
activations.  A program with fixed buffers also initialises the operator once (`"bind": "kept"`); one whose
activations move from call to call - an eager program with a caching allocator - initialises the operator for its
fresh output on every call (`"bind": "each"`), and then the initialisation is part of the pass.
"""
import math

import numpy as np
import torch

import shflbw_sparse_nn_amd as S


def listed():
    return [
        # ---- SpMM: D[M x N] = A_sparse[M x K] * B[K x N] (+ C), N counts tokens or samples
        # the small square problem of the benchmark: a launch or two of latency decides
        _spmm("small square", M=1024, K=1024, N=1024, V=64, d=0.25),
        # decoding: one projection for the fewest tokens the format takes, weight-bound
        _spmm("decode, 8 tokens", M=4096, K=4096, N=8, V=32, d=0.1),
        # decoding in an eager program: a small batch of tokens, fresh output and initialisation on every call
        _spmm("decode, eager", M=3072, K=768, N=32, V=64, d=0.2, bind="each"),
        # the benchmark's headline problem: an FFN or projection over a few thousand tokens
        _spmm("square 4096", M=4096, K=4096, N=4096, V=64, d=0.1),
        # short inner dimension and block height 32 (the second large problem of the benchmark)
        _spmm("short inner", M=4096, K=1024, N=4096, V=32, d=0.2),
        # tall, ragged, finest blocks, rows not permuted: an output vocabulary or embedding-like layer
        _spmm("tall ragged", M=33728, K=777, N=1000, V=16, d=0.1, permute=False),
        # the largest: prefill over many tokens with the residual added (D = A B + C), coarsest blocks
        _spmm("prefill, residual", M=8192, K=4096, N=16384, V=128, d=0.1, residual=True),
        # ---- convolution, "same" padding; H and W are input extents
        # the benchmark's two layers of a residual network: many filters at low density; stride 2 at higher density
        _conv("conv 14x14 wide", B=16, H=14, W=14, C=512, F=2048, R=3, S=3, stride=1, V=64, d=0.1),
        _conv("conv stride 2", B=32, H=28, W=28, C=256, F=512, R=3, S=3, stride=2, V=32, d=0.3),
        # the same operator over batch-innermost tensors (C-H-W-B in, F-H-W-B out), a large batch
        _conv("conv batch innermost", B=128, H=14, W=14, C=256, F=256, R=3, S=3, stride=1, V=64, d=0.1, layout="chwb"),
        # one image at a time in an eager program: the smallest convolution call
        _conv("conv one image, eager", B=1, H=28, W=28, C=128, F=128, R=3, S=3, stride=1, V=32, d=0.25, bind="each"),
        # 1x1 expansion of a bottleneck: little arithmetic, the activations decide
        _conv("conv 1x1 expand", B=16, H=56, W=56, C=64, F=256, R=1, S=1, stride=1, V=64, d=0.25),
    ]


def draw(rng):
    """One more case of the same ranges, at most as costly as the largest listed one."""
    while True:
        case = _draw_spmm(rng) if rng.random() < 0.55 else _draw_conv(rng)
        if _cost_ok(case):
            return case


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    host = np.random.default_rng(seed)
    conv = case["op"] == "conv"
    rows = case["F"] if conv else case["M"]
    cols = case["R"] * case["S"] * case["C"] if conv else case["K"]
    V = case["V"]
    nnzb, indptr, indices = S.random_mask(rows, cols, V, 1, case["d"], seed % (1 << 20))
    fan_in = max(1.0, nnzb / (rows // V))  # kept columns per row: outputs of unit scale
    values = (host.standard_normal(nnzb * V, dtype=np.float32) / math.sqrt(fan_in)).astype(np.float16)
    perm = host.permutation(rows).astype(np.int32) if case["permute"] else None

    def randn(*shape):
        return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float16)

    state = {"case": case, "stream": torch.cuda.current_stream().cuda_stream}
    if conv:
        B, H, W, C, F = (case[k] for k in ("B", "H", "W", "C", "F"))
        weight = S.BlockwiseSpFilter()
        weight.set(rows, cols, V, 1, indptr, indices, values, perm, case["R"], case["S"], C)
        chwb = case["layout"] == "chwb"
        Ho, Wo = _out_extents(case)
        state["x"] = randn(C, H, W, B) if chwb else randn(B, H, W, C)
        state["shape"] = (F, Ho, Wo, B) if chwb else (B, Ho, Wo, F)
        state["op"] = S.SpconvBlockwiseOp()
    else:
        weight = S.BlockwiseSpMatrix()
        weight.set(rows, cols, V, 1, indptr, indices, values, perm)
        state["x"] = randn(cols, case["N"])
        state["c"] = randn(rows, case["N"]) if case["residual"] else None
        state["shape"] = (rows, case["N"])
        state["op"] = S.SpmmBlockwiseOp()
    weight.transform_and_sync_device()
    state["weight"] = weight
    state["out"] = None
    if case["bind"] == "kept":
        state["out"] = torch.empty(state["shape"], dtype=torch.float16, device="cuda")
        _initialize(state, state["out"])
    return state


def run(state):
    out = state["out"]
    if out is None:
        out = torch.empty(state["shape"], dtype=torch.float16, device="cuda")
        _initialize(state, out)
    state["op"](state["stream"])
    return out


def work(case):
    conv = case["op"] == "conv"
    rows = case["F"] if conv else case["M"]
    cols = case["R"] * case["S"] * case["C"] if conv else case["K"]
    nnzb = _kept(case)
    weight = nnzb * case["V"] * 2 + (nnzb + rows // case["V"] + 1 + (rows if case["permute"] else 0)) * 4
    if conv:
        Ho, Wo = _out_extents(case)
        n = case["B"] * Ho * Wo
        # pixels that some tap reads
        h = case["H"] if case["R"] >= case["stride"] else min(case["H"], Ho * case["R"])
        w = case["W"] if case["S"] >= case["stride"] else min(case["W"], Wo * case["S"])
        dense = case["B"] * h * w * case["C"] + n * rows
    else:
        n = case["N"]
        dense = cols * n + rows * n * (2 if case["residual"] else 1)
    return {"bytes": weight + 2 * dense, "flops": 2 * nnzb * case["V"] * n}


def tolerance(case):
    # fp16 in and out, fp32 sums: a result differs where another order of the sum rounds to the neighbouring fp16 value
    # (2^-10 of the value), by two of those at most where the residual is added to a rounded product
    return {"rel": 1e-3, "max": 4e-3}


# ---------------------------------------------------------------------------------------
def _spmm(name, M, K, N, V, d, permute=True, residual=False, bind="kept"):
    case = dict(op="spmm", M=M, K=K, N=N, V=V, d=d, permute=permute, residual=residual, bind=bind)
    return dict(case, name=name) if name else case


def _conv(name, B, H, W, C, F, R, S, stride, V, d, permute=True, layout="nhwc", bind="kept"):
    case = dict(op="conv", B=B, H=H, W=W, C=C, F=F, R=R, S=S, stride=stride, V=V, d=d, permute=permute, layout=layout,
                bind=bind)
    return dict(case, name=name) if name else case


def _initialize(state, out):
    case, x = state["case"], state["x"]
    if case["op"] == "conv":
        state["op"].initialize(state["weight"], case["B"], case["H"], case["W"], case["stride"], x.data_ptr(),
                               out.data_ptr(), batch_innermost=case["layout"] == "chwb")
    else:
        c = state["c"]
        state["op"].initialize(state["weight"], case["N"], x.data_ptr(), out.data_ptr(), None if c is None else c.data_ptr())


def _out_extents(case):
    if case["layout"] == "chwb":  # the extents bound input and output alike
        return case["H"], case["W"]
    return tuple((case[e] + 2 * (case[k] // 2) - case[k]) // case["stride"] + 1 for e, k in (("H", "R"), ("W", "S")))


def _kept(case):
    """Kept V x 1 vectors of the weight."""
    conv = case["op"] == "conv"
    rows = case["F"] if conv else case["M"]
    cols = case["R"] * case["S"] * case["C"] if conv else case["K"]
    return int(round(case["d"] * (rows // case["V"]) * cols))


def _log_uniform(rng, lo, hi, step=1):
    return max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step)


def _draw_spmm(rng):
    V = rng.choice([16, 32, 32, 64, 64, 128])
    return _spmm(None, M=_log_uniform(rng, 512, 33792, V) // V * V, K=_log_uniform(rng, 64, 8192), N=_log_uniform(rng, 8, 16384, 8),
                 V=V, d=round(math.exp(rng.uniform(math.log(0.02), math.log(0.5))), 3), permute=rng.random() < 0.8,
                 residual=rng.random() < 0.2, bind="each" if rng.random() < 0.25 else "kept")


def _draw_conv(rng):
    V = rng.choice([16, 32, 32, 64, 64, 128])
    layout = "chwb" if rng.random() < 0.2 else "nhwc"
    B = _log_uniform(rng, 8, 128, 8) if layout == "chwb" or rng.random() < 0.5 else _log_uniform(rng, 1, 64)
    R, Sx = rng.choice([(3, 3), (3, 3), (3, 3), (1, 1), (1, 1), (5, 5), (1, 7)])
    H = _log_uniform(rng, 5, 56)
    W = H if rng.random() < 0.6 else _log_uniform(rng, 5, 56)
    return _conv(None, B=B, H=H, W=W, C=_log_uniform(rng, 16, 1024, 8), F=_log_uniform(rng, V, 2048, V), R=R, S=Sx,
                 stride=1 if rng.random() < 0.7 else 2, V=V, d=round(math.exp(rng.uniform(math.log(0.05), math.log(0.5))), 3),
                 permute=rng.random() < 0.8, layout=layout, bind="each" if rng.random() < 0.25 else "kept")


def _cost_ok(case):
    """Bytes, and kept vectors times columns (what the block height cannot help with), within the largest listed case."""
    largest = next(c for c in listed() if c["name"] == "prefill, residual")

    def cost(c):
        w = work(c)
        return w["bytes"], w["flops"] / c["V"]
    return all(a <= b for a, b in zip(cost(case), cost(largest)))
