"""Draws, times and fits the problems behind the estimate by which the library chooses the variant of an SpMM (the tables
g_role_split_estimates, g_slab_estimates and g_split_estimates in csrc/device.hip).

    python profiles/spmm_estimate_fit.py measure SEED OUT     on the GPU: 4620 problems, every variant of the tables, one to two minutes
    python profiles/spmm_estimate_fit.py check OUT...         the library's choice as it was when OUT was timed, against the fastest
    python profiles/spmm_estimate_fit.py fit V OUT...         weights for block height V, as rows of the tables

The tables hold what `fit` gave for seeds 1000, 2000 and 3000; seeds from 6000 on were timed with the library that holds the tables.
"""
import json
import math
import os
import random
import re
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
CUS = 256
FLOOR = 3.4  # us per launch, however little it does


# ---- problems ------------------------------------------------------------------------------------------------------
def problems(kind, n, seed):
    """`draw`: the SpMM cases of perf/cases.py; `edge`: long panels, tiles a little more than the compute units or twice as many;
    `wide`: few rows, many columns, as convolutions have them; `large`: up to four times the cost of the largest listed case."""
    from perf import cases as C
    rng, out = random.Random(seed), []
    largest = next(c for c in C.listed() if c["name"] == "prefill, residual")

    def cost(c):
        w = C.work(c)
        return w["bytes"], w["flops"] / c["V"]

    def spmm(rows, cols, n_cols, densities):
        V = rng.choice([16, 32, 32, 64, 64, 128])
        return C._spmm(None, M=C._log_uniform(rng, rows[0] or V, rows[1], V) // V * V, K=C._log_uniform(rng, *cols), N=C._log_uniform(rng, *n_cols, 8),
                       V=V, d=round(math.exp(rng.uniform(*map(math.log, densities))), 3))

    while len(out) < n:
        if kind == "draw":
            c = C._draw_spmm(rng)
        elif kind == "edge":
            c = spmm((512, 8192), (1024, 8192), (256, 8192), (0.05, 0.5))
            per_cu = c["M"] // c["V"] * -(-c["N"] // rng.choice([128, 256, 512])) / CUS
            if not (1.0 < per_cu < 1.6 or 2.0 < per_cu < 2.4):
                continue
        elif kind == "wide":
            c = spmm((0, 4096), (64, 16384), (64, 131072), (0.02, 0.5))
        else:
            c = spmm((512, 65536), (64, 16384), (256, 65536), (0.02, 0.5))
        if kind in ("wide", "large") and c["K"] * c["N"] * 2 > 2 ** 31:
            continue
        fits = all(a <= (4 if kind == "large" else 1) * b for a, b in zip(cost(c), cost(largest)))
        if fits and not (kind == "large" and C._cost_ok(c)):
            out.append(c)
    return out


def measure(seed, path):
    import numpy as np
    import torch
    import shflbw_sparse_nn_amd as S
    with open(os.path.join(ROOT, "shflbw_sparse_nn_amd", "csrc", "device.hip")) as f:
        known = set(re.findall(r'^    \{"((?:ws|slab|split)\w+)",', f.read(), re.M))
    stream = torch.cuda.current_stream().cuda_stream

    def window(ops, n):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        for i in range(n):
            ops[i % 3](stream)
        b.record()
        b.synchronize()
        return a.elapsed_time(b) * 1e3 / n

    with open(path, "w") as out:
        for kind, n, at, residual in (("draw", 2200, 1, False), ("edge", 700, 2, False), ("wide", 700, 3, False), ("draw", 900, 4, True),
                                      ("large", 120, 5, False)):
            for i, c in enumerate(problems(kind, n, seed + at)):
                M, K, N, V = (c[k] for k in "MKNV")
                nnzb, indptr, indices = S.random_mask(M, K, V, 1, c["d"], ((seed + at) * 7919 + i) % (1 << 20))
                values = np.resize(np.random.default_rng(i).standard_normal(1 << 16, dtype=np.float32).astype(np.float16), nnzb * V)
                w = S.BlockwiseSpMatrix()
                w.set(M, K, V, 1, indptr, indices, values, np.random.default_rng(i).permutation(M).astype(np.int32) if c["permute"] else None)
                w.transform_and_sync_device()
                half = dict(device="cuda", dtype=torch.float16)
                sets = [(torch.randn(K, N, **half), torch.empty(M, N, **half), torch.randn(M, N, **half) if residual else None) for _ in range(3)]
                names, ready, taken = S.spmm_variants(V), {}, None
                for v in [-1] + [j for j, name in enumerate(names) if name in known]:
                    if v >= 0 and (names[v].startswith("split") and N > 1024 or names[v].startswith("slab") and K > 1128):
                        continue
                    ops = [S.SpmmBlockwiseOp(v) for _ in sets]
                    for op, (b, d, cc) in zip(ops, sets):
                        state = op.initialize(w, N, b.data_ptr(), d.data_ptr(), None if cc is None else cc.data_ptr())
                    if v < 0:
                        taken = names[state.variant]
                    else:
                        ready[names[v]] = ops
                n_of = {name: max(6, min(90, int(500 / max(3.0, window(ops, 6)))) // 3 * 3) for name, ops in ready.items()}
                got = {name: [] for name in ready}
                for _ in range(7):
                    for name, ops in ready.items():
                        got[name].append(window(ops, n_of[name]))
                out.write(json.dumps(dict(M=M, K=K, N=N, V=V, d=c["d"], nnzb=int(nnzb), kind=kind, residual=residual, taken=taken,
                                          us={name: round(sorted(t)[3], 3) for name, t in got.items()})) + "\n")
                if i % 100 == 0:
                    out.flush()
                    print(kind, i, flush=True)


# ---- the estimate, as in csrc/device.hip -----------------------------------------------------------------------------
TWO_PER_CU = {"ws16x64x2c4p_k32_s6", "ws16x64x4c4p_k32_s4", "ws32x64x4c4p_k32_s3", "ws32x32x4c4p_k32_s6", "ws64x32x4c4p_k32_s4",
              "ws64x64x4c4p_k32_s3", "ws128x32x4c4p_k32_s4"}


def kind_of(name):
    return "slab" if name[1] == "l" else "split" if name[1] == "p" else "two" if name in TWO_PER_CU else "one"


def slab_deal(V, X, K, groups, n_tiles):
    least, batches = (X * V + 4095) // 4096, 2.0 * groups / X
    t_slab, t_panel = 1.0 + 1.5e-3 * K, 0.30 + 0.12 * batches if V == 16 else 0.45 + 0.21 * batches
    best, best_t = None, 0.0
    for r in (1, 2, 3):
        chunks = min(max(CUS * r // n_tiles, least, 1), X)
        rounds, panels = ((n_tiles * chunks + 7) // 8 * 8 + CUS - 1) // CUS, (-(-X // chunks) + 7) // 8
        t = rounds * (t_slab + panels * t_panel)
        if r == 1 or t < best_t * 0.95:
            best, best_t = (rounds, panels), t
    return best


def features(p, name):
    """Sizes of the parts of the estimate; the D terms by the way D is stored and what exceeds the Infinity Cache."""
    V, N, X = p["V"], p["N"], p["M"] // p["V"]
    vectors, t_d, c, kind = p["nnzb"] / X, 2.0 * p["M"] * N / 5e6, float(p["residual"]), kind_of(name)
    d_bytes, lines = 2 * p["M"] * N, N * 2 % 128 == 0
    all_bytes = d_bytes * (2 if p["residual"] else 1) + 2 * p["K"] * N
    half_lines = re.match(r"ws(32|64|128)x32x4c", name) and d_bytes >= 24 << 20
    mode = (2 if d_bytes >= 96 << 20 else 0) if lines else (1 if all_bytes >= 80 << 20 or half_lines else 0)
    D = [t_d * (mode == m) for m in range(3)] + [max(0.0, t_d - 53.7)]
    if kind == "slab":
        batches = 2 * math.ceil(vectors / 64)
        rounds, panels = slab_deal(V, X, p["K"], X * math.ceil(vectors / 64), -(-N // 64))
        return [rounds, rounds * p["K"] / 1000, rounds * panels, rounds * panels * batches] + D + [c * t_d, c * rounds * panels]
    if kind == "split":
        blocks = p["M"] / (16 if V == 16 else 32)
        wide = V != 16 and N > 32 and blocks * -(-N // 32) > CUS
        grid = math.ceil(blocks / 8) * 8 * -(-N // (64 if wide else 32))
        waves = 16 if grid <= CUS else 8
        steps = vectors / (32 if V == 16 else 16) / waves + 0.5
        mean = max(1.0, grid / (CUS if waves == 16 else 2 * CUS))
        rounds = 0.5 * (mean + math.ceil(mean))
        return [rounds, rounds * steps, rounds * steps * wide, t_d, c * t_d, c * rounds]
    width = int(re.match(r"ws\d+x(\d+)x(\d+)c", name).group(1)) * int(re.match(r"ws\d+x(\d+)x(\d+)c", name).group(2))
    return [X * -(-N // width) / CUS, vectors / 32 + 0.5] + D + [c * t_d, c]


START = {"one": [2.8, .8, .2, .5, .4, .5, .1, .8, .2],                      # base tile stage, D, c c_tile
         "two": [2.8, .8, .2, .5, .4, .5, .1, .8, .2, .3, .5, .8],          # ... second: start tile stage
         "slab": [2.2, 1.3, .5, .1, .15, .8, .8, .8, .1, 1., .05],          # base slab row panel batch, D, c c_panel
         "split": [2.4, 1.1, .6, .2, .8, .8, .1]}                           # base tile step wide_step d c c_round


def predict(torch, kind, F, q):
    if kind in ("slab", "split"):
        return q[0] + F @ q[1:]
    mean, stages, n = F[:, 0].clamp(min=1.0), F[:, 1], torch.ceil(F[:, 0])
    tiles = count = n
    if kind == "two":
        tiles = torch.where(mean <= 2, 1 + (mean - 1) * q[10], mean / 2 * (1 + q[10]))
        count = torch.floor(n / 2) * (1 + q[11]) + n - 2 * torch.floor(n / 2)
    t = q[0] + q[1] * tiles + q[2] * stages * count + F[:, 2:6] @ q[3:7] + q[7] * F[:, 6] + q[8] * F[:, 7] * tiles
    return t + q[9] * (n >= 2) if kind == "two" else t


def fit(V, data):
    """First near the measured times (variants far from the fastest count little), then more and more for the time of the variant
    with the least estimate."""
    import torch
    torch.set_default_dtype(torch.float64)
    names = sorted({name for p in data for name in p["us"]})
    theta = {name: torch.log(torch.expm1(torch.tensor(START[kind_of(name)]))).requires_grad_() for name in names}
    rows = {}
    for name in names:
        idx = [j for j, p in enumerate(data) if name in p["us"]]
        rows[name] = (torch.tensor(idx), torch.tensor([features(data[j], name) for j in idx]), torch.tensor([data[j]["us"][name] for j in idx]))
    us = torch.full((len(data), len(names)), float("inf"))
    for j, name in enumerate(names):
        us[rows[name][0], j] = rows[name][2]
    best = us.min(1).values
    loss_of = torch.where(torch.isinf(us), torch.zeros_like(us), us / best[:, None] - 1).clamp(max=1.5)
    for steps, weight, tau, lr in ((2500, 0, 1, .03), (2500, 10, .04, .03), (1200, 30, .03, .01), (1200, 60, .02, .01), (2400, 100, .015, .01),
                                   (2400, 200, .01, .01)):
        opt = torch.optim.Adam(theta.values(), lr=lr)
        for step in range(steps):
            if step == steps * 6 // 10:
                opt.param_groups[0]["lr"] = lr * .3
            loss, logs = 0, []
            for name in names:
                idx, F, t = rows[name]
                raw = predict(torch, kind_of(name), F, torch.nn.functional.softplus(theta[name]))
                error = torch.log(torch.logaddexp(raw * 6, torch.full_like(raw, FLOOR * 6)) / 6 / t)
                near = torch.exp(-2.0 * (t / best[idx] - 1).clamp(0, 2))
                loss = loss + (near * torch.nn.functional.smooth_l1_loss(error, torch.zeros_like(error), beta=.1, reduction="none")).sum() * 10 / len(data)
                logs.append(torch.full((len(data),), 50.0).index_put((idx,), torch.log(raw)))
            if weight:
                loss = loss + weight * 10 * (torch.softmax(-torch.stack(logs, 1) / tau, 1) * loss_of).sum(1).mean()
            opt.zero_grad()
            loss.backward()
            opt.step()
    return {name: [float("%.3g" % x) if x >= .004 else 0.0 for x in torch.nn.functional.softplus(theta[name]).tolist()] for name in names}


def table(weights):
    def f(x):
        return "%.3g" % x + ("f" if "." in "%.3g" % x else ".f")

    lines = []
    for name, q in weights.items():
        q, kind = [f(x) for x in q], kind_of(name)
        at = 3 if kind in ("one", "two") else 5
        if kind != "split":
            q = q[:at] + ["{" + ", ".join(q[at:at + 4]) + "}"] + q[at + 4:]
        if kind == "two":
            q = q[:6] + ["{" + ", ".join(q[6:]) + "}"]
        lines.append('    {"%s", %s},' % (name, ", ".join(q)))
    return "\n".join(lines)


def report(label, data, choice):
    for V in (16, 32, 64, 128, 0):
        part = [p for p in data if V in (0, p["V"])]
        r = [p["us"][choice(p)] / min(p["us"].values()) for p in part]
        if r:
            print("%s: block height %s, %d problems: %.4f times the fastest (geometric mean), %.2f at worst, more than 1.1 times on %d; %.0f us, fastest %.0f" % (
                label, V or "any", len(r), math.exp(sum(map(math.log, r)) / len(r)), max(r), sum(x > 1.1 for x in r),
                sum(p["us"][choice(p)] for p in part), sum(min(p["us"].values()) for p in part)))


def load(paths):
    data = []
    for path in paths:
        with open(path) as f:
            data += [json.loads(line) for line in f]
    return data


if __name__ == "__main__":
    if sys.argv[1] == "measure":
        measure(int(sys.argv[2]), sys.argv[3])
    elif sys.argv[1] == "check":
        for kind in ("draw", "edge", "wide", "large", ""):
            data = [p for p in load(sys.argv[2:]) if kind in ("", p["kind"])]
            report(kind or "all", data, lambda p: p["taken"])
    else:
        V = int(sys.argv[2])
        data = [p for p in load(sys.argv[3:]) if p["V"] == V]
        weights = fit(V, data)
        import torch
        q = {name: torch.tensor(v) for name, v in weights.items()}

        def choice(p):
            return min(p["us"], key=lambda name: float(predict(torch, kind_of(name), torch.tensor([features(p, name)]), q[name])))
        print(table(weights))
        report("fitted", data, choice)
