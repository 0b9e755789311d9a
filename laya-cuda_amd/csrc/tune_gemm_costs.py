"""The GEMM planner's cost constants above 512 rows (gemm.hip kForwardCosts, kReplayCosts): sweep, fit and check.

    python laya-cuda_amd/csrc/tune_gemm_costs.py sweep --seed 31 --count 700 --out <file>   (on the GPU)
    python laya-cuda_amd/csrc/tune_gemm_costs.py fit                                        (anywhere)

`sweep` times projections of widths 768 and 1,024 of random kind, depth and row count with every candidate
tile (and 1, 2, 4, 8 splits of fp32 products): graph replays over weights cold in every cache.  `fit` reads
gemm_cost_data.json.gz beside this file and prints the constants and how far their choice is from the best
tile measured.  The data holds three lists of [kind, M, N, K, [[tile, splits, us, us of the norm that adds the
splits], ...]]: "forward", stage times inside whole forwards at 21 to 31 row classes of three encoders (from a
build whose slots took their plans from the environment); "isolated", sweep --seed 31 --count 700; and
"held_out", sweep --seed 47 --count 300.
"""
import argparse
import ctypes as ct
import gzip
import json
import math
import random
import sys
from pathlib import Path

import numpy as np

HERE = Path(__file__).resolve().parent
KINDS = ["f32", "half", "gelu", "relu", "geglu", "qkv", "rope"]
# tile: (rows, columns, whether tiles past a multiple of 8 are walked across the XCDs)
TILES = {14: (64, 64, True), 31: (64, 64, False), 34: (128, 64, False), 23: (128, 64, True), 24: (64, 128, True),
         25: (128, 128, True), 18: (128, 128, True), 9: (128, 256, True), 8: (256, 128, True), 21: (256, 192, True),
         35: (256, 256, True)}
NO_ROPE = (14, 23, 24, 21)  # wave tiles of less than a head
CUS, MAX_SLABS = 256, {21: 16}


def problems(seed, count):
    rng = random.Random(seed)
    out = []
    for _ in range(count):
        d = rng.choice([768, 1024])
        kind = rng.choice(["f32", "f32", "half", "half", "gelu", "gelu", "relu", "geglu", "geglu", "qkv", "qkv", "rope",
                           "rope"])
        M = int(round(math.exp(rng.uniform(math.log(16), math.log(4096 if kind == "f32" else 65536)))))
        if kind == "half":
            M = max(M, rng.randint(600, 8000))
        if kind in ("qkv", "rope"):
            M = -(-M // 16) * 16
        inner = rng.choice([4 * d, 3 * d // 2])
        N, K = {"gelu": (4 * d, d), "relu": (4 * d, d)}.get(kind, (3 * d, d))
        if kind in ("f32", "half"):
            N, K = d, rng.choice([d, inner])
        out.append((kind, M, N, K, rng.choice(["f16", "bf16"])))
    return out


def sweep(args):
    sys.path.insert(0, str(HERE.parent))
    import torch
    from laya_cuda import _lib
    lib = _lib.load()

    def p(t):
        return ct.c_void_p(t.data_ptr()) if t is not None else None

    pool = torch.empty(300 << 20, dtype=torch.float16, device="cuda").normal_(0, 0.02)  # 600 MB of weights
    xs = torch.empty(65536 * 4096 + 4096 * 64, dtype=torch.float16, device="cuda").normal_()
    outs = torch.empty(700 << 20, dtype=torch.uint8, device="cuda")

    def time(kind, M, N, K, dtype, tile, splits):
        code, half = (_lib.F16, torch.float16) if dtype == "f16" else (_lib.BF16, torch.bfloat16)
        weights, x = pool.view(half), xs.view(half)
        n = min(64 if M < 600 else 24 if M < 8000 else 8, weights.numel() // (N * K))
        turns, w = 3 if 3 * M * K <= x.numel() else 1, N // 3
        assert M * N * (4 * splits if kind == "f32" else 2) <= outs.numel() and M * K <= x.numel()
        bias = torch.zeros(N, device="cuda") if kind not in ("f32", "geglu", "rope") else None
        cos, pos = torch.ones(1024, 32, device="cuda"), (torch.arange(M, device="cuda") % 1000).int()

        def launch(i, stream):
            a, b = p(x[(i % turns) * M * K:]), p(weights[(i % n) * N * K:])
            if kind in ("qkv", "rope"):
                tables = (p(cos), p(cos), p(pos)) if kind == "rope" else (None, None, None)
                return lib.laya_op_qkv(a, b, p(bias), p(outs), p(outs[2 * M * w:]), p(outs[4 * M * w:]), *tables, code, M,
                                       w, tile, stream)
            return lib.laya_op_linear(a, b, p(bias), p(outs), KINDS.index(kind), code, M, N, K, splits, tile, stream)

        if launch(0, ct.c_void_p(torch.cuda.current_stream().cuda_stream)) != 0:
            return None
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for i in range(n):
                launch(i, ct.c_void_p(torch.cuda.current_stream().cuda_stream))
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        graph.replay()
        us = []
        for _ in range(5 if M < 8000 else 3):
            start.record()
            graph.replay()
            end.record()
            end.synchronize()
            us.append(start.elapsed_time(end) * 1e3 / n)
        return sorted(us)[len(us) // 2]

    rows = []
    for kind, M, N, K, dtype in problems(args.seed, args.count):
        timed = []
        for tile in TILES:
            for splits in ((1, 2, 4, 8) if kind == "f32" else (1,)):
                if splits == 1 or K // 64 >= 2 * splits:
                    us = time(kind, M, N, K, dtype, tile, splits)
                    if us is not None:
                        timed.append([tile, splits, round(us, 2), 0])
        rows.append([kind, M, N, K, timed])
        print(kind, M, N, K, min((t[2], t[0], t[1]) for t in timed), flush=True)
    Path(args.out).write_text(json.dumps(rows))


def legal(tile, N, kind):
    return not (N % TILES[tile][1] or kind == "rope" and tile in NO_ROPE or kind == "f32" and tile == 35)


def features(tile, M, N, K, splits, kind):
    """What a, s, r, o, o32, q and p of gemm.hip's TileCost multiply."""
    bm, bn, across = TILES[tile]
    work = -(-M // bm) * (N // bn) * splits
    rounds, mb = -(-work // CUS), M * N * (4 * splits if kind == "f32" else 2) * 1e-6
    f32 = kind == "f32"
    return [1, rounds * -(-(K // 64) // splits), rounds - 1, 0 if f32 else mb, mb if f32 else 0,
            min(8, N // bn) * M * K * 2e-6 / math.sqrt(rounds) if across and work % 8 else 0,
            mb if kind == "rope" else 0]


def fit(data):
    from scipy.optimize import least_squares
    points = {}
    for kind, M, N, K, timed in data:
        if M > 512:
            for tile, splits, us, _ in timed:
                if tile in TILES and legal(tile, N, kind):
                    points.setdefault(tile, []).append(features(tile, M, N, K, splits, kind) + [us])
    out = {}
    for tile, rows in points.items():
        A, us = np.array(rows, float)[:, :7], np.array(rows, float)[:, 7]
        found = least_squares(lambda x: (A @ x) / us - 1, [3, .3, 1.5, .1, .1, .01, .05],
                              bounds=([0] * 7, [15, 5, 20, 3, 3, 1, 3]), loss="soft_l1", f_scale=0.2)
        out[tile] = found.x * A.any(0)
    return out


def choose(costs, M, N, K, kind):
    best = None
    for tile, cost in costs.items():
        if not legal(tile, N, kind) or K // 64 > MAX_SLABS.get(tile, 1 << 30):
            continue
        for splits in ((1, 2, 4, 8) if kind == "f32" else (1,)):
            if splits > 1 and (K // 64 < 2 * splits or M * N * 4 * splits > 16 << 20):
                break
            us = float(np.dot(cost, features(tile, M, N, K, splits, kind)))
            us += 0.12 * splits * M / 512 if kind == "f32" else 0
            if best is None or us < best[0]:
                best = (us, tile, splits)
    return best[1:]


def regret(costs, data):
    """Mean and largest ratio of the chosen launch's time to the best one's; fp32 with the norm's time."""
    ratios = []
    for kind, M, N, K, timed in data:
        if M > 512:
            total = {(t, s): us + (norm if norm else 0.12 * s * M / 512 if kind == "f32" else 0)
                     for t, s, us, norm in timed if t in TILES}
            ratios.append(total[choose(costs, M, N, K, kind)] / min(total.values()))
    return f"mean {np.mean(ratios):.4f}, largest {max(ratios):.3f} of {len(ratios)}"


def main():
    ap = argparse.ArgumentParser(description=__doc__.split("\n")[0])
    ap.add_argument("do", choices=["sweep", "fit"])
    ap.add_argument("--seed", type=int, default=31)
    ap.add_argument("--count", type=int, default=700)
    ap.add_argument("--out", default="sweep.json")
    args = ap.parse_args()
    if args.do == "sweep":
        return sweep(args)
    data = json.loads(gzip.decompress((HERE / "gemm_cost_data.json.gz").read_bytes()))
    forward, isolated, held = data["forward"], data["isolated"], data["held_out"]
    half = fit([x for i, x in enumerate(forward) if i // 4 % 2 == 0])  # every other row class, four projections each
    print("forwards, fitted to every other row class:", regret(half, [x for i, x in enumerate(forward) if i // 4 % 2]))
    print("isolated, fitted to the first sweep:", regret(fit(isolated), held))
    for name, rows in (("kForwardCosts", forward), ("kReplayCosts", isolated + held)):
        costs = fit(rows)
        print(f"{name}, fitted to everything:", regret(costs, rows))
        for tile, cost in costs.items():
            print("    {%d, 1, %s}," % (tile, ", ".join("%.3ff" % c for c in cost)))


if __name__ == "__main__":
    main()
