"""Regenerate gemm_plans.inc: measured (tile, split-K) launches of laya_op_linear's fp32 products.

For every encoder shape family below, every packed-row class up to 2,048 rows (the classes
laya_cuda.runtime rounds requests to) and both MFMA input types, each fp32 product of a forward is timed
through laya_op_linear with every tile id and 1, 2, 4 and 8 splits, and with the library's heuristic plan
(tile -2); the launches take twelve input and weight matrices in turn, so each reads its operands from
beyond L2 as a forward does.  A problem gets a table row only when the best measured launch beats the
heuristic by more than 3%; laya_op_linear's tile -1 looks rows up (exact match on CUs, M, N, K, type).

Run on the target GPU from the repository root, then rebuild:
    python laya-cuda_amd/csrc/tune_gemm_plans.py [--out path]
"""
import argparse
import ctypes as ct
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parents[2]
sys.path.insert(0, str(ROOT / "laya-cuda_amd"))

import torch  # noqa: E402

from laya_cuda import _lib  # noqa: E402

DTYPE_ID = {"f16": 1, "bf16": 2}  # kernels.hpp DType

LAYERS = 12  # weight matrices timed in turn

# (name, width d, depths of the out and down projections)
FAMILIES = [("bert-768", 768, (768, 3072)), ("bert-1024", 1024, (1024, 4096)), ("modernbert-768", 768, (768, 1152, 3072))]


def row_classes(limit=2048):
    """Packed-row classes of laya_cuda.runtime._round_rows up to `limit`."""
    out, m = [], 32
    while m <= limit:
        out.append(m)
        m += 32 if m < 256 else 64 if m < 512 else 128
    return out


def main():
    ap = argparse.ArgumentParser(description=__doc__.split("\n")[0])
    ap.add_argument("--out", default=str(Path(__file__).with_name("gemm_plans.inc")))
    ap.add_argument("--max-rows", type=int, default=2048)
    args = ap.parse_args()
    lib = _lib.load()
    dev = torch.device("cuda:0")
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    stream = ct.c_void_p(torch.cuda.current_stream().cuda_stream)
    p = lambda t: ct.c_void_p(t.data_ptr()) if t is not None else None
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)

    def timed(call):
        """Best of three timings of five back-to-back launches (us per launch); None if refused."""
        if call() != 0:
            return None
        best = None
        for _ in range(3):
            start.record()
            for _ in range(5):
                call()
            end.record()
            end.synchronize()
            us = start.elapsed_time(end) * 1e3 / 5
            best = us if best is None else min(best, us)
        return best

    rows, seen, began = [], set(), time.time()
    maxm = args.max_rows
    for name, N, depths in FAMILIES:
        for dtype in ("f16", "bf16"):
            tdt = torch.float16 if dtype == "f16" else torch.bfloat16
            lib_dtype = _lib.F16 if dtype == "f16" else _lib.BF16
            for K in depths:
                # One input and one weight matrix per layer, used in turn: as in a forward, each launch
                # reads operands that are not in its L2 (a loop over one pair would time L2-resident ones).
                xs = [torch.zeros(maxm, K, device=dev, dtype=tdt) for _ in range(LAYERS)]
                ws = [(torch.randn(N, K, device=dev) * 0.02).to(tdt) for _ in range(LAYERS)]
                turn = [0]
                out = torch.zeros(8 * maxm * N, device=dev)  # up to eight partials
                for M in row_classes(maxm):
                    key = (M, N, K, dtype)
                    if key in seen:  # the same problem in another family: measured once
                        continue
                    seen.add(key)

                    def launch(tile, splits):
                        def call():
                            x, w = xs[turn[0] % LAYERS], ws[turn[0] % LAYERS]
                            turn[0] += 1
                            return lib.laya_op_linear(p(x), p(w), None, p(out), 0, lib_dtype, M, N, K, splits, tile, stream)
                        return call
                    heuristic = timed(launch(-2, 1))
                    best = None
                    for tile in range(64):  # ids past the tile menu are refused (not timed)
                        for splits in (1, 2, 4, 8):
                            if splits > 1 and K // 64 // splits < 2:
                                continue
                            us = timed(launch(tile, splits))
                            if us is not None and (best is None or us < best[0]):
                                best = (us, tile, splits)
                    if heuristic is None or best is None:
                        continue
                    gain = 1 - best[0] / heuristic
                    if gain > 0.03:
                        rows.append((cus, M, N, K, DTYPE_ID[dtype], best[1], best[2], heuristic, best[0]))
                    print(f"{name} {dtype} M={M} N={N} K={K}: heuristic {heuristic:.2f} us, "
                          f"best t{best[1]} s{best[2]} {best[0]:.2f} us ({gain * 100:+.1f}%)", flush=True)
                del xs, ws, out
                torch.cuda.empty_cache()
    with open(args.out, "w") as fh:
        fh.write("// Measured plans of the fp32 split-K projections: {CUs, M, N, K, epilogue, MFMA type, RoPE, tile,\n"
                 f"// splits}}, at packed-row classes up to {maxm:,} rows, timed on {torch.cuda.get_device_name(0)} ({cus} CUs) "
                 "through\n// laya_op_linear with the tiles and 1/2/4/8 splits against the heuristic plan (tile -2); a row is kept\n"
                 "// where the best measured launch beat the heuristic by more than 3% (heuristic -> measured us per\n"
                 "// launch).  Forwards take their plans from the cost model (gemm.hip); these rows serve\n"
                 "// laya_op_linear's tile -1 with fp32 output, whose callers sum as many partials as the row splits.\n"
                 "// Regenerate with tune_gemm_plans.py, then rebuild the library.\n")
        for cus_, M, N, K, dt, tile, splits, h, b in rows:
            fh.write(f"    {{{cus_}, {M}, {N}, {K}, 0, {dt}, 0, {tile}, {splits}}},  // {h:.2f} -> {b:.2f}\n")
    print(f"{len(rows)} plans written to {args.out} in {time.time() - began:.0f} s", flush=True)


if __name__ == "__main__":
    main()
