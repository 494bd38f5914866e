"""Decode-batch projection GEMMs (serving, Llama-2-7B and -13B, TP=1): hipBLASLt vs the decode MFMA GEMM.

For every projection shape and decode batch M (the serving graph buckets' block heights): what
``linear_nt`` runs without a plan table -- the few-row and tiled kernels where their rules take the
product, else the library GEMM y = x @ W^T with the shipped TunableOp table -- and every (BN, split-K)
plan of ``kernels/decode_gemm.hip`` for the batch's block height.  The weights rotate over copies
totalling > 512 MB, so each launch reads W from HBM as in a decode step (13 GB of weights per step; a
repeated 100 MB matrix would be served by the 256 MB Infinity Cache).  Writes the plans that beat the
library by > 3% where ``linear_nt`` leaves the product to it to ``--plans`` (the serving engine's
table, configs/kernels/decode_gemm_plans.json).

    python -m lumen.bench.decode_gemm_probe [--ms 64,128,192,256] [--plans out.json]
"""
from __future__ import annotations

import argparse
import json

import torch

SHAPES = (("qkv", 12288, 4096), ("o", 4096, 4096), ("gate_up", 22016, 4096),
          ("down", 4096, 11008), ("lm_head", 32000, 4096),
          ("qkv_13b", 15360, 5120), ("o_13b", 5120, 5120), ("gate_up_13b", 27648, 5120),
          ("down_13b", 5120, 13824), ("lm_head_13b", 32000, 5120))


def _time(fn, n_w, iters=40):
    for i in range(6):
        fn(i % n_w)
    torch.cuda.synchronize()
    s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    s.record()
    for i in range(iters):
        fn(i % n_w)
    e.record()
    torch.cuda.synchronize()
    return s.elapsed_time(e) / iters * 1000.0


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--ms", default="64,128,192,256")
    ap.add_argument("--plans", default=None, help="write winning plans here (JSON)")
    ap.add_argument("--win", type=float, default=0.97, help="plan kept if dgemm < win x library")
    a = ap.parse_args()
    from lumen.ops import gemm
    from lumen.ops.gemm import DG_BNS, DG_BNS8, decode_gemm, decoded_rows, dg_bucket, linear_nt
    from lumen.utils.gemm_tuning import load_tuned_gemms

    load_tuned_gemms()
    gemm.DGEMM = False                             # (linear_nt as it is without plans)
    dev = torch.device("cuda")
    ms = [int(x) for x in a.ms.split(",")]
    plans, rows = [], []
    tot = {}
    for name, N, K in SHAPES:
        n_w = max(2, -(-512 * 2**20 // (N * K * 2)))
        Ws = [torch.randn(N, K, device=dev, dtype=torch.bfloat16) * 0.02 for _ in range(n_w)]
        for m in ms:
            x = torch.randn(m, K, device=dev, dtype=torch.bfloat16)
            with decoded_rows():
                lib = _time(lambda i: linear_nt(x, Ws[i]), n_w)
                taken = bool(gemm.split_plan(m, N, K) or gemm.tile_ok(x, Ws[0]) or gemm.thin_ok(x, Ws[0]))
            bm = dg_bucket(m)
            best = None
            cands = [(b, 4) for b in DG_BNS[bm]] + [(b, 8) for b in DG_BNS8.get(bm, ())]
            for bn, nw in cands:
                for s in (1, 2, 3, 4, 6, 8):
                    if s > K // 64 or -(-N // bn) * s > 4 * 256:
                        continue
                    try:
                        us = _time(lambda i: decode_gemm(x, Ws[i], bm, bn, s, nw), n_w)
                    except Exception as e:  # noqa: BLE001
                        print(json.dumps({"shape": name, "M": m, "BN": bn, "S": s, "NW": nw,
                                          "error": repr(e)[:200]}), flush=True)
                        continue
                    rows.append({"shape": name, "M": m, "BM": bm, "BN": bn, "S": s, "NW": nw,
                                 "us": round(us, 2)})
                    if best is None or us < best[0]:
                        best = (us, bn, s, nw)
            ref = x.float() @ Ws[0].float().t()
            err = ((decode_gemm(x, Ws[0], bm, best[1], best[2], best[3]).float() - ref).norm()
                   / ref.norm()).item()
            rec = {"shape": name, "M": m, "N": N, "K": K, "library": not taken, "now_us": round(lib, 2),
                   "dgemm_us": round(best[0], 2), "BM": bm, "BN": best[1], "S": best[2],
                   "NW": best[3],
                   "speedup": round(lib / best[0], 3), "rel_err": round(err, 5),
                   "now_TBps": round(N * K * 2 / lib / 1e6, 2),
                   "dgemm_TBps": round(N * K * 2 / best[0] / 1e6, 2)}
            print(json.dumps(rec), flush=True)
            layers = 1 if name.startswith("lm_head") else 40 if name.endswith("13b") else 32
            t = tot.setdefault((name.endswith("13b"), m), [0.0, 0.0])
            win = not taken and best[0] < a.win * lib
            t[0] += lib * layers
            t[1] += (best[0] if win else lib) * layers
            if win:
                plans.append({"N": N, "K": K, "BM": bm, "BN": best[1], "S": best[2],
                              "NW": best[3], "M_measured": m, "us": round(best[0], 2), "lib_us": round(lib, 2)})
        del Ws
        torch.cuda.empty_cache()
    for (wide, m), (l, d) in sorted(tot.items()):
        print(json.dumps({"model": "13b" if wide else "7b", "M": m, "step_projections_ms_now": round(l / 1e3, 3),
                          "step_projections_ms_planned": round(d / 1e3, 3)}), flush=True)
    for r in rows:
        print(json.dumps(dict(r, sweep=True)))
    if a.plans:
        # one plan per (N, K, BM): the measured M of each bucket is its block height
        with open(a.plans, "w") as f:
            json.dump({"source": "lumen/bench/decode_gemm_probe.py (weights rotated over "
                                 "> 512 MB: HBM-resident like a decode step)",
                       "plans": plans}, f, indent=1)


if __name__ == "__main__":
    main()
