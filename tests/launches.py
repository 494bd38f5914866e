"""The kernels that a call launches, by the profiler's record."""
import json
import os
import tempfile

import torch


def launches(run):
    """[(name, grid, block)] of the kernels of ``run()``, in order of their start."""
    from torch.profiler import ProfilerActivity, profile

    run()                                                    # (what a first call builds)
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CPU, ProfilerActivity.CUDA]) as p:
        run()
        torch.cuda.synchronize()
    with tempfile.TemporaryDirectory() as d:
        path = os.path.join(d, "trace.json")
        p.export_chrome_trace(path)
        with open(path) as f:
            events = json.load(f)["traceEvents"]
    ks = sorted((e for e in events if e.get("cat") == "kernel"), key=lambda e: e["ts"])
    assert ks, "no kernel was recorded"
    return [(e["name"], tuple(e["args"]["grid"]), tuple(e["args"]["block"])) for e in ks]
