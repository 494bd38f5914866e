"""The scans whose chunks are built ahead (seqmix/head_scan_ahead.hip) against the token loops of the oracle: portions that end on
and beside a chunk, sequences that start and go on, decoded rows behind them, head sizes on and off the blocks of 32."""
import pytest
import torch

from lumen.ops import _seqmix
from test_silonex_ops import run_scan, step_of

pytestmark = pytest.mark.gpu


def routed(monkeypatch, run):
    names, call = [], _seqmix.call
    monkeypatch.setattr(_seqmix, "call", lambda name, *a: (names.append(name), call(name, *a))[1])
    run()
    monkeypatch.undo()
    return names


@pytest.mark.parametrize("kind", ["ssd", "delta", "const"])
@pytest.mark.parametrize("H,G,Dk,Dv", [(4, 2, 16, 24), (3, 3, 64, 64), (10, 2, 33, 40), (6, 1, 128, 128), (2, 1, 96, 8), (1, 1, 32, 96)])
def test_chunks_built_ahead(monkeypatch, H, G, Dk, Dv, kind):
    spans, slots = [(0, 96), (40, 129), (5, 97), (0, 64), (9, 1), (0, 1)], [2, 0, 5, 7, 1, 4]
    seg, cu = step_of(spans, slots, 4, "cuda")
    kw = dict(silu_in=True, decay=[0.0, 1.0, 0.5, 0.999, 0.9, 0.99][:H]) if kind == "const" else dict(scale=0.5)
    if kind == "const" and H > 6:
        kw["decay"] = [0.0, 1.0] + [0.9 + 0.01 * i for i in range(H - 2)]
    names = routed(monkeypatch, lambda: run_scan(kind, seg, cu, spans, slots, H, H if kind == "const" else G, Dk, Dv, "cuda", torch.bfloat16, **kw))
    assert names == ["sm_head_scan_ahead", "sm_head_scan_step"]


@pytest.mark.parametrize("kind", ["ssd", "delta"])
@pytest.mark.parametrize("shift", [30.0, -12.0])
@pytest.mark.parametrize("rows", [96, 300, 1000])
def test_one_long_portion_of_extreme_steps(monkeypatch, rows, shift, kind):
    seg, cu = step_of([(7, rows)], [3], None, "cuda")
    names = routed(monkeypatch, lambda: run_scan(kind, seg, cu, [(7, rows)], [3], 4, 2, 128, 64, "cuda", torch.bfloat16, scale=0.3, a_shift=shift))
    assert names == ["sm_head_scan_ahead"]


@pytest.mark.parametrize("lens,H,Dv,ahead", [([95], 4, 32, False), ([96], 4, 32, True), ([100, 91], 4, 32, False), ([96] * 4, 16, 128, True),
                                             ([96] * 4, 17, 128, False), ([200], 4, 36, False), ([200], 3, 32, True)])
def test_the_rule(monkeypatch, lens, H, Dv, ahead):
    spans, slots = [(0, n) for n in lens], list(range(len(lens)))
    seg, cu = step_of(spans, slots, len(lens), "cuda")
    names = routed(monkeypatch, lambda: run_scan("ssd", seg, cu, spans, slots, H, 1, 16, Dv, "cuda", torch.bfloat16, scale=0.5))
    assert names == ["sm_head_scan_ahead" if ahead else "sm_head_scan_chunk"]
