"""The scans whose chunks are built ahead (seqmix/head_scan_ahead.hip) against the token loops of the oracle: portions that end on
and beside a chunk, sequences that start and go on, decoded rows behind them, head sizes on and off the blocks of 32."""
import pytest
import torch

from lumen.ops import _seqmix, recurrent
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
    monkeypatch.setattr(recurrent, "AHEAD_MIN_ROWS", dict.fromkeys(recurrent.AHEAD_MIN_ROWS, (96, 96, 96)))     # (the edges, where it does not pay too)
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


@pytest.mark.parametrize("known", [False, True])
@pytest.mark.parametrize("kind,lens,H,G,Dk,Dv,ahead", [
    ("ssd", [111], 4, 1, 16, 32, False), ("ssd", [112], 4, 1, 16, 32, True), ("ssd", [111, 109], 4, 1, 64, 32, False), ("ssd", [159] * 4, 16, 16, 64, 32, False),
    ("ssd", [160] * 4, 16, 16, 64, 64, True), ("ssd", [112] * 4, 16, 1, 64, 64, True), ("ssd", [319] * 4, 17, 17, 64, 32, False),
    ("ssd", [320] * 4, 17, 17, 64, 32, True), ("ssd", [400] * 4, 17, 1, 16, 128, False), ("ssd", [95], 4, 1, 72, 32, False), ("ssd", [96] * 4, 16, 1, 128, 128, True),
    ("ssd", [96] * 2, 4, 1, 33, 32, True), ("ssd", [223] * 4, 17, 17, 72, 32, False), ("delta", [95], 4, 1, 16, 32, False), ("delta", [96] * 4, 16, 16, 64, 32, True),
    ("delta", [111] * 4, 17, 17, 64, 32, False), ("delta", [112] * 4, 17, 17, 128, 32, True), ("const", [191], 6, 6, 64, 32, False), ("const", [192], 6, 6, 64, 32, True),
    ("const", [96], 6, 6, 72, 32, True), ("const", [300] * 6, 6, 6, 64, 32, False), ("ssd", [200], 4, 1, 16, 36, False), ("ssd", [200], 3, 1, 16, 32, True)])
def test_the_rule(monkeypatch, kind, lens, H, G, Dk, Dv, ahead, known):
    """Rows a sequence from which the second launch pays, by what a chunk is to build, the keys' size and sequences x heads."""
    from lumen.ops.recurrent import head_scan

    T = sum(lens)
    seg, _ = step_of([(0, n) for n in lens], list(range(len(lens))), len(lens), "cuda")
    if known:
        seg.fresh, seg.keys = True, (T, max(lens))
    f = lambda *s: torch.randn(*s, device="cuda").bfloat16()  # noqa: E731
    zero = torch.zeros(H, device="cuda")
    decay = zero - 0.1 if kind == "const" else (f(T, H), zero, zero)
    state = torch.zeros(len(lens), H, Dk, Dv, device="cuda")
    names = routed(monkeypatch, lambda: head_scan(f(T, G * Dk), f(T, G * Dk), f(T, H * Dv), state, seg, H, Dk, Dv, decay,
                                                  beta=f(T, H) if kind == "delta" else None, rep=H // G, key_eps=1e-6))
    assert names == ["sm_head_scan_ahead" if ahead else "sm_head_scan_chunk"]


def test_the_longest_sequence_counts_where_the_host_knows_it(monkeypatch):
    """Rows of 1024 and three times 40: the chain that is saved is the long one's."""
    from lumen.ops.recurrent import head_scan
    from lumen.ops.segments import whole_sequences

    seg, H = whole_sequences([1024, 40, 40, 40], "cuda"), 16
    q, k, v = (torch.randn(1144, H * 64, device="cuda").bfloat16() for _ in range(3))
    state = torch.zeros(4, H, 64, 64, device="cuda")
    run = lambda: head_scan(q, k, v, state, seg, H, 64, 64, torch.full((H,), -0.1, device="cuda"))  # noqa: E731
    assert routed(monkeypatch, run) == ["sm_head_scan_ahead"]
    seg.fresh = False
    assert routed(monkeypatch, run) == ["sm_head_scan_chunk"]
