"""The decoded rows' DyT convolution in one launch: exactly what the separate kernels leave behind."""
import pytest
import torch

from lumen.ops import _seqmix
from lumen.ops import conv as conv_mod
from lumen.ops.segments import SegBatch

pytestmark = pytest.mark.gpu
dev = "cuda"


@pytest.mark.parametrize("taps", [1, 2, 4, 8])
@pytest.mark.parametrize("S,W,dt", [(1, 4, torch.bfloat16), (3, 260, torch.float16),
                                    (64, 2048, torch.bfloat16), (17, 1024, torch.float32)])
def test_dyt_canon_rows(S, W, dt, taps, monkeypatch):
    g = torch.Generator().manual_seed(S + taps)
    r = lambda *s: torch.randn(*s, generator=g).to(dev)  # noqa: E731
    x, norm, cw = r(S, W), (1 + r(W), r(W), r(1)), r(W, taps)
    tail = r(S + 2, max(taps - 1, 0), W)
    i32 = dict(dtype=torch.int32, device=dev)
    start = torch.arange(S, **i32) * 3 % 11                      # also positions below the window
    slot = torch.randperm(S + 2, generator=g)[:S].to(**i32)
    seg = SegBatch(torch.arange(S + 1, **i32), slot, start, torch.arange(S, **i32), start)
    called = []
    real = _seqmix.call
    monkeypatch.setattr(_seqmix, "call", lambda name, *a: (called.append(name), real(name, *a)))
    t1, t2 = tail.clone(), tail.clone()
    got = conv_mod.dyt_canon(x, norm, cw, t1, seg, dt)
    assert called == ["sm_dyt_canon_rows"]
    monkeypatch.setattr(SegBatch, "portions", lambda self: (self.S, self.T))
    want = conv_mod.dyt_canon(x, norm, cw, t2, seg, dt)
    assert "sm_dyt_canon" in called
    assert torch.equal(got, want)
    assert torch.equal(t1, t2)

