"""A decode step's inputs into static graph buffers, and the decoded rows' DyT convolution, each in one
launch: exactly what the separate copies, fills and kernels leave behind."""
import pytest
import torch

from lumen.ops import _seqmix
from lumen.ops import conv as conv_mod
from lumen.ops.segments import SegBatch
from lumen.serve.model_runner import fill_step

pytestmark = pytest.mark.gpu
dev = "cuda"


@pytest.mark.parametrize("n,bucket,width,ld", [(1, 1, 1, 1), (1, 8, 3, 7), (64, 64, 40, 64), (257, 512, 9, 9),
                                               (5, 8, 0, 4)])
@pytest.mark.parametrize("strided", [False, True])
def test_fill_step(n, bucket, width, ld, strided, monkeypatch):
    g = torch.Generator().manual_seed(n)
    i32 = lambda *s: torch.randint(0, 1 << 30, s, generator=g, dtype=torch.int32).to(dev)  # noqa: E731
    i64 = lambda *s: torch.randint(0, 1 << 40, s, generator=g).to(dev)  # noqa: E731
    cut = (lambda t: t.repeat_interleave(2, -1)[..., ::2]) if strided else (lambda t: t)
    src = [cut(i32(n)) for _ in range(3)]
    tok, slot, tab = cut(i64(n)), cut(i64(n)), cut(i32(n, width))
    pads = [None, 7, -1]
    dst = [i32(bucket) for _ in range(3)]
    td, sd, bd = i64(bucket), i64(bucket), i32(bucket, ld)
    want = [d.clone() for d in dst + [td, sd, bd]]
    for w, s, p in zip(want, src, pads):
        w[:n] = s
        if p is not None:
            w[n:] = p
    want[3][:n], want[4][:n] = tok, slot
    want[4][n:] = -1
    want[5][:n, :width] = tab
    called = []
    real = _seqmix.call
    monkeypatch.setattr(_seqmix, "call", lambda name, *a: (called.append(name), real(name, *a)))
    fill_step(list(zip(src, dst, pads)), tok, td, slot, sd, tab, bd, n, bucket)
    # one launch for contiguous rows (of one entry, any stride is), copies for the others
    one = all(t.is_contiguous() for t in src + [tok, slot, tab])
    assert called == ["sm_fill_step"] * one and (one or strided)
    for w, d in zip(want, dst + [td, sd, bd]):
        assert torch.equal(w, d)


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

