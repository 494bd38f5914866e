"""A step of decoded rows of the DyT stack: residual, convolution and token shift in one launch against one after the other (the
same fp32 operations: the same bits), and the scans that form their low-rank decay themselves."""
import pytest
import torch

from lumen.ops import conv
from lumen.ops.norm import dyt_residual
from lumen.ops.recurrent import delta_scan, token_shift, wkv_scan
from lumen.ops.segments import SegBatch

pytestmark = pytest.mark.gpu
dev = "cuda"


def rows(n, starts, empty=()):
    """n segments of one row (``empty``: of none) on slots in no order."""
    i32 = dict(dtype=torch.int32, device=dev)
    lens = torch.tensor([0 if i in empty else 1 for i in range(n)])
    cu = torch.cat([torch.zeros(1, dtype=torch.long), lens.cumsum(0)]).to(**i32)
    slot = torch.randperm(n + 2)[:n].to(**i32)
    pos = torch.tensor(starts[:n] * (n // len(starts) + 1))[:n].to(**i32)
    return SegBatch(cu, slot, pos, torch.arange(n, **i32), pos, None, None)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,W,taps,empty", [(1, 4, 1, ()), (3, 260, 4, (2,)), (8, 2048, 4, ()), (33, 96, 8, (30, 31, 32)), (5, 42, 3, ())])
def test_joined_and_shifted(n, W, taps, empty, dt):
    torch.manual_seed(n + W)
    seg = rows(n, [0, 5, 1, 2], empty)
    norm, post = (tuple(t.to(dev) for t in (torch.randn(W) + 1, torch.randn(W) * 0.1, torch.tensor(0.7))) for _ in range(2))
    cw, mu = torch.randn(W, taps, device=dev), torch.rand(5, W, device=dev)
    x, y = torch.randn(n, W, device=dev), torch.randn(n, W, device=dev).to(dt)
    tail, prev = torch.randn(n + 2, taps - 1, W, device=dev), torch.randn(n + 2, W, device=dev)
    live = seg.cu[-1].item()
    for joined in (False, True):
        for shifted in (False, True):
            xa, xb, ta, tb, pa, pb = x.clone(), x.clone(), tail.clone(), tail.clone(), prev.clone(), prev.clone()
            got = conv.dyt_canon(xa, norm, cw, ta, seg, dt, (y, post) if joined else None, (mu, pa) if shifted else None)
            if joined:
                dyt_residual(xb, y, post, None, dt)
            want = conv.dyt_canon(xb, norm, cw, tb, seg, dt)
            if shifted:
                want = token_shift(want, mu, pb, seg)
            assert torch.equal(got[..., :live, :], want[..., :live, :]) and torch.equal(ta, tb) and torch.equal(pa, pb)
            assert torch.equal(xa[:live], xb[:live])


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,H,D,rank", [(1, 2, 24, 8), (8, 16, 128, 16), (9, 3, 64, 64), (4, 4, 40, 24)])
def test_low_rank_decay(n, H, D, rank, dt):
    torch.manual_seed(n + D)
    seg, HD = rows(n, [3, 0, 1]), H * D
    t = [torch.randn(n, HD, device=dev).to(dt) for _ in range(5)]
    wide = torch.randint(-1, 2, (n, rank + 8), device=dev).to(dt)
    wl = wide[:, 8:]                                       # columns of a wider projection
    w2 = torch.randint(-1, 2, (HD, rank), device=dev).to(dt) / 4
    full = (wl.double() @ w2.double().t()).to(dt)          # exact in 16 bits: multiples of a quarter up to 16
    w0, u, nw = torch.randn(HD, device=dev), torch.randn(HD, device=dev), torch.rand(HD, device=dev)
    state = torch.randn(n + 2, H, D, D, device=dev)
    for scan, extra in ((wkv_scan, ()), (delta_scan, (0.6, 1e-6))):
        ins = (t[0], t[1], t[2])
        rest = (t[3],) if scan is wkv_scan else (t[3], t[4])
        sa, sb = state.clone(), state.clone()
        a = scan(*ins, wl, *rest, w0, u, nw, sa, seg, H, D, 1e-5, *extra, w2)
        b = scan(*ins, full, *rest, w0, u, nw, sb, seg, H, D, 1e-5, *extra)
        assert torch.equal(a, b) and torch.equal(sa, sb)
