"""Decoded rows of chunk attention (keys that double as values) at the edges of a step of the waves, in float64."""
import pytest
import torch

from lumen.ops.attention import chunk_sink_attention
from lumen.ops.segments import SegBatch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,ulp", [(torch.bfloat16, 2.0 ** -8), (torch.float16, 2.0 ** -11)])
@pytest.mark.parametrize("H,G,D,bs", [(4, 2, 32, 16), (2, 2, 64, 16), (4, 1, 128, 24), (2, 1, 256, 16)])
@pytest.mark.parametrize("chunk,sink", [(0, True), (100, False), (1024, True)])
def test_decoded_rows(H, G, D, bs, chunk, sink, dt, ulp):
    lens = [1, 2, 15, 16, 17, 128, 129, 255, 257, 512, 1024, 1025, 2100]
    T, per = len(lens), (max(lens) + bs - 1) // bs
    g = torch.Generator(device="cuda").manual_seed(D)
    i32 = dict(dtype=torch.int32, device="cuda")
    tables = torch.randperm(T * per, generator=torch.Generator().manual_seed(D)).view(T, per).to(**i32)
    cache = torch.randn(T * per, bs, G, D, device="cuda", generator=g).to(dt)
    q = torch.randn(T, H * D + 8, device="cuda", generator=g).to(dt)[:, :H * D]
    pos, ar = torch.tensor(lens, **i32) - 1, torch.arange(T + 1, **i32)
    seg = SegBatch(ar, ar[:T], pos, ar[:T], pos, tables, None)
    got = chunk_sink_attention(q, cache, seg, H, G, D, 0.5, chunk, 1e-6, sink).view(T, H, D).double()
    qd = q.double().view(T, H, D)
    qd = qd / torch.sqrt(qd.square().mean(-1, keepdim=True) + 1e-6)
    for t, n in enumerate(lens):
        lo = (n - 1) // chunk * chunk if chunk else 0
        j = torch.arange(lo, n, device="cuda")
        k = cache[tables[t].long()[j // bs], j % bs].double()              # [n, G, D]
        kn = (k / torch.sqrt(k.square().mean(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, 1)
        s = (kn * qd[t]).sum(-1) * 0.5
        e = torch.exp(s)
        want = (e[..., None] * k.repeat_interleave(H // G, 1)).sum(0) / (e.sum(0) + float(sink))[:, None]
        # one rounding; fp32 sums of up to 2100 weights
        assert ((got[t] - want).abs() <= ulp * want.abs() + 2e-5 * want.abs().max()).all(), n
