"""Decoded rows behind tables of a server's longest context: the row kernel with few heads a workgroup, and both forms of the
latent kernel, against plain attention in float64, at the edges of their tiles of 64 and 128 keys."""
import pytest
import torch

from lumen.ops.attention import row_attention
from lumen.ops.segments import SegBatch

pytestmark = pytest.mark.gpu
dev = "cuda"


def step(ctx, g, blocks=256, bs=16):
    """One decoded row per sequence: row t of sequence t sees ``ctx[t]`` keys, in cache blocks in no order."""
    T = len(ctx)
    need = [-(-c // bs) for c in ctx]
    free = torch.randperm(sum(need) + 1, generator=g).tolist()
    tables = torch.zeros(T, blocks, dtype=torch.int32)
    for t, n in enumerate(need):
        tables[t, :n] = torch.tensor([free.pop() for _ in range(n)], dtype=torch.int32)
    i32 = dict(dtype=torch.int32, device=dev)
    seq, pos = torch.arange(T, **i32), torch.tensor(ctx, **i32) - 1
    return SegBatch(torch.arange(T + 1, **i32), seq, pos, seq, pos, tables.to(dev), None), sum(need) + 1, tables


def plain(q, rows, scale):
    """q [H, D], rows: per head its keys [n, D] and values [n, Dv], float64."""
    return torch.stack([torch.softmax(scale * (k @ q[h]), 0) @ v for h, (k, v) in enumerate(rows)])


def close(got, want, mag, dt):
    """One rounding of the result; weights and sums in fp32 (weights of 16 + 8 bits at least), over values of size ``mag``."""
    tol = want.abs() * torch.finfo(dt).eps / 2 + mag * 2.0 ** -13
    assert ((got.double().cpu() - want).abs() <= tol).all()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,H,G", [(1, 16, 4), (4, 32, 8), (8, 16, 16), (9, 16, 2), (16, 8, 2), (17, 12, 3), (32, 16, 4)])
def test_few_rows(T, H, G, dt):
    g = torch.Generator().manual_seed(T)
    ctx = [(1, 63, 64, 65, 200, 128, 129, 300)[t % 8] for t in range(T)]
    seg, nb, tables = step(ctx, g)
    q, k, v = (torch.randn(*s, generator=g).to(dt) for s in ((T, H, 128), (nb, 16, G, 128), (nb, 16, G, 128)))
    out = torch.empty(T, H, 128, dtype=dt, device=dev)
    row_attention(q.to(dev), None, k.to(dev), v.to(dev), 128, out, seg, H, G, 0.088)
    for t, n in enumerate(ctx):
        rows = tables[t].long()[torch.arange(n) // 16] * 16 + torch.arange(n) % 16
        kk, vv = k.view(-1, G, 128)[rows].double(), v.view(-1, G, 128)[rows].double()
        want = plain(q[t].double(), [(kk[:, h * G // H], vv[:, h * G // H]) for h in range(H)], 0.088)
        close(out[t], want, vv.abs().max(), dt)


@pytest.mark.parametrize("sink,window", [(False, 0), (True, 0), (False, 100), (True, 200)])
@pytest.mark.parametrize("T,H,G", [(16, 8, 2), (1, 16, 4), (5, 4, 4)])
def test_splits_past_a_rows_last_tile_are_not_read(T, H, G, sink, window):
    """32 splits for rows of 1 - 30 tiles, in memory that held NaN."""
    g = torch.Generator().manual_seed(T + window)
    ctx = [(1, 64, 65, 1900, 128, 129, 700, 640)[t % 8] for t in range(T)]
    seg, nb, tables = step(ctx, g)
    dt = torch.bfloat16
    q, k, v = (torch.randn(*s, generator=g).to(dt) for s in ((T, H, 128), (nb, 16, G, 128), (nb, 16, G, 128)))
    s = torch.randn(H, generator=g)
    out = torch.empty(T, H, 128, dtype=dt, device=dev)
    qd, kd, vd, sd = q.to(dev), k.to(dev), v.to(dev), s.to(dev)
    for n in (T * H * 32 * 2, T * H * 32 * 128):
        torch.full((n,), float("nan"), device=dev)         # freed at once: the workspaces lie here
    row_attention(qd, None, kd, vd, 128, out, seg, H, G, 0.088, sink=sd if sink else None, window=window)
    for t, n in enumerate(ctx):
        at = torch.arange(max(0, n - window) if window else 0, n)
        rows = tables[t].long()[at // 16] * 16 + at % 16
        kk, vv = k.view(-1, G, 128)[rows].double(), v.view(-1, G, 128)[rows].double()
        want = []
        for h in range(H):
            z = 0.088 * (kk[:, h * G // H] @ q[t, h].double())
            z = torch.cat([z, s[h:h + 1].double()]) if sink else z
            want.append(torch.softmax(z, 0)[:len(at)] @ vv[:, h * G // H])
        close(out[t], torch.stack(want), vv.abs().max(), dt)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,H,R,D2", [(1, 16, 512, 64), (9, 16, 256, 32), (600, 3, 256, 32), (5, 20, 384, 64), (7, 4, 512, 8),
                                      (6, 16, 192, 64), (600, 2, 64, 0)])
def test_latent_rows(T, H, R, D2, dt):
    g = torch.Generator().manual_seed(T + R)
    few = (1, 31, 32, 33, 127, 128, 129, 161, 300)
    ctx = [few[t % 9] if T < 100 else 1 + t % 40 for t in range(T)]
    seg, nb, tables = step(ctx, g)
    D = R + D2
    q = torch.randn(T, H, D, generator=g).to(dt)
    c = torch.randn(nb, 16, D, generator=g).to(dt)
    spare = next(b for b in range(nb) if not any((tables[t, :-(-n // 16)] == b).any() for t, n in enumerate(ctx)))
    c[spare] = float("nan")                                   # the block that no row's table names
    vt = c[:, :, :R].transpose(1, 2).contiguous()
    out = torch.empty(T, H, R, dtype=dt, device=dev)
    qd, cd = q.to(dev), c.to(dev)
    row_attention(qd[:, :, :R], qd[:, :, R:] if D2 else None, cd, cd, R, out, seg, H, 1, 0.05, vt=vt.to(dev))
    for t in range(0, T, max(1, T // 40)):
        n = ctx[t]
        rows = tables[t].long()[torch.arange(n) // 16] * 16 + torch.arange(n) % 16
        k = c.view(-1, D)[rows].double()
        close(out[t], plain(q[t].double(), [(k, k[:, :R])] * H, 0.05), k.abs().max(), dt)
