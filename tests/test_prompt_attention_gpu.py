"""Attention of prompt portions in tiles of 128 rows and 64 keys (seqmix/window_attention.hip, seqmix/attention.hip)
where the tiles' edges, the block table and the moving reference of the weights can go wrong: portions around 32, 64
and 128 rows, cached context, blocks that are not a power of two, more blocks than the kernels hold in LDS, scores
that creep upwards, and unowned cache rows full of NaN."""
import pytest
import torch

from lumen.ops.attention import chunk_sink_attention, chunk_sink_attention_ref, row_attention, row_attention_ref
from lumen.ops.segments import SegBatch, tile_list

pytestmark = pytest.mark.gpu
DTYPES = [(torch.bfloat16, 2.0 ** -8), (torch.float16, 2.0 ** -11)]


def portions(lens, starts, bs, g, *shapes):
    """Portions of whole tiles and their caches, one per (heads, size): scrambled blocks, NaN where no key is."""
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    total = [s + n for s, n in zip(starts, lens)]
    nb = [(t + bs - 1) // bs for t in total]
    order = torch.randperm(sum(nb) + 3, generator=g).tolist()
    tables = torch.zeros(len(lens), max(nb), dtype=torch.int32)
    caches = [torch.full((sum(nb) + 3, bs, *s), float("nan")) for s in shapes]
    for i, n in enumerate(nb):
        for b in range(n):
            tables[i, b] = order.pop()
            for c in caches:
                rows = min(bs, total[i] - b * bs)
                c[tables[i, b], :rows] = torch.randn(rows, *c.shape[2:], generator=g)
    i32 = dict(dtype=torch.int32, device="cuda")
    seg = SegBatch(torch.tensor(cu, **i32), torch.arange(len(lens), **i32), torch.tensor(starts, **i32),
                   torch.cat([torch.full((n,), i) for i, n in enumerate(lens)]).int().cuda(),
                   torch.cat([torch.arange(n) + s for s, n in zip(starts, lens)]).int().cuda(),
                   tables.cuda(), None, torch.tensor(tile_list(cu, len(lens)), **i32).view(-1, 2), cu[-1], 128)
    return cu[-1], seg, caches


def close(out, ref, ulp):
    # the output's rounding (half an ulp), the weights' ~16 bits and the products' fp32 sums, relative to the
    # largest entry: under two ulps of it
    assert torch.isfinite(out).all()
    err = (out.float() - ref.float()).abs().max() / ref.float().abs().max()
    assert err < 2 * ulp, err


@pytest.mark.parametrize("dtype,ulp", DTYPES)
@pytest.mark.parametrize("lens,starts,bs,window,keep", [
    ([31, 32, 33, 63, 64, 65, 1], [0, 0, 1, 0, 70, 3, 5], 16, 0, 0),
    ([127, 128, 129], [0, 64, 1], 12, 70, 5), ([130, 66], [200, 61], 16, 64, 130), ([40, 5], [560, 0], 1, 0, 0),
    ([33], [700], 1, 620, 7)])
@pytest.mark.parametrize("H,G,D,Dv", [(4, 2, 128, 128), (2, 2, 32, 64), (2, 1, 128, 256)])
def test_window_tiles(H, G, D, Dv, lens, starts, bs, window, keep, dtype, ulp):
    g = torch.Generator().manual_seed(D + bs + len(lens))
    T, seg, (k, v) = portions(lens, starts, bs, g, (G, D), (G, Dv))
    k, v = k.to(dtype).cuda(), v.to(dtype).cuda()
    q = torch.randn(T, H, D, generator=g).to(dtype).cuda()
    for cap, slopes in ((0.0, None), (3.0, torch.rand(H, generator=g).cuda() * 0.1)):
        out, ref = (torch.zeros(T, H, Dv, dtype=dt, device="cuda") for dt in (dtype, torch.float32))
        row_attention(q, None, k, v, Dv, out, seg, H, G, D ** -0.5, cap, slopes=slopes, window=window, keep_first=keep)
        row_attention_ref(q.float(), None, k.float(), v.float(), Dv, ref, seg, H, G, D ** -0.5, cap, slopes=slopes,
                          window=window, keep_first=keep)
        close(out, ref, ulp)


@pytest.mark.parametrize("dtype,ulp", DTYPES)
@pytest.mark.parametrize("lens,starts,bs,chunk", [
    ([31, 32, 33, 63, 64, 65, 1], [0, 0, 1, 0, 70, 3, 5], 16, 0), ([127, 128, 129], [0, 64, 1], 12, 75),
    ([40, 5], [560, 0], 1, 0)])
@pytest.mark.parametrize("H,G,D", [(4, 2, 128), (2, 1, 96), (2, 2, 256)])
def test_chunk_tiles(H, G, D, lens, starts, bs, chunk, dtype, ulp):
    g = torch.Generator().manual_seed(D + bs + len(lens))
    T, seg, (k,) = portions(lens, starts, bs, g, (G, D))
    k = k.to(dtype).cuda()
    q = torch.randn(T, H * D, generator=g).to(dtype).cuda()
    out = chunk_sink_attention(q, k, seg, H, G, D, 0.3, chunk, 1e-6)
    close(out, chunk_sink_attention_ref(q.float(), k.float(), seg, H, G, D, 0.3, chunk, 1e-6), ulp)


@pytest.mark.parametrize("dtype,ulp", DTYPES)
@pytest.mark.parametrize("rise", [0.01, 0.07, 0.5, -0.5])
def test_scores_that_creep(rise, dtype, ulp):
    """The score grows by ``rise`` per key: under and over what moves the reference within a tile."""
    T, H, G, D = 300, 1, 1, 64
    g = torch.Generator().manual_seed(7)
    _, seg, (k, v) = portions([T], [0], 16, g, (G, D), (G, D))
    k[:, :, :, 0] = 0.0
    for j in range(T):
        k[seg.tables[0, j // 16].item(), j % 16, 0, 0] = rise * j
    k, v = k.to(dtype).cuda(), v.to(dtype).cuda()
    q = torch.zeros(T, H, D)
    q[:, :, 0] = 1.0
    q = q.to(dtype).cuda()
    out, ref = (torch.zeros(T, H, D, dtype=dt, device="cuda") for dt in (dtype, torch.float32))
    row_attention(q, None, k, v, D, out, seg, H, G, 1.0)
    row_attention_ref(q.float(), None, k.float(), v.float(), D, ref, seg, H, G, 1.0)
    close(out, ref, ulp)
