"""The latent attention that shares key tiles among rows (seqmix/latent_tile.hip) against the row-by-row
reference in fp32: portions around the eight-row workgroups and the 32-key tiles, cached context, every score
option, partial head blocks, block sizes, and unowned cache rows full of NaN."""
import pytest
import torch

import lumen.ops.attention as A
from lumen.ops.segments import SegBatch, tile_list

pytestmark = pytest.mark.gpu


def step(lens, starts, bs, R, Dr, dtype, g):
    """A step of portions (rows with one length each; decoded rows last), scrambled blocks, NaN elsewhere."""
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    total = [s + n for s, n in zip(starts, lens)]
    nb = [(t + bs - 1) // bs for t in total]
    order = torch.randperm(sum(nb) + 3, generator=g).tolist()
    tables = torch.zeros(len(lens), max(nb), dtype=torch.int32)
    lat = torch.full((sum(nb) + 3, bs, R + Dr), float("nan"))
    for i, n in enumerate(nb):
        for b in range(n):
            tables[i, b] = order.pop()
            rows = min(bs, total[i] - b * bs)
            lat[tables[i, b], :rows] = torch.randn(rows, R + Dr, generator=g)
    lat = lat.to(dtype).cuda()
    vt = lat[:, :, :R].transpose(1, 2).contiguous()
    portions = sum(1 for n in lens if n > 1 or n == lens[0])
    i32 = dict(dtype=torch.int32, device="cuda")
    seg = SegBatch(torch.tensor(cu, **i32), torch.arange(len(lens), **i32), torch.tensor(starts, **i32),
                   torch.cat([torch.full((n,), i) for i, n in enumerate(lens)]).int().cuda(),
                   torch.cat([torch.arange(n) + s for s, n in zip(starts, lens)]).int().cuda(),
                   tables.cuda(), None, torch.tensor(tile_list(cu, portions), **i32).view(-1, 2),
                   cu[portions], 128)
    return cu[-1], seg, lat, vt


@pytest.mark.parametrize("dtype,ulp", [(torch.bfloat16, 2.0 ** -8), (torch.float16, 2.0 ** -11)])
@pytest.mark.parametrize("H,Dr,bs,opts", [
    (16, 64, 16, ()), (5, 0, 32, ("softcap", "sink")), (20, 64, 64, ("temp", "gate")),
    (32, 0, 16, ("r", "sink", "gate", "softcap", "temp"))])
def test_tiled_rows(H, Dr, bs, opts, dtype, ulp, monkeypatch):
    monkeypatch.setattr(A, "LATENT_TILE_ROWS", 1)
    R = 512
    g = torch.Generator().manual_seed(H + bs)
    lens, starts = [130, 7, 8, 9, 33, 2, 40, 1, 1], [0, 0, 25, 100, 31, 64, 0, 90, 33]
    T, seg, lat, vt = step(lens, starts, bs, R, Dr, dtype, g)
    assert seg.tile_rows == T - 2
    q = torch.randn(T, H, R + 2 * Dr, generator=g).to(dtype).cuda()
    q1, q2 = q[:, :, :R], q[:, :, R + Dr:] if Dr else None
    f = lambda *s: torch.randn(*s, generator=g).cuda()  # noqa: E731
    kw = dict(softcap=5.0 if "softcap" in opts else 0.0, q_temp=(0.3, 16) if "temp" in opts else None,
              r1=f(H).abs() if "r" in opts else None, r2=f(H).abs() if "r" in opts else None,
              sink=f(H) if "sink" in opts else None,
              gate=f(T, H + 3).to(dtype)[:, :H] if "gate" in opts else None)
    scale = 0.05
    calls = []
    import lumen.ops._seqmix as sm
    orig = sm.call
    monkeypatch.setattr(sm, "call", lambda n, *a: (calls.append(n), orig(n, *a))[1])
    out = torch.zeros(H, T, R, dtype=dtype, device="cuda")
    A.row_attention(q1, q2, lat, lat, R, out.transpose(0, 1), seg, H, 1, scale, vt=vt, **kw)
    assert calls[0] == "sm_latent_tiles" and calls[1] == "sm_latent_attn"
    want = torch.zeros(T, H, R, device="cuda")
    clean = torch.nan_to_num(lat.float())
    A.row_attention_ref(q1.float(), q2.float() if Dr else None, clean, clean, R, want, seg, H, 1, scale,
                        **{k: (v.float() if torch.is_tensor(v) else v) for k, v in kw.items()})
    got = out.transpose(0, 1).float()
    # one rounding of the result; weights carried to 2^-16, fp32 sums over <= 140 keys
    assert torch.isfinite(got).all()
    assert ((got - want).abs() <= want.abs() * ulp + 1e-4 * want.abs().max()).all()


@pytest.mark.parametrize("rows,kernel", [(2047, "sm_latent_attn"), (2048, "sm_latent_tiles")])
def test_rule_and_row_kernel_agree(rows, kernel, monkeypatch):
    """The rule's two sides at its edge (rows x 16-head blocks), and the same step on the row kernel."""
    import lumen.ops._seqmix as sm

    H, R, Dr, bs = 16, 512, 64, 16
    g = torch.Generator().manual_seed(rows)
    T, seg, lat, vt = step([1024, rows - 1024], [0, 0], bs, R, Dr, torch.bfloat16, g)
    assert seg.tile_rows * ((H + 15) // 16) == rows
    q = torch.randn(T, H, R + Dr, generator=g).bfloat16().cuda()
    calls = []
    orig = sm.call
    monkeypatch.setattr(sm, "call", lambda n, *a: (calls.append(n), orig(n, *a))[1])
    out = [torch.zeros(H, T, R, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    for o, at in zip(out, (A.LATENT_TILE_ROWS, 1 << 30)):
        monkeypatch.setattr(A, "LATENT_TILE_ROWS", at)
        A.row_attention(q[:, :, :R], q[:, :, R:], lat, lat, R, o.transpose(0, 1), seg, H, 1, 0.05, vt=vt)
    assert calls == [kernel, "sm_latent_attn"]
    a, b = (o.float() for o in out)
    assert torch.isfinite(a).all()
    # each rounds an fp32 result once: a unit apart at most, and sums over <= 1024 keys in another order
    assert ((a - b).abs() <= b.abs() * 2.0 ** -7 + 1e-4 * b.abs().max()).all()


def test_sizes_the_tiled_kernel_has():
    """The sizes it has, and sizes of which each is one step outside."""
    import lumen.ops._seqmix as sm

    assert sm.latent_tiles_ok(2, 512, 576, 512, 16, 256) and sm.latent_tiles_ok(1, 512, 512, 512, 4096, 4096)
    for dt, Dv, Dk, D1, bs, mb in ((0, 512, 576, 512, 16, 4), (2, 256, 320, 256, 16, 4),
                                   (2, 512, 544, 512, 16, 4), (2, 512, 576, 512, 8, 4),
                                   (2, 512, 576, 512, 48, 4), (2, 512, 576, 512, 16, 4097)):
        assert not sm.latent_tiles_ok(dt, Dv, Dk, D1, bs, mb)
