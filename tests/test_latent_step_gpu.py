"""A decode step's latent-attention inputs and queries in one launch each, and the gated token slice in its projection's
epilogue, against the separate forms in float64."""
import pytest
import torch

from launches import launches
from lumen.ops.attention import LATENT_STEP_MAX_T, latent_inputs, latent_query, latent_write_ref
from lumen.ops.embedding import gated_token_project, gated_token_slice_ref
from lumen.ops.norm import group_rms_norm_ref
from lumen.ops.rope import rotate_interleaved_ref

pytestmark = pytest.mark.gpu
ULP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -22}


def near(got, want, dt, sums=1e-5):
    """One rounding of the result (its neighbour where an fp32 sum ends differently), fp32 sums."""
    err = (got.double() - want.double()).abs()
    assert (err <= 2 * ULP[dt] * want.double().abs() + sums * want.double().abs().max()).all(), err.max()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,Q,R,Dr,dims,pad", [(1, 768, 512, 64, 64, 0), (65, 48, 64, 8, 4, 3), (7, 300, 100, 0, 0, 5),
                                               (LATENT_STEP_MAX_T, 64, 32, 6, 6, 0),
                                               (LATENT_STEP_MAX_T + 1, 64, 32, 6, 6, 0)])
def test_inputs(T, Q, R, Dr, dims, pad, dt):
    g = torch.Generator(device="cuda").manual_seed(T)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    z = r(T, Q + R + Dr + pad).to(dt)[:, :Q + R + Dr]
    wq, wn, f = 1 + 0.1 * r(Q), 1 + 0.1 * r(R), 1.0 / 100 ** torch.linspace(0, 1, max(1, dims // 2), device="cuda")
    nb, bs = T // 16 + 2, 16
    slots = torch.randperm(nb * bs, generator=torch.Generator().manual_seed(T))[:T].cuda()
    if T > 3:
        slots[3] = -1
    pos = torch.randint(0, 3000, (T,), device="cuda", generator=g, dtype=torch.int32)
    c1, v1 = torch.zeros(nb, bs, R + Dr, device="cuda", dtype=dt), torch.zeros(nb, R, bs, device="cuda", dtype=dt)
    c2, v2 = c1.clone().double(), v1.clone().double()
    qn = latent_inputs(z, Q, wq, wn, f if dims else None, pos, slots, c1, R, dims, 1e-6, v1)
    latent_write_ref(z[:, Q:], wn, f, pos, slots, c2, R, dims, 1e-6, v2)
    near(qn, group_rms_norm_ref(z[:, :Q].double(), wq, 1, 1e-6, torch.float64), dt)
    near(c1, c2, dt, 1e-4)                                # angles of up to 3000 in fp32: 2e-4 of a turn's last bits
    near(v1, v2, dt)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,H,D,R,Dr,dims", [(1, 16, 128, 512, 64, 64), (64, 3, 64, 64, 0, 0), (65, 2, 192, 128, 8, 4),
                                             (130, 5, 256, 192, 16, 16), (17, 2, 96, 64, 32, 32), (9, 2, 128, 96, 64, 64),
                                             (LATENT_STEP_MAX_T + 3, 1, 64, 64, 8, 8)])
def test_query(T, H, D, R, Dr, dims, dt):
    g = torch.Generator(device="cuda").manual_seed(T)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    q, uk = r(T, H, D + Dr).to(dt), (r(H, D, R) / D ** 0.5).to(dt)
    f = 1.0 / 100 ** torch.linspace(0, 1, max(1, dims // 2), device="cuda")
    pos = torch.randint(0, 3000, (T,), device="cuda", generator=g, dtype=torch.int32)
    want = torch.matmul(q[:, :, :D].double().transpose(0, 1), uk.double())
    turned = q.clone().view(T, H * (D + Dr))
    if dims:
        rotate_interleaved_ref(turned, pos, H, D + Dr, D, dims, f)
    got = latent_query(q, uk, uk.transpose(1, 2).contiguous(), D, pos, dims, f)
    near(got, want, dt)
    assert torch.equal(q[:, :, :D], turned.view(T, H, D + Dr)[:, :, :D])
    near(q, turned.view(T, H, D + Dr), dt, 1e-4)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,W,dim,cols", [(1, 2048, 128, 512), (8, 64, 4, 12), (33, 1024, 60, 60), (64, 4096, 256, 1024),
                                          (65, 512, 16, 64), (5, 100, 12, 48)])
def test_gated_token_slice(T, W, dim, cols, dt):
    g = torch.Generator(device="cuda").manual_seed(T)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    x, w, table = r(T, W).to(dt), (r(dim, W) / W ** 0.5).to(dt), r(50, cols).to(dt)
    tok = torch.randint(0, 50, (T,), device="cuda", generator=g)
    for col0 in (0, cols - dim):
        got = gated_token_project(x, w, table, tok, col0)
        want = gated_token_slice_ref(x.double() @ w.double().t(), table.double(), tok, col0)
        near(got, want, dt, 2 * ULP[dt])                  # (separate launches round the product as well)
    with pytest.raises(ValueError):
        gated_token_project(x, w, table, tok, cols - dim + 1)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,H,R,Dr,Dv,ctx,gated", [(1, 16, 512, 64, 128, 700, False), (17, 4, 512, 64, 64, 130, True),
                                                   (64, 16, 512, 0, 256, 40, True), (40, 16, 256, 32, 16, 300, False),
                                                   (300, 32, 512, 64, 48, 9, True), (5, 2, 512, 64, 24, 90, True)])
def test_sums_and_expansion(T, H, R, Dr, Dv, ctx, gated, dt):
    """Many splits of the keys, few, one; a size that keeps the separate product (24 columns)."""
    from lumen.ops.attention import row_attention, transposed_values_ok
    from lumen.ops.segments import SegBatch

    g = torch.Generator(device="cuda").manual_seed(T)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    bs, i32 = 16, dict(dtype=torch.int32, device="cuda")
    assert transposed_values_ok(dt, R, Dr, bs, "cuda")
    lens = torch.randint(1, ctx + 1, (T,), generator=torch.Generator().manual_seed(T))
    lens[0] = ctx
    per = (ctx + bs - 1) // bs
    tables = torch.randperm(64 * per)[torch.arange(T * per) % (64 * per)].view(T, per).to(**i32)
    cache = r(64 * per, bs, R + Dr).to(dt)
    vt = cache[:, :, :R].transpose(1, 2).contiguous()
    pos = (lens - 1).to(**i32)
    ar = torch.arange(T + 1, **i32)
    seg = SegBatch(ar, ar[:T], pos, ar[:T], pos, tables, None)
    qa, q2 = r(H, T, R).to(dt), r(T, H, Dr).to(dt) if Dr else None
    gate = r(T, H).to(dt) if gated else None
    uv = (r(H, Dv, R) / R ** 0.5).to(dt)
    kw = dict(vt=vt, gate=gate, sink=r(H) if gated else None)
    ol = torch.empty(H, T, R, dtype=dt, device="cuda")
    row_attention(qa.transpose(0, 1), q2, cache, cache, R, ol.transpose(0, 1), seg, H, 1, 0.05, **kw)
    o = torch.zeros(T, H, Dv + 4, dtype=dt, device="cuda")[:, :, :Dv]
    out = torch.empty_like(ol).transpose(0, 1)
    got = row_attention(qa.transpose(0, 1), q2, cache, cache, R, out, seg, H, 1, 0.05, expand=(uv, o), **kw)
    assert (got is o) == (Dv % 16 == 0)
    if got is o:
        # the same rows, their last bit apart where the splits' sum ends differently, through sums of R products
        want = torch.matmul(ol.double(), uv.double().transpose(1, 2).contiguous()).transpose(0, 1)
        near(o, want, dt, ULP[dt])
    else:
        assert torch.equal(got.transpose(0, 1), ol)


def rows_behind(T, H, R, Dr, ctx, dt):
    """Decoded rows of up to ``ctx`` keys, the first of all of them: (queries, cache, transposed values, segments)."""
    from lumen.ops.segments import SegBatch

    g = torch.Generator(device="cuda").manual_seed(T + ctx)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g).to(dt)  # noqa: E731
    bs, per, i32 = 16, (ctx + 15) // 16, dict(dtype=torch.int32, device="cuda")
    lens = torch.randint(1, ctx + 1, (T,), generator=torch.Generator().manual_seed(T))
    lens[0] = ctx
    tables = torch.randperm(64 * per, generator=torch.Generator().manual_seed(ctx))[torch.arange(T * per) % (64 * per)].view(T, per).to(**i32)
    cache, pos, ar = r(64 * per, bs, R + Dr), (lens - 1).to(**i32), torch.arange(T + 1, **i32)
    return r(T, H, R), r(T, H, Dr), cache, cache[:, :, :R].transpose(1, 2).contiguous(), SegBatch(ar, ar[:T], pos, ar[:T], pos, tables, None)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,H,R,Dr,ctx,kernel,splits", [
    (8, 16, 256, 32, 2100, ("latent_row_kernel<", ", 4, 9, 8>("), 17), (3, 16, 384, 64, 127, ("latent_row_kernel<", ", 6, 14, 8>("), 1),
    (3, 16, 512, 64, 64, ("latent_row_kernel<", ", 8, 18, 4>("), 1), (130, 17, 384, 64, 1030, ("latent_row_kernel<", ", 6, 14, 8>("), 4),
    (224, 17, 512, 32, 140, ("latent_row_kernel<", ", 8, 17, 8>("), 1), (225, 17, 512, 64, 140, ("latent_attn_kernel<", ", 8, true>("), 1),
    (256, 32, 384, 0, 70, ("latent_attn_kernel<", ", 6, true>("), 1)])
def test_rows_of_each_tile_and_split(T, H, R, Dr, ctx, kernel, splits, dt):
    """The rounding of the result and ~16 bits of the weights: under two ulps of the largest entry."""
    from lumen.ops.attention import row_attention, row_attention_ref

    q, q2, cache, vt, seg = rows_behind(T, H, R, Dr, ctx, dt)
    q2 = q2 if Dr else None
    out, ref = torch.empty_like(q), torch.empty(T, H, R, device="cuda")
    run = lambda: row_attention(q, q2, cache, cache, R, out, seg, H, 1, 0.05, vt=vt)  # noqa: E731
    (name, grid, _), *_ = launches(run)
    assert all(k in name for k in kernel) and grid == (T, (H + 15) // 16, splits), (name, grid)
    row_attention_ref(q.float(), q2.float() if Dr else None, cache.float(), cache.float(), R, ref, seg, H, 1, 0.05)
    assert (out.float() - ref).abs().max() < 2 * ULP[dt] * ref.abs().max()


@pytest.mark.parametrize("T,H,R,ctx,grid", [(1, 16, 512, 40, 1), (16, 16, 512, 300, 16), (17, 16, 512, 300, 9), (48, 16, 128, 300, 12), (49, 32, 128, 40, 7),
                                            (65, 32, 256, 9, 5), (300, 32, 128, 20, 19)])
def test_rows_of_an_expansion_have_a_cu(T, H, R, ctx, grid):
    """Workgroups of the expansion take 16 rows, or fewer while each has a CU of its own."""
    from lumen.ops.attention import row_attention

    dt = torch.bfloat16
    q, q2, cache, vt, seg = rows_behind(T, H, R, 64, ctx, dt)
    uv, o = (torch.randn(H, 64, R, device="cuda") / R ** 0.5).to(dt), torch.empty(T, H, 64, dtype=dt, device="cuda")
    ol, args = torch.empty_like(q), (seg, H, 1, 0.05)
    row_attention(q, q2, cache, cache, R, ol, *args, vt=vt)
    run = lambda: row_attention(q, q2, cache, cache, R, torch.empty_like(q), *args, vt=vt, expand=(uv, o))  # noqa: E731
    (name, g, _) = launches(run)[-1]
    assert "latent_out_kernel" in name and g == (grid, H, 1)
    want = torch.matmul(ol.double().transpose(0, 1), uv.double().transpose(1, 2).contiguous()).transpose(0, 1)
    near(o, want, dt, ULP[dt])
