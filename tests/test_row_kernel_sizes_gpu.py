"""Which row kernel a call takes: rows held in registers while a row's chain of loads is what it costs, in LDS or by passes where many
rows hide that, at the edges of either; each against float64."""
import pytest
import torch

from launches import launches
from lumen.ops import attention as A
from lumen.ops import norm
from test_step_rows_gpu import gen, near

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def kernel(run):
    (name, _, _), = launches(run)
    return name


@pytest.mark.parametrize("T,W,groups,held", [
    (1, 512, 1, 1), (768, 512, 1, 1), (769, 512, 1, 0), (2000, 1024, 1, 1), (769, 1536, 1, 0), (1025, 768, 2, 1), (1025, 768, 1, 1), (1025, 640, 1, 0), (1025, 2048, 2, 2), (1500, 1536, 4, 2),
    (768, 2560, 1, 3), (769, 2560, 1, 0), (1500, 3072, 1, 3), (5, 3072, 2, 3), (1024, 4096, 1, 4), (1025, 4096, 1, 0), (1025, 4096, 4, 0), (769, 3584, 2, 0),
    (3, 4100, 1, 0)])
def test_gated_norms(T, W, groups, held):
    r = gen(W + T)
    o, z, w = r(T, W), r(T, W).to(BF16), r(W)
    name = kernel(lambda: norm.gated_rms_norm(o, z, w, groups, 1e-6, "silu", True))
    assert (f"gated_rms_wide_kernel<__hip_bfloat16, {held}>" in name) if held else "gated_rms_kernel<" in name
    a = torch.sigmoid(z.double()) * z.double()
    p = (o.double() * a).reshape(T, groups, -1)
    near(norm.gated_rms_norm(o, z, w, groups, 1e-6, "silu", True), (p / torch.sqrt((p * p).mean(-1, keepdim=True) + 1e-6)).reshape(T, W) * w.double())


@pytest.mark.parametrize("T,W,held", [(1, 256, 1), (769, 256, 0), (769, 512, 0), (4096, 768, 1), (4097, 1024, 0), (1024, 2048, 2), (1025, 2048, 0),
                                      (768, 2560, 3), (769, 2560, 0), (5, 3072, 3), (768, 4096, 4), (769, 4096, 0), (769, 3072, 0), (2, 4100, 0)])
def test_stream_norms(T, W, held):
    r = gen(W + T)
    x, y, w = r(T, W), r(T, W).to(BF16), r(W)
    want = x.double() + y.double()
    h = norm.residual_rms(x, y, w, 1e-6)
    near(x, want)
    near(h, want / torch.sqrt((want * want).mean(-1, keepdim=True) + 1e-6) * w.double())
    name = kernel(lambda: norm.residual_rms(x, y, w, 1e-6))
    assert (f"stream_row_kernel<__hip_bfloat16, {held}>" in name) if held else "stream_rms_kernel<" in name


def heads_of(T, H, G, D, dims):
    r = gen(H * D + T)
    slots = torch.randperm(T, generator=torch.Generator().manual_seed(T)).cuda()
    caches = [torch.zeros(T, 1, G, D, device="cuda", dtype=BF16) for _ in range(2)]
    return r(T, (H + 2 * G) * D).to(BF16), r, slots, caches


@pytest.mark.parametrize("T,H,G,D,lanes", [(1, 2, 1, 128, 0), (70, 3, 1, 128, 0), (5, 1, 1, 512, 0), (3, 4, 1, 128, 1), (70, 2, 2, 128, 0),
                                           (5, 4, 2, 64, 1), (2, 16, 4, 128, 1), (2, 32, 32, 128, 0)])
def test_head_norms(T, H, G, D, lanes):
    """Four heads and fewer to norm keep a wave each."""
    z, r, slots, (kc, vc) = heads_of(T, H, G, D, 0)
    wq, wk = r(D), r(D)
    got = z.clone()
    A.head_norm_write(got, wq, wk, slots, kc, vc, H, G, D, D, 1e-6)
    x = z.double().view(T, H + 2 * G, D)
    unit = x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6)
    near(got[:, :H * D], (unit[:, :H] * wq.double()).reshape(T, -1), 1e-5)
    near(kc[slots, 0].flatten(1), (unit[:, H:H + G] * wk.double()).reshape(T, -1), 1e-5)
    assert torch.equal(vc[slots, 0].flatten(1), z[:, (H + G) * D:])
    name = kernel(lambda: A.head_norm_write(got, wq, wk, slots, kc, vc, H, G, D, D, 1e-6))
    assert ("head_norm_write_lanes<" if lanes else "head_norm_write_kernel<") in name


@pytest.mark.parametrize("T,H,G,D,dims,held", [(512, 8, 2, 64, 64, 1), (513, 8, 2, 64, 64, 0), (513, 2, 1, 128, 0, 0), (512, 32, 8, 128, 128, 2),
                                               (513, 32, 8, 128, 128, 0), (600, 16, 4, 128, 128, 0), (600, 32, 32, 128, 128, 2), (3073, 16, 4, 128, 128, 1), (3073, 8, 2, 64, 64, 0), (3, 33, 32, 128, 128, 0)])
def test_row_norms_with_rotation(T, H, G, D, dims, held):
    z, r, slots, (kc, vc) = heads_of(T, H, G, D, dims)
    wq, wk, pos = r(H * D), r(G * D), torch.arange(T, device="cuda", dtype=torch.int32) % 90
    f = 1.0 / 100 ** torch.linspace(0, 1, max(1, dims // 2), device="cuda")
    got = z.clone()
    run = lambda: A.row_norm_rotary_write(got, wq, wk, pos, slots, kc, vc, H, G, D, D, dims, f, 1.0, 1e-6)  # noqa: E731
    run()
    a = (pos.float().view(T, 1, 1) * f.view(1, 1, -1)).double()

    def want(x, w, n):
        x = (x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6) * w.double()).view(T, n, D)
        u, v = x[..., :dims // 2], x[..., dims // 2:dims]
        return torch.cat([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin(), x[..., dims:]], -1).flatten(1) if dims else x.flatten(1)

    zd = z.double()
    near(got[:, :H * D], want(zd[:, :H * D], wq, H), 1e-5)
    near(kc[slots, 0].flatten(1), want(zd[:, H * D:(H + G) * D], wk, G), 1e-5)
    assert torch.equal(vc[slots, 0].flatten(1), z[:, (H + G) * D:])
    name = kernel(run)
    assert (f"row_norm_rotary_held<__hip_bfloat16, {held}>" in name) if held else "row_norm_rotary_kernel<" in name
