"""A decode step's latent-attention inputs and queries in one launch each, and the gated token slice in its projection's
epilogue, against the separate forms in float64."""
import pytest
import torch

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
