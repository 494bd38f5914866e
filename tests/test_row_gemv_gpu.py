"""The norm, one row's projection and its activation in one launch (seqmix/row_gemv.hip): the separate kernels' result
over K that ends inside a step or a wave's share, few and many rows, with and without a residual."""
import pytest
import torch

from lumen.ops.activation import swiglu
from lumen.ops.gemm import row_norm_linear, row_norm_ok
from lumen.ops.norm import rms_norm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,ulp", [(torch.bfloat16, 2.0 ** -8), (torch.float16, 2.0 ** -11)])
@pytest.mark.parametrize("K,N", [(8, 4), (520, 12), (1024, 4096), (1536, 100), (2048, 20000), (2056, 64), (3072, 52), (4096, 6000),
                                 (4104, 32), (6144, 24), (8192, 4100)])
@pytest.mark.parametrize("gated,with_res", [(False, True), (True, True), (True, False), (False, False)])
def test_row_norm_linear(K, N, gated, with_res, dtype, ulp):
    g = torch.Generator().manual_seed(K + N)
    f = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    x, w, nw = f(1, K).to(dtype).cuda(), (f(N, K) * K ** -0.5).to(dtype).cuda(), (1 + 0.1 * f(K)).to(dtype).cuda()
    res = (3 * f(1, K)).to(dtype).cuda() if with_res else None
    with torch.no_grad():
        assert row_norm_ok(x, nw, res, w)
        y, s = row_norm_linear(x, nw, 1e-5, res, w, gated)
        yn, sn = rms_norm(x, nw, 1e-5, res)
    assert torch.equal(s, sn)
    ref = yn.double() @ w.double().t()                        # (the normed row rounds as the norm kernel's)
    if gated:
        ref = torch.nn.functional.silu(ref[:, :N // 2]) * ref[:, N // 2:]
    assert y.shape == ref.shape
    # the result's rounding (the type's unit roundoff, 2^-8 or 2^-11 of each entry: half the spacing 2^-7 or 2^-10 of
    # numbers from 1 on) and the fp32 sums of K products of rms 1 / sqrt(K)
    assert ((y.double() - ref).abs() <= 1.01 * ulp * ref.abs() + 2e-5 * max(1.0, float(ref.abs().max()))).all()


def test_refusals():
    x, w, nw = (torch.ones(*s, dtype=torch.bfloat16, device="cuda") for s in ((1, 64), (8, 64), (64,)))
    with torch.no_grad():
        assert row_norm_ok(x, nw, None, w)
        big = torch.ones(1, 8200, dtype=torch.bfloat16, device="cuda")
        for bad in ((x.expand(2, 64), nw, None, w), (x, nw.float(), None, w), (x, nw, None, w[:6]), (x, nw[:32], None, w),
                    (x, nw, x.half(), w), (x, nw, None, w.t().contiguous().t()), (x.cpu(), nw, None, w),
                    (big, big[0], None, big.expand(8, -1).contiguous())):
            assert not row_norm_ok(*bad)
    assert not row_norm_ok(x.clone().requires_grad_(), nw, None, w)


@pytest.mark.parametrize("K", [8, 264, 512, 1032, 2104, 2560, 3080, 4616, 5640, 6152, 7176])
@pytest.mark.parametrize("gated", [False, True])
def test_nothing_behind_a_row_is_read(K, gated):
    """K well below what the kernel's form is built for: the weights lie in a larger buffer of NaN."""
    g = torch.Generator().manual_seed(K)
    N = 24
    buf = torch.full((N + 40, K), float("nan"), dtype=torch.bfloat16, device="cuda")
    w = buf[:N]
    w.copy_(torch.randn(N, K, generator=g) * K ** -0.5)
    x, nw = torch.randn(1, K, generator=g).bfloat16().cuda(), torch.ones(K, dtype=torch.bfloat16, device="cuda")
    with torch.no_grad():
        assert row_norm_ok(x, nw, None, w)
        y, _ = row_norm_linear(x, nw, 1e-5, None, w, gated)
        ref = rms_norm(x, nw, 1e-5, None)[0].double() @ w.double().t()
    if gated:
        ref = torch.nn.functional.silu(ref[:, :N // 2]) * ref[:, N // 2:]
    assert ((y.double() - ref).abs() <= 1.01 * 2.0 ** -8 * ref.abs() + 2e-5 * max(1.0, float(ref.abs().max()))).all()


@pytest.mark.parametrize("dtype,ulp", [(torch.bfloat16, 2.0 ** -8), (torch.float16, 2.0 ** -11)])
@pytest.mark.parametrize("K,N", [(8, 3), (520, 12), (1024, 4096), (2048, 20000), (2104, 65), (3072, 52), (5640, 32), (8192, 4100)])
def test_row_of_a_stream(K, N, dtype, ulp):
    """An fp32 row that a sublayer's output joins, or alone; bias, activation, fp32 results."""
    from lumen.ops.gemm import row_stream_linear, row_stream_ok

    g = torch.Generator().manual_seed(K + N)
    f = lambda *s: torch.randn(*s, generator=g).cuda()  # noqa: E731
    x, y, nw, w, b = 3 * f(1, K), f(1, K).to(dtype), 1 + 0.1 * f(K), (f(N, K) * K ** -0.5).to(dtype), f(N).to(dtype)
    for yy, bias, act, out32 in ((y, None, None, False), (y, b, "relu2", False), (None, None, None, True), (y, b, "silu", True)):
        keep = x.clone()
        with torch.no_grad():
            assert row_stream_ok(x, yy, nw, w, bias)
            z, s = row_stream_linear(x, yy, nw, 1e-6, w, bias, act, out32)
        assert torch.equal(x, keep) and (s is x if yy is None else torch.equal(s, x + yy.float()))
        n = s.double() / torch.sqrt(s.double().square().mean(-1, keepdim=True) + 1e-6) * nw.double()
        # the normed row is rounded once: a neighbour of the float64 one where they lie on both sides of a tie
        ref = n.float().to(dtype).double() @ w.double().t()
        flip = ulp * 2.0 ** -10 * (n.abs() @ w.double().abs().t())
        ref = ref + (0 if bias is None else bias.double())
        if act:
            ref = torch.relu(ref) ** 2 if act == "relu2" else torch.nn.functional.silu(ref)
        assert z.dtype == (torch.float32 if out32 else dtype)
        tol = (0 if out32 else 1.01 * ulp * ref.abs()) + (2e-5 + 4 * flip.max()) * max(1.0, float(ref.abs().max()))
        assert ((z.double() - ref).abs() <= tol).all(), (z.double() - ref).abs().max()
    assert not row_stream_ok(x, y.float(), nw, w) and not row_stream_ok(x.to(dtype), y, nw, w)
    assert not row_stream_ok(x, y, nw.to(dtype), w) and not row_stream_ok(x, y, nw, w, b[:-1])
    assert not row_stream_ok(x.expand(2, K), None, nw, w)
