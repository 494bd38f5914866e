"""Split-K GEMM against float64, over the edges of its tiles and slices, and the rule that picks it."""
import pytest
import torch

from lumen.ops import gemm
from lumen.ops._native import native

pytestmark = pytest.mark.gpu
dev = "cuda"


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K,S", [(65, 128, 128, 2), (256, 128, 128, 2), (257, 132, 192, 3), (300, 388, 576, 4),
                                     (513, 260, 1088, 8), (1, 4, 320, 5), (512, 4096, 8192, 4), (700, 1000, 512, 2)])
def test_split_gemm(M, N, K, S, dt):
    g = torch.Generator().manual_seed(M + K)
    x = torch.randn(M, K + 8, generator=g).to(dt).to(dev)[:, :K]          # rows of a wider buffer
    w = torch.randn(N, K, generator=g).to(dt).to(dev)
    y = native().split_gemm(x, w, S)
    xd, wd = x.double().cpu(), w.double().cpu()
    want, mag = xd @ wd.t(), xd.abs() @ wd.abs().t()
    # one rounding to dt, and K fp32 additions of products that are exact in fp32
    tol = want.abs() * torch.finfo(dt).eps / 2 + mag * K * 2.0 ** -24 + torch.finfo(dt).tiny
    assert ((y.double().cpu() - want).abs() <= tol).all()


def test_non_finite_stays_in_its_row():
    x = torch.randn(300, 8192, device=dev).bfloat16()
    w = torch.randn(2048, 8192, device=dev).bfloat16()
    x[17, 5000] = float("nan")
    S = gemm.split_slices(x, w)
    assert S > 1
    bad = ~torch.isfinite(gemm.split_linear(x, w, S)).all(1)
    assert bad.nonzero().flatten().tolist() == [17]


def test_rule():
    x, w = torch.randn(512, 8192, device=dev).bfloat16(), torch.randn(4096, 8192, device=dev).bfloat16()
    assert gemm.split_slices(x, w) == 4
    for a, b in ((x[:64], w), (x[:, :8128], w[:, :8128]), (x.float(), w.float()), (x.cpu(), w.cpu()),
                 (x, w.t().contiguous().t()), (x, w[:256]), (x, w.repeat(2, 1)[:, :]), (x.half(), w)):
        s = gemm.split_slices(a, b)
        assert s == (2 if b.shape[0] == 8192 else 0)
    xr = x.clone().requires_grad_()
    y = gemm.mm_nt(xr, w)
    assert gemm.split_slices(xr, w) == 0 and y.requires_grad          # differentiable: the library's
    with torch.no_grad():
        assert gemm.split_slices(xr, w) == 4
        got = gemm.mm_nt(xr, w)
    # both round one fp32-accumulated product: at most one unit apart plus the sums' own error
    ref = x.double() @ w.double().t()
    tol = ref.abs() * 2.0 ** -9 + (x.double().abs() @ w.double().abs().t()) * 8192 * 2.0 ** -24
    assert ((got.double() - ref).abs() <= tol).all()
    assert torch.equal(torch.func.vmap(lambda v: gemm.matmul_nt(v, w))(x[None]), torch.matmul(x[None], w.t()))


@pytest.mark.parametrize("M,N,K", [(4010, 11264, 2048), (1900, 22016, 2048), (2305, 16384, 4096)])
def test_whole_wave_columns(M, N, K):
    x = torch.randn(M, K, device=dev).bfloat16()
    w = torch.randn(N, K, device=dev).bfloat16()
    n1 = gemm.wave_cols(M, N, K)
    assert n1 and gemm._split_plan(x, w) == n1
    y = gemm.mm_nt(x, w)
    for c in (0, n1 - 8, N - 8):                                # both sides of the cut, and the last columns
        xd, wd = x.double(), w[c:c + 16].double()
        want, mag = xd @ wd.t(), xd.abs() @ wd.abs().t()
        tol = want.abs() * 2.0 ** -8 + mag * K * 2.0 ** -24     # one rounding, K fp32 additions
        assert ((y[:, c:c + 16].double() - want).abs() <= tol).all()
    assert gemm._split_plan(x.requires_grad_(), w) == 0         # differentiable: in one piece
