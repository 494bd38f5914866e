"""Products on one round of 256 x 32 ni tiles against float64, over the edges of the tiles, and the rule that picks them."""
import pytest
import torch

from lumen.ops import gemm
from lumen.ops._native import native

dev = "cuda"


def bound(x, w, b, dt):
    """float64 result and what one rounding to dt and K + 1 fp32 additions of exact products may differ by."""
    xd, wd = x.double().cpu(), w.double().cpu()
    want, mag = xd @ wd.t(), xd.abs() @ wd.abs().t()
    if b is not None:
        want, mag = want + b.double().cpu(), mag + b.double().cpu().abs()
    return want, want.abs() * torch.finfo(dt).eps / 2 + mag * (x.shape[1] + 1) * 2.0 ** -24 + torch.finfo(dt).tiny


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("ni", [3, 4, 5, 6])
@pytest.mark.parametrize("M,N,K,lead,bias", [(256, 192, 64, 0, False), (257, 100, 128, 8, True), (1, 4, 192, 0, True),
                                             (513, 388, 256, 64, False), (300, 1004, 320, 0, True), (2049, 160, 576, 0, False)])
def test_tile_gemm(M, N, K, lead, bias, ni, dt):
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K + lead, generator=g).to(dt).to(dev)[:, :K]       # rows of a wider buffer
    w = torch.randn(N, K + lead, generator=g).to(dt).to(dev)[:, :K]
    b = torch.randn(N, generator=g).to(dt).to(dev) if bias else None
    want, tol = bound(x, w, b, dt)
    assert ((native().tile_gemm(x, w, ni, b).double().cpu() - want).abs() <= tol).all()
    for at in (8, 4):                                                     # into columns: 16-byte and 8-byte stores
        y = torch.full((M, N + 16), 7.0, dtype=dt, device=dev)
        native().tile_gemm(x, w, ni, b, y[:, at:at + N])
        assert ((y[:, at:at + N].double().cpu() - want).abs() <= tol).all()
        assert (y[:, :at] == 7.0).all() and (y[:, at + N:] == 7.0).all()


@pytest.mark.gpu
def test_refused():
    x, w = torch.randn(300, 128, device=dev).bfloat16(), torch.randn(64, 128, device=dev).bfloat16()
    for bad in (lambda: native().tile_gemm(x, w, 2), lambda: native().tile_gemm(x, w, 7),
                lambda: native().tile_gemm(x, w[:, :64], 4), lambda: native().tile_gemm(x, w.half(), 4),
                lambda: native().tile_gemm(x[:, :96], w[:, :96], 4), lambda: native().tile_gemm(x, w[:62], 4),
                lambda: native().tile_gemm(x, w, 4, w[0, :32]), lambda: native().tile_gemm(x.cpu(), w.cpu(), 4),
                lambda: native().tile_gemm(x, w, 4, None, torch.empty(300, 60, device=dev).bfloat16())):
        with pytest.raises((ValueError, RuntimeError)):
            bad()


def test_columns_rule():
    for M in (256, 300, 512, 1000, 2048, 4010, 8000, 70000):
        for N in (64, 512, 1536, 2048, 2112, 3072, 5632, 11264, 22528):
            ni = gemm.tile_columns(M, N, 2048)
            if ni:
                round_ = -(-M // 256) * -(-N // (32 * ni))
                assert 3 <= ni <= 6 and round_ <= 256 and M * N >= 0.75 * 256 * 8192 * ni
    assert gemm.tile_columns(255, 22528, 2048) == 0 and gemm.tile_columns(4010, 2048, 448) == 0
    assert gemm.tile_columns(4010, 2048, 2048) == 4 and gemm.tile_columns(4010, 4096, 2048) == 0


@pytest.mark.gpu
def test_routes():
    x, w = torch.randn(4010, 512, device=dev).bfloat16(), torch.randn(2112, 512, device=dev).bfloat16()
    b = torch.randn(2112, device=dev).bfloat16()
    assert gemm.tile_ok(x, w) == 5
    for a, c in ((x[:200], w), (x.float(), w.float()), (x.cpu(), w.cpu()), (x, w.t().contiguous().t()), (x.half(), w),
                 (x[:, 1:449], w[:, 1:449]), (x.clone().requires_grad_(), w), (x[:, :500], w[:, :500])):
        assert gemm.tile_ok(a, c) == 0
    want, tol = bound(x, w, b, torch.bfloat16)
    assert ((gemm.project(x, w, b).double().cpu() - want).abs() <= tol).all()
    want, tol = bound(x, w, None, torch.bfloat16)
    assert ((gemm.project(x, w).double().cpu() - want).abs() <= tol).all()
    x[17, 300] = float("inf")
    bad = ~torch.isfinite(gemm.matmul_nt(x, w)).all(1)
    assert bad.nonzero().flatten().tolist() == [17]
    n1 = gemm.round_cols(4010, 5632, 4096)                                # one wave of the library's and one of tiles
    assert n1 == 4096 and gemm.tile_columns(4010, 5632 - n1, 4096) == 3
    assert gemm.round_cols(4010, 4096, 4096) == gemm.round_cols(4010, 8192, 4096) == gemm.round_cols(3000, 9216, 4096) == 0
    x, w = torch.randn(4010, 4096, device=dev).half(), torch.randn(5632, 4096, device=dev).half()
    assert gemm._split_plan(x, w) == n1
    y = gemm.mm_nt(x, w)
    for c in (0, n1 - 8, n1, 5616):
        want, tol = bound(x[:64], w[c:c + 16], None, torch.float16)
        assert ((y[:64, c:c + 16].double().cpu() - want).abs() <= tol).all()
