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
    for a, c in ((x[:64], w), (x.float(), w.float()), (x.cpu(), w.cpu()), (x, w.t().contiguous().t()), (x.half(), w),
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


# 64- and 128-row tiles: one row and one past a tile, columns past one, fewer stages of k than the ring has and more, walks apart
@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("mj,ni", [(2, 1), (2, 2), (2, 3), (2, 4), (2, 5), (2, 6), (2, 8), (4, 2), (4, 3), (4, 4), (4, 5), (4, 6), (4, 8),
                                   (8, 3), (8, 4)])
@pytest.mark.parametrize("M,N,K,lead,bias", [(64, 512, 64, 0, False), (65, 260, 384, 8, True), (17, 1004, 448, 0, True),
                                             (129, 100, 128, 64, False), (257, 36, 1088, 0, True)])
def test_row_tiles(M, N, K, lead, bias, mj, ni, dt):
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K + lead, generator=g).to(dt).to(dev)[:, :K]
    w = torch.randn(N, K + lead, generator=g).to(dt).to(dev)[:, :K]
    b = torch.randn(N, generator=g).to(dt).to(dev) if bias else None
    want, tol = bound(x, w, b, dt)
    for apart in (False, True):
        y = torch.full((M, N + 16), 7.0, dtype=dt, device=dev)
        native().tile_gemm(x, w, ni, b, y[:, 4:4 + N], mj, apart)
        assert ((y[:, 4:4 + N].double().cpu() - want).abs() <= tol).all()
        assert (y[:, :4] == 7.0).all() and (y[:, 4 + N:] == 7.0).all()


def test_few_tiles_rule():
    forms = {(2, n) for n in (1, 2, 3, 4, 5, 6, 8)} | {(4, n) for n in (2, 3, 4, 5, 6, 8)} | {(8, 3)}
    for M in (1, 16, 17, 33, 64, 65, 128, 129, 176, 177, 256, 257, 500, 1000, 70000):
        for N in (64, 4096, 7168, 8192, 12288, 22016, 24576, 32000, 64000, 128256, 1 << 20):
            for K in (64, 1024, 2048, 2816, 4096, 5632, 8192):
                code = gemm.few_tiles(M, N, K)
                if code:
                    assert 17 <= M and 1024 <= K < 8192 and (code >> 4 & 15, code & 15) in forms
                    assert (code > 255) == (K % 2048 == 0 and M <= 256)
                    if M <= 256:                        # asked only for as many columns or results
                        assert N >= gemm.FEW_MIN_N
                    assert M * N >= gemm.FEW_MIN_MN or N >= gemm.FEW_MIN_N


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(33, 8192, 2048), (64, 32000, 1024), (20, 22016, 1024), (100, 24576, 2048), (200, 12288, 1024),
                                   (1000, 3072, 1024)])
def test_few_route(M, N, K):
    x, w = torch.randn(M, K, device=dev).bfloat16(), torch.randn(N, K, device=dev).bfloat16()
    b = torch.randn(N, device=dev).bfloat16()
    code = gemm.tile_ok(x, w)
    assert code == gemm.few_tiles(M, N, K) > 0
    y = native().tile_gemm(x, w, code & 15, None, None, code >> 4 & 15, code > 255)
    for out in (gemm.linear_nt(x, w), gemm.project(x, w), gemm.matmul_nt(x, w)):
        assert torch.equal(out, y)
    assert torch.equal(gemm.project(x, w, b), native().tile_gemm(x, w, code & 15, b, None, code >> 4 & 15, code > 255))
    for a, c in ((x[:, :-8], w[:, :-8]), (x.float(), w.float()), (x, w.half()), (x[:, 1:], w[:, 1:])):     # the general paths take these
        assert gemm.tile_ok(a, c) == 0


# slabs of 64- and 128-row tiles: the slices' sums over tiles' edges, and the rule's forms
@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("mj", [2, 4, 8])
@pytest.mark.parametrize("M,N,K,S", [(64, 128, 128, 2), (65, 260, 832, 12), (129, 100, 1088, 5), (17, 4, 192, 3), (200, 1000, 448, 2)])
def test_row_slices(M, N, K, S, mj, dt):
    g = torch.Generator().manual_seed(M + K)
    x, w = torch.randn(M, K, generator=g).to(dt).to(dev), torch.randn(N, K, generator=g).to(dt).to(dev)
    want, tol = bound(x, w, None, dt)
    for apart in (False, True):
        assert ((native().split_gemm(x, w, S, mj, apart).double().cpu() - want).abs() <= tol).all()


def test_split_plan_rule():
    for M in (1, 16, 17, 32, 33, 64, 65, 128, 129, 192, 193, 240, 241, 256, 257, 1000, 5000):
        for N in (4, 1024, 2048, 3072, 4096, 5120, 6144, 8192, 12288, 32000):
            for K in (64, 2048, 3072, 4096, 5632, 8192, 11264, 32768):
                code = gemm.split_plan(M, N, K)
                if code:
                    S, mj = code & 15, code >> 4 & 15 or 8
                    tiles = -(-M // (32 * mj)) * -(-N // 128)
                    assert 2 <= S <= K // 64 and mj in (2, 4, 8) and 128 <= tiles * S <= 256 and K >= 3072
                    assert code < 256 or M <= 256
    assert gemm.split_plan(512, 4096, 8192) == 4 and gemm.split_plan(64, 2048, 8192) == 12 + 32


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(64, 4096, 11008), (33, 5120, 4096), (100, 4096, 5632), (180, 3072, 8448),
                                   (64, 8192, 8192)])
def test_split_route(M, N, K):
    x, w = torch.randn(M, K, device=dev).bfloat16(), torch.randn(N, K, device=dev).bfloat16()
    code = gemm.split_plan(M, N, K)
    y = native().split_gemm(x, w, code & 15, code >> 4 & 15 or 8, code > 255)
    for out in (gemm.linear_nt(x, w), gemm.project(x, w)):
        assert torch.equal(out, y)


def test_short_tiles_rule():
    for M in (1, 64, 65, 256, 257, 300, 512, 1000, 1024, 1025, 4010):
        for N in (4, 64, 576, 1024, 2048, 5632, 11264):
            for K in (64, 128, 1024, 1536, 2048, 2112, 3072, 4096):
                code = gemm.short_tiles(M, N, K)
                if code:
                    ni = code & 15
                    assert code >> 4 == 4 and 2 <= ni <= 5 and ni * K <= 6144 and 64 < M and M * K <= 1 << 20
                    assert -(-M // 128) * -(-N // (32 * ni)) <= 256
    assert gemm.short_tiles(300, 576, 2048) == 2 + 64 and gemm.short_tiles(64, 576, 2048) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,bias", [(65, 576, 2048, True), (200, 2048, 1024, False), (257, 576, 2048, True), (300, 3072, 1024, False), (1000, 100, 128, True), (480, 2048, 2048, False)])
def test_short_route(M, N, K, bias):
    x, w = torch.randn(M, K, device=dev).bfloat16(), torch.randn(N, K, device=dev).bfloat16()
    b = torch.randn(N, device=dev).bfloat16() if bias else None
    code = gemm.short_tiles(M, N, K)
    got = gemm.project(x, w, b)
    assert code and torch.equal(got, native().tile_gemm(x, w, code & 15, b, None, 4, False))
    want, tol = bound(x, w, b, torch.bfloat16)
    assert ((got.double().cpu() - want).abs() <= tol).all()
    w.requires_grad_()                                      # differentiable: the library's
    assert gemm.project(x, w, b).requires_grad


def test_short_slices_rule():
    for M in (64, 65, 128, 300, 372, 373, 682, 1000):
        for N in (4, 1000, 1024, 2048, 3072, 4096):
            for K in (2048, 3072, 3136, 4224, 5632, 8128, 8192):
                code = gemm.short_slices(M, N, K)
                if code:
                    S = code & 15
                    assert code >> 4 == 4 and 2 <= S <= K // 64 and 64 < M and M * K <= 1 << 21 and 3072 < K < 8192
                    assert -(-M // 128) * -(-N // 128) * S <= 256
    assert gemm.short_slices(300, 2048, 5632) == 5 + 64


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(65, 2048, 5632), (300, 2048, 5632), (400, 1024, 3200)])
def test_short_slices_route(M, N, K):
    x, w = torch.randn(M, K, device=dev).bfloat16(), torch.randn(N, K, device=dev).bfloat16()
    code = gemm.short_slices(M, N, K)
    want, tol = bound(x, w, None, torch.bfloat16)
    for got in (gemm.project(x, w), gemm.linear_nt(x, w)):
        assert code and torch.equal(got, native().split_gemm(x, w, code & 15, 4, False))
        assert ((got.double().cpu() - want).abs() <= tol).all()
