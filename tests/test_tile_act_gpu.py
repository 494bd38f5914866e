"""Gated activation in the epilogue of tiled products against float64, over the edges of the tiles, and the rule that picks it."""
import pytest
import torch
import torch.nn.functional as F

from lumen.ops import moe
from lumen.ops._seqmix import DT, call

dev = "cuda"
ACTS = {"silu": F.silu, "relu": torch.relu, "gelu_tanh": lambda v: F.gelu(v, approximate="tanh"),
        "relu2": lambda v: torch.relu(v).square()}


def reference(x, w, act):
    g, u = (x.double().cpu() @ w.double().cpu().t()).chunk(2, -1)
    if isinstance(act, str):
        return ACTS[act](g) * u
    g, u = g.clamp(max=act.limit_shared), u.clamp(-act.limit_shared, act.limit_shared)
    return g * torch.sigmoid(act.slope * g) * (u + act.shift)


def bound(x, w, want, dt):
    """One rounding of the result; gate and up are off by K fp32 additions each, the activation (slope at most 1.13, squared ReLU
    2 |g|) by 2^-20 of itself (exponential and reciprocal units)."""
    K = x.shape[1]
    a = x.double().cpu().abs() @ w.double().cpu().abs().t()
    g, u = (x.double().cpu() @ w.double().cpu().t()).chunk(2, -1)
    eg, eu = (a * K * 2.0 ** -24).chunk(2, -1)
    lip = 1.2 + 2 * g.abs()
    return (want.abs() * (torch.finfo(dt).eps / 2 + 2.0 ** -20) + lip * eg * (u.abs() + 8) + (g.abs() + g * g) * eu
            + torch.finfo(dt).tiny)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("act", ["silu", "relu", "gelu_tanh", "relu2", moe.ClampedGate(1.5, 1.25, 1.7, 1.0)])
def test_tile_act(act, dt):
    for M, K, ff, lead in ((256, 64, 64, 0), (257, 128, 104, 8), (1, 192, 8, 0), (513, 320, 200, 0), (300, 256, 1000, 64)):
        g = torch.Generator().manual_seed(M + ff)
        x = torch.randn(M, K + lead, generator=g).to(dt).to(dev)[:, :K]
        w = (torch.randn(2 * ff, K, generator=g) / K ** 0.5).to(dt).to(dev)
        want = reference(x, w, act)
        tol = bound(x, w, want, dt)
        code, c = (moe.GATE_ACTS[act], (0.0,) * 3) if isinstance(act, str) else (4, (act.limit_shared, act.slope, act.shift))
        for ni in (4, 6, 8):
            y = torch.full((M, ff), 7.0, dtype=dt, device=dev)
            mid = ff // 16 * 8                                       # a range of columns; the others stay
            call("sm_tile_act", DT[dt], x, x.stride(0), w, y, M, K, ff, mid, ff, ni, code, *c)
            assert (y[:, :mid] == 7.0).all()
            assert ((y[:, mid:].double().cpu() - want[:, mid:]).abs() <= tol[:, mid:]).all(), (M, ff, ni)
        y = moe.tile_act(x, w, ff, act)
        assert ((y.double().cpu() - want).abs() <= tol).all(), (M, ff)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("act", ["silu", moe.ClampedGate(8.0, 8.0, 1.0, 1.0)])
def test_activation_is_rounded_from_full_fp32(act, dt):
    """Rows of one 1, so gate and up are exact.  The exponential is off by 2 units of 2^-24, the sum, the division and two
    products and a sum by one each: what lies 8 units and more from the middle of two 16-bit values is rounded to the nearer one."""
    K, ff = 64, 8192
    g = torch.Generator().manual_seed(5)
    x = torch.eye(K, dtype=dt, device=dev)
    w = torch.cat([torch.rand(ff, K, generator=g) * 18 - 15, torch.randn(ff, K, generator=g) * 4]).to(dt).to(dev)
    want = reference(x, w, act)
    near = want.to(dt)
    step = 2.0 ** torch.frexp(want.abs())[1].double() * torch.finfo(dt).eps / 2       # between neighbours
    apart = (step / 2 - (near.double() - want).abs()) / want.abs() > 8 * 2.0 ** -24
    apart &= want.abs() > 2 * torch.finfo(dt).tiny
    assert apart.double().mean() > 0.8
    assert (moe.tile_act(x, w, ff, act).cpu()[apart] == near[apart]).all()


def test_rounds_cover_the_columns_once():
    for M in (1, 65, 256, 257, 300, 1500, 4010, 8000, 20000, 65536):
        tm = -(-M // 256)
        for ff in (8, 104, 1408, 2816, 5632, 5640, 11000, 11008, 14336):
            at, rounds = 0, moe.act_rounds(M, ff)
            for k, (c0, c1, ni) in enumerate(rounds):
                assert c0 == at < c1 and c0 % 8 == 0
                whole = 256 // tm * 128                                  # columns of a whole round of 128-column tiles
                if (c1 - c0) % whole == 0:
                    assert ni == 8 and k == 0
                else:                                                    # the rest: one round, of the narrowest tiles that make it one
                    fits = [n for n in (4, 6, 8) if tm * -(-(c1 - c0) // (16 * n)) <= 256]
                    assert c1 == ff and ni == fits[0]
                at = c1
            assert at == ff and len(rounds) <= 2
    assert moe.act_rounds(70000, 5632) == () and not moe._act_tiles_pay(70000, 5632, 2048)
    assert moe._act_tiles_pay(4010, 5632, 2048) and not moe._act_tiles_pay(300, 11264, 4096)


@pytest.mark.gpu
def test_routes():
    x, w = torch.randn(700, 1024, device=dev).bfloat16(), torch.randn(5632, 1024, device=dev).bfloat16()
    assert moe.tile_act_ok(x, w, 2816)
    for a, b, ff, gated in ((x[:64], w, 2816, True), (x.float(), w.float(), 2816, True), (x, w, 2816, False), (x.cpu(), w.cpu(), 2816, True),
                            (x.clone().requires_grad_(), w, 2816, True), (x, w, 1408, True), (x.half(), w, 2816, True),
                            (x[:, 4:1020], w[:, 4:1020], 2816, True), (x, w.t().contiguous().t(), 2816, True)):
        assert not moe.tile_act_ok(a, b, ff, gated=gated)
    y = moe.ff_act(x, w, 2816)
    want = reference(x, w, "silu")
    assert ((y.double().cpu() - want).abs() <= bound(x, w, want, torch.bfloat16)).all()
    x[17, 300] = float("nan")
    bad = ~torch.isfinite(moe.ff_act(x, w, 2816)).all(1)
    assert bad.nonzero().flatten().tolist() == [17]
