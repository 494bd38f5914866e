"""A decode step's norm, router product and routing in one launch, against the separate launches and float64."""
import pytest
import torch

from lumen.ops import moe
from lumen.ops.moe import dyt_residual_routed, residual_rms_routed, route_groups_ref, route_topk_ref, routed_groups
from lumen.ops.norm import dyt_residual, residual_rms

pytestmark = pytest.mark.gpu


def _rows(T, W, E, dt, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    return r, r(T, W).to(dt), (r(E, W) / W ** 0.5).to(dt), r(E).to(dt)


@pytest.fixture
def calls(monkeypatch):
    n, run = [], moe._route_rows
    monkeypatch.setattr(moe, "_route_rows", lambda *a, **k: (n.append(a[0]), run(*a, **k))[1])
    return n


def _same(got, want, top):
    # logits' fp32 sums in another order: 1e-5 of a weight of one
    assert (got.double() - want).abs().max() < 1e-5
    assert ((got != 0).sum(1) <= top).all()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,W,E,top", [(1, 8, 1, 1), (5, 520, 3, 2), (64, 2048, 16, 3), (2, 1024, 64, 8),
                                       (7, 4096, 33, 4), (3, 8192, 9, 9), (1, 2056, 8, 2)])
def test_given_rows(T, W, E, top, dt, calls):
    r, h, R, _ = _rows(T, W, E, dt)
    z = h.double() @ R.double().t()
    corr = 0.1 * r(E)
    G = 3 if E % 3 == 0 else 1
    for score, norm in (("sigmoid", True), ("softmax", False)):
        k = min(top, max(1, G - 1) * (E // G))
        got = routed_groups(h, R, corr, k, G, max(1, G - 1), 2.0, 1e-20, 2, score, norm)
        _same(got, route_groups_ref(z.float(), corr, k, G, max(1, G - 1), 2.0, 1e-20, 2, score, norm).double(), k)
        assert torch.equal(got, routed_groups(torch.cat([h, h], 1)[:, :W], R, corr, k, G, max(1, G - 1), 2.0, 1e-20, 2, score,
                                              norm))
    assert calls == [0] * 4


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,W,E,top", [(1, 8, 2, 1), (64, 2048, 8, 2), (3, 1032, 16, 3), (2, 8192, 5, 2), (9, 4096, 64, 4),
                                       (2, 2048, 16, 1), (2, 2048, 17, 1), (3, 1024, 32, 2), (3, 1024, 33, 2), (1, 2048, 60, 3)])
def test_with_the_norm(T, W, E, top, dt, calls):
    r, y, R, b = _rows(T, W, E, dt)
    x0, w = r(T, W), 1 + 0.1 * r(W)
    ulp = 2.0 ** -7 if dt == torch.bfloat16 else 2.0 ** -10
    x, xs = x0.clone(), x0.clone()
    h, wt = residual_rms_routed(x, y, w, 1e-6, R, top, normalize=False)
    hs = residual_rms(xs, y, w, 1e-6)
    assert torch.equal(x, xs)
    assert ((h.float() - hs.float()).abs() <= ulp * hs.float().abs()).all()       # a root's last bit, then rounded
    _same(wt, route_groups_ref((h.double() @ R.double().t()).float(), None, top, 1, 1, 1.0, normalize=False).double(), top)
    norm = lambda: (1 + 0.1 * r(W), 0.1 * r(W), 0.5 + 0.1 * r(()).abs())  # noqa: E731
    post, pre = norm(), norm()
    x, xs = x0.clone(), x0.clone()
    x2, h, wt = dyt_residual_routed(x, y, post, pre, R, b, top, dt)
    _, hs = dyt_residual(xs, y, post, pre, dt)
    assert x2 is x and torch.equal(x, xs) and torch.equal(h, hs)
    _same(wt, route_topk_ref(h.double() @ R.double().t() + b.double(), top).double(), top)
    assert calls == [1, 2]


def test_other_rows_keep_the_separate_launches(calls):
    r, h, R, _ = _rows(4, 64, 8, torch.bfloat16)
    for hh, RR in ((h[:, ::2], R[:, :32].contiguous()), (h.float(), R.float()), (torch.cat([h] * 17), R),
                   (h, r(72, 64).bfloat16())):
        z = (hh.double() @ RR.double().t()).float()
        _same(routed_groups(hh, RR, None, 2, 1, 1), route_groups_ref(z, None, 2, 1, 1, 1.0).double(), 2)
    assert calls == []
    with pytest.raises(ValueError):
        routed_groups(h, R, None, 2, 3, 1)
