"""Projections of up to 64 rows on one shared ring per workgroup: sums over slices of K that meet in a norm, and the
activation in the epilogue, against float64."""
import pytest
import torch

from lumen.ops import gemm, moe, norm
from lumen.ops.moe import ClampedGate, ff_act, gated_act_ref, mid_act, mid_act_ok, scaled_act_ref
from lumen.ops.norm import group_rms_norm_ref, project_group_rms

pytestmark = pytest.mark.gpu
ULP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _rows(M, K, N, dt, pad=0):
    g = torch.Generator(device="cuda").manual_seed(M * 7 + K)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    return r, r(M, K + pad).to(dt)[:, :K], (r(N, K) / K ** 0.5).to(dt)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K,groups,pad", [(2, 1024, 128, 4, 0), (7, 2048, 384, 1, 8), (16, 256, 1152, 1, 0),
                                              (17, 3072, 640, 4, 0), (63, 8192, 256, 2, 0), (64, 2048, 5632, 4, 16),
                                              (33, 4096, 512, 16, 0)])
def test_slices_and_norm(M, N, K, groups, pad, dt, monkeypatch):
    n, run = [], gemm.mid_slabs
    monkeypatch.setattr(gemm, "mid_slabs", lambda *a: (n.append(1), run(*a))[1])
    r, a, w = _rows(M, K, N, dt, pad)
    x0, nw = r(M, N), 1 + 0.1 * r(N)
    y = a.double() @ w.double().t()
    assert (run(a, w).double().sum(0) - y).abs().max() < 3e-6 * y.abs().max() * K ** 0.5
    want = x0.double() + group_rms_norm_ref(y, nw, groups, 1e-6, torch.float64)
    for cast in (dt, None, torch.float32):
        x = x0.clone()
        got, xb = project_group_rms(x, a, w, nw, groups, 1e-6, cast)
        assert got is x and (xb is None) == (cast is not dt)
        assert (x.double() - want).abs().max() < 1e-5 * want.abs().max()          # fp32 sums
        if xb is not None:
            assert torch.equal(xb, x.to(dt))
    assert len(n) == 3


def test_other_shapes_keep_the_separate_launches(monkeypatch):
    monkeypatch.setattr(gemm, "mid_slabs", None)
    for M, N, K, groups in ((1, 1024, 128, 1), (65, 1024, 128, 1), (4, 1024, 64, 1), (4, 1024, 128, 8), (4, 320, 128, 1)):
        r, a, w = _rows(M, K, N, torch.bfloat16)
        x0, nw = r(M, N), 1 + 0.1 * r(N)
        x, xb = project_group_rms(x0.clone(), a, w, nw, groups, 1e-6, torch.bfloat16)
        want = x0.double() + group_rms_norm_ref(a.double() @ w.double().t(), nw, groups, 1e-6, torch.float64)
        assert (x.double() - want).norm() < 4e-3 * want.norm()                    # the product is rounded in between


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,ff,K,pad", [(33, 4, 128, 0), (48, 36, 256, 8), (64, 5632, 2048, 0), (34, 100, 640, 0),
                                        (17, 4128, 384, 0), (64, 8192, 128, 0)])
def test_activation(M, ff, K, pad, dt):
    for gated, act in ((True, "silu"), (True, "relu"), (True, "gelu_tanh"), (True, ClampedGate(7.0, 2.0, 1.702, 1.0)),
                       (False, "relu2"), (False, "silu")):
        r, h, w = _rows(M, K, (2 if gated else 1) * ff, dt, pad)
        z = (h.double() @ w.double().t())
        ref = gated_act_ref if gated else scaled_act_ref
        want = ref(z.float(), None, 0, 0, ff, act).double()
        got = mid_act(h, w, ff, act, gated)
        # one rounding of the result, fp32 sums through the activation
        assert ((got.double() - want).abs() <= ULP[dt] * want.abs() + 3e-5 * want.abs().max()).all(), (gated, act)
        if mid_act_ok(h, w, ff, act, gated):
            assert torch.equal(ff_act(h, w, ff, act, gated), got)


def test_rules():
    _, h, w = _rows(33, 1024, 2 * 8224, torch.bfloat16)
    assert not mid_act_ok(h, w, 8224)                       # 257 tiles
    assert mid_act_ok(h, w[:2 * 8192], 8192) and not mid_act_ok(h[:17], w[:2 * 4064], 4064)
    assert mid_act_ok(h[:17], w[:2 * 4096], 4096) and not mid_act_ok(h[:16], w[:2 * 4096], 4096)
    assert not mid_act_ok(h.float(), w[:2 * 8192].float(), 8192) and not mid_act_ok(h[:, :512], w[:2 * 8192, :512].contiguous(), 8192)
    assert moe.MID_MAX_M == 64 and norm.project_group_rms is project_group_rms
