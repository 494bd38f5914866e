"""The few-row GEMM (seqmix/thin_gemm.hip) against float64 at the edges of its tiles: rows 1 .. 64
around every row class, columns that end inside a tile, k ranges with fewer stages than waves, strided
rows, bias, fp32 results; and the rule that sends a projection to it."""
import pytest
import torch

from launches import launches
from lumen.ops.gemm import project, thin_linear, thin_ok
from lumen.ops.moe import (ClampedGate, gated_act_ref, moe_dense, scaled_act_ref, thin_act,
                           thin_act_ok)

pytestmark = pytest.mark.gpu


def bound(x, w, out_bits):
    """fp32 accumulation in any order: K ulp of the sum of absolute products; then one rounding."""
    mag = x.double().abs() @ w.double().abs().t()
    return mag * x.shape[1] * 2.0 ** -24 * 2, 2.0 ** -out_bits


@pytest.mark.parametrize("dtype,bits", [(torch.bfloat16, 8), (torch.float16, 11)])
@pytest.mark.parametrize("M", [1, 2, 8, 9, 16, 17, 32, 33, 63, 64])
@pytest.mark.parametrize("N,K", [(4, 64), (16, 64), (20, 128), (60, 448), (256, 512), (1028, 704),
                                 (2048, 5632), (8196, 256), (8192, 4096)])
def test_thin_linear(M, N, K, dtype, bits):
    g = torch.Generator(device="cuda").manual_seed(M * 131 + N + K)
    x = torch.randn(M, K + 24, device="cuda", generator=g).to(dtype)[:, 8:8 + K]
    w = (torch.randn(N, K, device="cuda", generator=g) / K ** 0.5).to(dtype)
    b = torch.randn(N, device="cuda", generator=g).to(dtype)
    exact = x.double() @ w.double().t()
    acc, ulp = bound(x, w, bits)
    y = thin_linear(x, w)
    assert ((y.double() - exact).abs() <= acc + exact.abs() * ulp + 1e-30).all()
    y = thin_linear(x, w, b, torch.float32)
    want = exact + b.double()
    assert y.dtype == torch.float32
    assert ((y.double() - want).abs() <= acc + want.abs() * 2.0 ** -23).all()


def test_rows_do_not_mix_and_non_finite_rows_stay_theirs():
    x = torch.randn(11, 256, device="cuda").bfloat16()
    x[3, 5], x[7, 9] = float("inf"), float("nan")
    w = torch.randn(96, 256, device="cuda").bfloat16()
    y, ref = thin_linear(x, w), x.float() @ w.float().t()
    keep = [i for i in range(11) if i not in (3, 7)]
    assert torch.isfinite(y[keep]).all()
    assert torch.equal(torch.isnan(y[[3, 7]]), torch.isnan(ref[[3, 7]]))
    assert torch.equal(y[keep], thin_linear(x, w)[keep])


def test_the_rule_and_what_it_leaves_to_the_library():
    w = torch.randn(128, 256, device="cuda").bfloat16()
    x = torch.randn(5, 512, device="cuda").bfloat16()
    assert thin_ok(x[:, :256], w)
    for xs, ws in ((x[:, 4:260], w), (x[:, ::2], w), (x[:, :256], w[::2]), (x[:, :256], w[:126]),
                   (x[:, :250], w[:, :250].contiguous()), (x[:0, :256], w),
                   (x[:, :256].float(), w.float()), (x[:, :256].half(), w)):
        assert not thin_ok(xs, ws)
        if xs.dtype == ws.dtype:
            torch.testing.assert_close(project(xs, ws), torch.nn.functional.linear(xs, ws))
    assert not thin_ok(torch.randn(65, 256, device="cuda").bfloat16(), w)


def test_captured_call_replays_on_new_rows():
    x = torch.randn(3, 512, device="cuda").bfloat16()
    w = torch.randn(640, 512, device="cuda").bfloat16()
    thin_linear(x, w)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = thin_linear(x, w)
    for _ in range(3):
        x.copy_(torch.randn(3, 512, device="cuda"))
        graph.replay()
        assert torch.equal(y, thin_linear(x, w))


def routed(M, E, top, g):
    """[M, E] weights with ``top`` non-zero ones a row."""
    idx = torch.rand(M, E, device="cuda", generator=g).topk(top, 1).indices
    return torch.zeros(M, E, device="cuda").scatter_(
        1, idx, 0.2 + torch.rand(M, top, device="cuda", generator=g))


@pytest.mark.parametrize("dtype,tol", [(torch.bfloat16, 2.0 ** -8), (torch.float16, 2.0 ** -11)])
@pytest.mark.parametrize("act,gated,weigh", [("silu", True, "output"), ("relu", True, "output"),
                                             (ClampedGate(1.0, 0.7, 1.702, 1.0), True, "input"),
                                             ("relu2", False, "output")])
@pytest.mark.parametrize("M,E,top,ff,ffs", [(1, 17, 3, 64, 128), (3, 8, 2, 128, 0), (8, 16, 4, 192, 64),
                                            (17, 5, 1, 48, 32), (32, 64, 2, 64, 64), (9, 0, 0, 0, 208)])
def test_act_and_skipped_experts(M, E, top, ff, ffs, act, gated, weigh, dtype, tol):
    g = torch.Generator(device="cuda").manual_seed(M * 7 + E)
    K, k, W = 320, 2 if gated else 1, 96
    h = torch.randn(M, K, device="cuda", generator=g).to(dtype)
    gu = (torch.randn(k * (E * ff + ffs), K, device="cuda", generator=g) / K ** 0.5).to(dtype)
    down = torch.randn(W, E * ff + ffs, device="cuda", generator=g).to(dtype)
    wts = routed(M, E, top, g) if E else None
    fn = gated_act_ref if gated else scaled_act_ref
    args = (act, weigh) if gated else (act,)
    want = fn(h.double() @ gu.double().t(), wts, E, ff, ffs, *args).double()   # (fp32 formulas)
    assert thin_act_ok(h, wts, gu, E, ff, ffs, act, gated, weigh)
    a = thin_act(h, gu, wts, E, ff, ffs, act, gated, weigh)
    # one rounding to 16 bits; the fp32 sums and the activation add 1e-5 of the sums' size (~1)
    assert ((a.double() - want).abs() <= want.abs() * tol + 4e-5).all()
    ref = a.double() @ down.double().t()
    y = moe_dense(h, wts, gu, down, E, ff, ffs, act, gated, weigh, top or None)
    slack = (a.double().abs() @ down.double().abs().t()) * 1e-5
    assert ((y.double() - ref).abs() <= slack + ref.abs() * tol).all()
    # blocks nobody chose may hold anything: they are neither read nor multiplied
    if E and ff % 64 == 0 and ffs % 64 == 0:
        dead = (wts == 0).all(0).nonzero().flatten().tolist()
        for e in dead:
            gu[e * k * ff:(e + 1) * k * ff] = float("nan")
            down[:, e * ff:(e + 1) * ff] = float("nan")
        if M * top <= 3 * E:
            assert torch.equal(moe_dense(h, wts, gu, down, E, ff, ffs, act, gated, weigh, top), y)


def test_no_chosen_expert_gives_the_shared_one_alone():
    h = torch.randn(2, 128, device="cuda").bfloat16()
    gu = torch.randn(2 * (4 * 64 + 64), 128, device="cuda").bfloat16()
    down = torch.randn(32, 4 * 64 + 64, device="cuda").bfloat16()
    wts = torch.zeros(2, 4, device="cuda")
    y = moe_dense(h, wts, gu, down, 4, 64, 64, top=1)
    ref = moe_dense(h, None, gu[512:], down[:, 256:].contiguous(), 0, 0, 64)
    assert torch.equal(y, ref)
    assert not moe_dense(h, wts, gu[:512], down[:, :256].contiguous(), 4, 64, 0, top=1).any()


def test_one_row_of_a_wide_model_skips_experts():
    """Width 4096, where one dense row goes to the GEMV: experts nobody chose may hold anything."""
    g = torch.Generator(device="cuda").manual_seed(4)
    K, E, top, ff, ffs, W = 4096, 16, 3, 64, 128, 64
    h = torch.randn(1, K, device="cuda", generator=g).bfloat16()
    gu = (torch.randn(2 * (E * ff + ffs), K, device="cuda", generator=g) / K ** 0.5).bfloat16()
    down = torch.randn(W, E * ff + ffs, device="cuda", generator=g).bfloat16()
    wts = routed(1, E, top, g)
    a = gated_act_ref(h.double() @ gu.double().t(), wts, E, ff, ffs).bfloat16().double()
    ref = a @ down.double().t()
    for e in (wts == 0).all(0).nonzero().flatten().tolist():
        gu[e * 2 * ff:(e + 1) * 2 * ff] = float("nan")
        down[:, e * ff:(e + 1) * ff] = float("nan")
    y = moe_dense(h, wts, gu, down, E, ff, ffs, top=top)
    # each activation may round to the other side (2^-7 of it at most, two neighbours), then the result rounds
    slack = (a.abs() @ down.double().nan_to_num().abs().t()) * 2.0 ** -7
    assert ((y.double() - ref).abs() <= slack + ref.abs() * 2.0 ** -8).all()


@pytest.mark.parametrize("dtype,bits", [(torch.bfloat16, 8), (torch.float16, 11)])
@pytest.mark.parametrize("M", [9, 17, 31, 33, 49, 64])
@pytest.mark.parametrize("N,K", [(256, 4096), (260, 192), (2112, 320), (2116, 320), (2052, 128), (5000, 192)])
def test_rows_in_groups(M, N, K, dtype, bits):
    """Few tiles: the rows are cut into groups of 16 or 32 with workgroups of their own."""
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn(M, K + 8, device="cuda", generator=g).to(dtype)[:, :K]
    w = (torch.randn(N, K, device="cuda", generator=g) / K ** 0.5).to(dtype)
    y, exact = thin_linear(x, w), x.double() @ w.double().t()
    acc, ulp = bound(x, w, bits)
    assert ((y.double() - exact).abs() <= acc + exact.abs() * ulp + 1e-30).all()


@pytest.mark.parametrize("dtype,bits", [(torch.bfloat16, 8), (torch.float16, 11)])
@pytest.mark.parametrize("M", [1, 7, 8, 9, 16])
@pytest.mark.parametrize("N,K", [(4, 1024), (12, 1088), (2044, 1024), (2048, 1536), (2052, 1024), (40, 4096)])
def test_tiles_of_eight_columns(M, N, K, dtype, bits):
    """Up to 2048 columns of 1024 and more."""
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn(M, K + 8, device="cuda", generator=g).to(dtype)[:, :K]
    w = (torch.randn(N, K, device="cuda", generator=g) / K ** 0.5).to(dtype)
    b = torch.randn(N, device="cuda", generator=g).to(dtype)
    want = x.double() @ w.double().t() + b.double()
    acc, ulp = bound(x, w, bits)
    y = thin_linear(x, w, b)
    assert ((y.double() - want).abs() <= acc + want.abs() * (ulp + 2.0 ** -22) + 1e-30).all()
    E, ff, ffs = 15, K // 16 // 64 * 64, K - 15 * (K // 16 // 64 * 64)
    wts = torch.zeros(M, E, device="cuda")
    wts[0, 3], wts[M - 1, E - 1] = 0.5, 0.5
    on = torch.zeros(E, dtype=torch.bool, device="cuda")
    on[3] = on[E - 1] = True
    seen = torch.cat([on.repeat_interleave(ff), torch.ones(ffs, dtype=torch.bool, device="cuda")])
    want = (x.double() * seen) @ w.double().t()
    y = thin_linear(x, w.masked_fill(~seen, float("nan")), None, torch.float32, (wts, E, ff, ffs))
    assert ((y.double() - want).abs() <= acc + want.abs() * 2.0 ** -23).all()


@pytest.mark.parametrize("dtype,tol", [(torch.bfloat16, 2.0 ** -8), (torch.float16, 2.0 ** -11)])
@pytest.mark.parametrize("M,K,ff", [(1, 1024, 4112), (8, 1088, 6144), (9, 1024, 4112), (16, 1024, 6144), (16, 1024, 6160), (7, 1024, 8208)])
def test_gated_tiles_of_eight_columns(M, K, ff, dtype, tol):
    """One and two rounds of 16-column tiles and up to half of another."""
    g = torch.Generator(device="cuda").manual_seed(M + ff)
    h = torch.randn(M, K, device="cuda", generator=g).to(dtype)
    w = (torch.randn(2 * ff, K, device="cuda", generator=g) / K ** 0.5).to(dtype)
    z = h.double() @ w.double().t()
    for act in ("silu", ClampedGate(1.0, 0.7, 1.702, 1.0)):
        got = thin_act(h, w, None, 0, 0, ff, act, True, "output").double()
        gate, up = z[:, :ff], z[:, ff:]
        if act == "silu":
            want = gate * torch.sigmoid(gate) * up
        else:
            gate, up = gate.clamp(max=act.limit_shared), up.clamp(-act.limit_shared, act.limit_shared)
            want = gate * torch.sigmoid(act.slope * gate) * (up + act.shift)
        assert ((got - want).abs() <= 1.05 * tol * want.abs() + 2e-5 * want.abs().max()).all()


@pytest.mark.parametrize("M,N,K,grid", [(17, 2048, 512, (128, 2)), (32, 2048, 2048, (128, 2)), (17, 2052, 512, (129, 1)), (32, 2112, 1024, (132, 1)),
                                        (33, 2048, 512, (128, 2)), (64, 2052, 512, (65, 2))])
def test_groups_of_rows_where_each_has_a_cu(M, N, K, grid):
    """17 - 32 rows go in two groups of 16 while all of their workgroups have a CU each."""
    x, w = torch.randn(M, K, device="cuda").bfloat16(), torch.randn(N, K, device="cuda").bfloat16()
    (name, g, _), = launches(lambda: thin_linear(x, w))
    assert "thin_kernel" in name and g[:2] == grid
    want = x.double() @ w.double().t()
    acc, ulp = bound(x, w, 8)
    assert ((thin_linear(x, w).double() - want).abs() <= acc + want.abs() * ulp).all()


@pytest.mark.parametrize("M,N,K,waves", [(1, 256, 64, 4), (8, 64, 960, 4), (8, 256, 1024, 8), (9, 16, 512, 4), (16, 256, 960, 4), (17, 256, 768, 4),
                                         (17, 128, 832, 8), (32, 16, 64, 4), (33, 64, 448, 4), (64, 256, 768, 4), (64, 256, 832, 8), (63, 256, 4096, 8)])
def test_waves_of_small_matrices(M, N, K, waves):
    """Eight waves of a workgroup want more than three stages of 64 for each pair of them."""
    x, w = torch.randn(M, K, device="cuda").bfloat16(), torch.randn(N, K, device="cuda").bfloat16()
    (name, _, block), = launches(lambda: thin_linear(x, w))
    assert "thin_kernel" in name and block[0] == 64 * waves
    want = x.double() @ w.double().t()
    acc, ulp = bound(x, w, 8)
    assert ((thin_linear(x, w).double() - want).abs() <= acc + want.abs() * ulp).all()


@pytest.mark.parametrize("M,N,K,grid", [(33, 4096, 128, (128, 2)), (33, 4112, 128, (256, 1)), (64, 4100, 960, (256, 1)), (64, 4112, 1024, (129, 2)),
                                        (33, 8188, 64, (256, 1)), (64, 7680, 1024, (240, 2)), (33, 7684, 1024, (256, 1)), (64, 1996, 256, (125, 2)), (20, 112, 832, (7, 2)),
                                        (64, 128, 832, (8, 4)), (50, 140, 832, (9, 4)), (64, 2404, 512, (76, 2))])
def test_groups_of_rows_past_a_round_of_columns(M, N, K, grid):
    """33 - 64 rows of more than 4096 columns go in two groups from k of 1024 on, up to 7680; later groups start some tiles on."""
    x, w = torch.randn(M, K, device="cuda").bfloat16(), torch.randn(N, K, device="cuda").bfloat16()
    (name, g, _), = launches(lambda: thin_linear(x, w))
    assert "thin_kernel" in name and g[:2] == grid
    want = x.double() @ w.double().t()
    acc, ulp = bound(x, w, 8)
    assert ((thin_linear(x, w).double() - want).abs() <= acc + want.abs() * ulp).all()
