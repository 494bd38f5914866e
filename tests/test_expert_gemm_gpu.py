"""Products over the rows that chose an expert (seqmix/expert_gemm.hip) against float64: tiles of 64 - 256 pairs and 128 / 256
columns and their remainders, contractions of 32 more than whole stages, experts nobody or everybody chose, rows with
fewer choices than `top`, several thousand rows, row strides, every activation, replays of a captured call."""
import pytest
import torch

from launches import launches
from lumen.ops import moe as M

pytestmark = pytest.mark.gpu


def layer(T, W, E, top, ff, ffs, gated, dtype, seed, skew=0.0):
    g = torch.Generator().manual_seed(seed)
    k = 2 if gated else 1
    h = torch.randn(T, W, generator=g).to(dtype).cuda()
    gu = (torch.randn(k * (E * ff + ffs), W, generator=g) * W ** -0.5).to(dtype).cuda()
    down = (torch.randn(W, E * ff + ffs, generator=g) * ff ** -0.5).to(dtype).cuda()
    z = torch.randn(T, E, generator=g) + skew * torch.arange(E)
    return h, M.route_topk_ref(z, top).cuda(), gu, down


def exact(h, wts, gu, down, E, ff, ffs, act, gated, weigh):
    """Every expert in float64; one expert's product at a time."""
    h, out = h.double(), 0
    for e in range(E + (ffs > 0)):
        n, k = (ff if e < E else ffs), 2 if gated else 1
        z = h @ gu[k * e * ff:k * (e * ff + n)].double().t()
        w = wts[:, e:e + 1].double() if e < E else torch.ones(1, 1, device=h.device, dtype=torch.float64)
        if not gated:
            a = M._ACT_FN[act](z) * w
        else:
            a, u = z[:, :n], z[:, n:]
            if weigh == "input":
                a, u = a * w, u * w
            if isinstance(act, str):
                a = M._ACT_FN[act](a) * u
            else:
                lim = act.limit if e < E else act.limit_shared
                a, u = a.clamp(max=lim), u.clamp(-lim, lim)
                a = a * torch.sigmoid(act.slope * a) * (u + act.shift)
            if weigh == "output":
                a = a * w
        out = out + a @ down[:, e * ff:e * ff + n].double().t()
    return out


def check(out, ref, dtype):
    # the activations' and the result's rounding, each half an ulp (rms ~0.3 ulp): 0.3 sqrt(2) ulp, doubled
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    err = (out.double() - ref).norm() / ref.norm()
    assert err < 0.85 * ulp, err


CLAMP = M.ClampedGate(0.7, 0.5, 1.7, 1.0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,W,E,top,ff,ffs,act,gated,weigh,skew", [
    (1, 64, 1, 1, 32, 0, "silu", True, "output", 0), (127, 192, 5, 2, 96, 160, "gelu_tanh", True, "output", 0),
    (129, 320, 8, 2, 128, 64, "silu", True, "input", 0), (300, 128, 6, 6, 288, 0, "relu", True, "output", 0),
    (257, 256, 16, 4, 160, 0, "relu2", False, "output", 3.0), (260, 512, 64, 3, 64, 96, CLAMP, True, "output", 0),
    (90, 1088, 7, 3, 1056, 1056, CLAMP, True, "input", 0), (5000, 64, 9, 2, 32, 32, "silu", False, "output", 0.5),
    (513, 2048, 8, 2, 1408, 1408, "silu", True, "output", 0)])
def test_chosen_experts(T, W, E, top, ff, ffs, act, gated, weigh, skew, dtype):
    h, wts, gu, down = layer(T, W, E, top, ff, ffs, gated, dtype, T + W, skew)
    if T > 1:
        wts[T // 2] = 0.0                                     # a row without experts, one with fewer
        wts[T // 3] *= wts[T // 3] == wts[T // 3].max()
    args = (E, top, ff, ffs, act, gated, weigh)
    assert M.chosen_ok(h, wts, gu, down, *args)
    out = M.moe_chosen(h, wts, gu, down, *args)
    check(out, exact(h, wts, gu, down, E, ff, ffs, act, gated, weigh), dtype)
    wide = torch.zeros(T, W + 24, dtype=dtype, device="cuda")
    wide[:, :W] = h                                           # another row stride, the same bits
    assert torch.equal(M.moe_chosen(wide[:, :W], wts, gu, down, *args), out)
    if not ffs and T > 1:
        assert not out[T // 2].any()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,W,E,top,ff,ffs,act,gated,weigh", [
    (100, 192, 8, 2, 544, 480, "gelu_tanh", True, "output"), (3000, 192, 5, 2, 1440, 800, CLAMP, True, "input"),
    (5000, 128, 9, 2, 1312, 96, "silu", True, "output"), (2500, 320, 16, 3, 1056, 0, "relu2", False, "output"),
    (6000, 64, 8, 2, 1408, 1408, "gelu_tanh", False, "output"), (40, 1024, 16, 2, 608, 0, "relu", True, "output"),
    (9000, 640, 4, 2, 288, 288, "relu2", True, "output"), (1030, 2048, 4, 1, 1408, 0, CLAMP, True, "output"),
    (1100, 704, 3, 2, 1888, 0, "silu", True, "input"), (700, 256, 4, 2, 1408, 1408, "relu", False, "output"),
    (2500, 320, 6, 3, 1056, 96, "silu", False, "output")])
def test_tiles_of_64_and_256_pairs(T, W, E, top, ff, ffs, act, gated, weigh, dtype):
    """Whole rounds of 256 pairs by 256 rows and what is left over uncut, in halves and in quarters (some of them empty), for every
    activation; 64 pairs; stages of 64 and a last one of 32."""
    h, wts, gu, down = layer(T, W, E, top, ff, ffs, gated, dtype, T + W)
    wts[T // 2] = 0.0
    out = M.moe_chosen(h, wts, gu, down, E, top, ff, ffs, act, gated, weigh)
    check(out, exact(h, wts, gu, down, E, ff, ffs, act, gated, weigh), dtype)


def test_more_choices_than_top_stay_in_bounds():
    """Weights that break the promise: a row's first `top` experts count."""
    T, W, E, top, ff = 200, 64, 8, 2, 64
    h, wts, gu, down = layer(T, W, E, 5, ff, 0, True, torch.bfloat16, 3)
    kept = wts * (torch.cumsum((wts != 0).int(), 1) <= top)
    check(M.moe_chosen(h, wts, gu, down, E, top, ff, 0), exact(h, kept, gu, down, E, ff, 0, "silu", True, "output"),
          torch.bfloat16)


def test_route_and_refusals():
    h, wts, gu, down = layer(65, 128, 4, 2, 64, 0, True, torch.bfloat16, 1)
    seen, real = [], M.moe_chosen
    M.moe_chosen = lambda *a: (seen.append(1), real(*a))[1]
    try:
        M.moe(h, wts, gu, down, 4, 2, 64, 0)
        M.moe(h[:64].contiguous(), wts[:64].contiguous(), gu, down, 4, 2, 64, 0)      # a small stack: the thin GEMM
    finally:
        M.moe_chosen = real
    assert len(seen) == 1
    for bad in ((h.float(), wts, gu, down), (h, wts.half(), gu, down), (h, wts, gu[:-1], down), (h, wts, gu, down.t())):
        assert not M.chosen_ok(*bad, 4, 2, 64, 0)
        with pytest.raises(ValueError):
            M.moe_chosen(*bad, 4, 2, 64, 0)
    assert not M.chosen_ok(h.requires_grad_(), wts, gu, down, 4, 2, 64, 0)


def test_replays():
    T, W, E, top, ff, ffs = 150, 256, 8, 2, 128, 128
    h, wts, gu, down = layer(T, W, E, top, ff, ffs, True, torch.bfloat16, 5)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        M.moe_chosen(h, wts, gu, down, E, top, ff, ffs)
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = M.moe(h, wts, gu, down, E, top, ff, ffs)
    for i in range(4):
        h2, w2, _, _ = layer(T, W, E, top, ff, ffs, True, torch.bfloat16, 50 + i, 0.4 * i)
        h.copy_(h2)
        wts.copy_(w2)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, M.moe_chosen(h2, w2, gu, down, E, top, ff, ffs))


@pytest.mark.parametrize("T,W,E,top,ff,ffs,act,down", [(256, 4096, 8, 2, 2816, 0, 4, 2), (256, 2048, 4, 1, 5632, 0, 4, 8), (4096, 2048, 8, 2, 1408, 1408, 8, 8),
                                                       (64, 2048, 8, 2, 1408, 1408, 2, 2), (512, 4096, 8, 2, 2816, 0, 8, 4)])
def test_tiles_by_the_rounds_to_be_expected(T, W, E, top, ff, ffs, act, down):
    """64 rows an expert by the mean are more than one tile of 64 for half of them, and a round that was not counted."""
    h, wts, gu, w2 = layer(T, W, E, top, ff, ffs, True, torch.bfloat16, 3)
    args = (E, top, ff, ffs, "silu", True, "output")
    names = [n for n, _, _ in launches(lambda: M.moe_chosen(h, wts, gu, w2, *args)) if "expert_kernel<" in n]
    got = [n.split("expert_kernel<")[1].split(">")[0].split(", ")[1:3] for n in names]
    assert got == [["0", str(act)], ["2", str(down)]]
