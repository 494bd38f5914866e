"""Attention of decoded rows, heads of 128 (step_attention.hip) and latent rows (row_attention.hip), with every score shaping they
take, against the torch reference in fp32, at the edges of their groups of 16 keys and tiles of 64 and 128, in caches whose other
rows hold NaN."""
import pytest
import torch

from lumen.ops.attention import row_attention, row_attention_ref
from lumen.ops.segments import SegBatch

pytestmark = pytest.mark.gpu
CTX = (1, 15, 16, 17, 63, 64, 65, 127, 129, 300, 700)


def step(ctx, bs, g, device="cpu"):
    need = [-(-c // bs) for c in ctx]
    free = torch.randperm(sum(need) + 2, generator=g).tolist()
    tables = torch.zeros(len(ctx), max(need) + 3, dtype=torch.int32)
    for t, n in enumerate(need):
        tables[t, :n] = torch.tensor([free.pop() for _ in range(n)], dtype=torch.int32)
    i32 = dict(dtype=torch.int32)
    seq, pos = torch.arange(len(ctx), **i32), torch.tensor(ctx, **i32) - 1
    return SegBatch(torch.arange(len(ctx) + 1, **i32), seq, pos, seq, pos, tables, None), sum(need) + 2


def on_gpu(seg):
    c = lambda x: None if x is None else x.cuda()  # noqa: E731
    return SegBatch(c(seg.cu), c(seg.slot), c(seg.start), c(seg.row_seg), c(seg.positions), c(seg.tables), None)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind", ["plain", "cap_window", "bias_sink_gate", "slopes_keep", "talk", "talk_window"])
@pytest.mark.parametrize("T,H,G,bs", [(11, 16, 4, 16), (1, 8, 2, 16), (11, 12, 6, 32), (11, 16, 2, 8), (3, 32, 8, 16), (300, 4, 2, 16)])
def test_shapings(T, H, G, bs, kind, dt):
    g = torch.Generator().manual_seed(H + T)
    ctx = [CTX[(t + (5 if T == 1 else 0)) % len(CTX)] if T < 100 else 1 + t % 70 for t in range(T)]
    seg, nb = step(ctx, bs, g)
    k, v = (torch.full((nb * bs, G, 128), float("nan")).to(dt) for _ in range(2))
    for t, n in enumerate(ctx):
        rows = seg.tables[t].long()[torch.arange(n) // bs] * bs + torch.arange(n) % bs
        k[rows], v[rows] = (torch.randn(n, G, 128, generator=g).to(dt) for _ in range(2))
    k, v = k.view(nb, bs, G, 128), v.view(nb, bs, G, 128)
    q = torch.randn(T, H * 128 + 24, generator=g).to(dt)[:, :H * 128]            # rows of a wider projection
    rnd = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    kw = {"plain": {}, "cap_window": dict(softcap=3.0, window=100),
          "bias_sink_gate": dict(r1=rnd(H).abs(), r2=rnd(H).abs(), sink=rnd(H), gate=rnd(T, H).to(dt), q_temp=(0.4, 32)),
          "slopes_keep": dict(slopes=0.02 * rnd(H).abs(), window=70, keep_first=5),
          "talk": dict(softcap=5.0, r1=rnd(H).abs(), r2=rnd(H).abs(), sink=rnd(H), q_temp=(0.4, 32), talk=torch.eye(H) + 0.2 * rnd(H, H)),
          "talk_window": dict(talk=torch.eye(H) + 0.2 * rnd(H, H), window=90, keep_first=3)}[kind]
    want = row_attention_ref(q.view(T, H, 128), None, k, v, 128, torch.empty(T, H, 128), seg, H, G, 0.088, **kw)
    out = torch.empty(T, H, 128, dtype=dt, device="cuda")
    kw = {n: x.cuda() if torch.is_tensor(x) else x for n, x in kw.items()}
    row_attention(q.cuda().view(T, H, 128), None, k.cuda(), v.cuda(), 128, out, on_gpu(seg), H, G, 0.088, **kw)
    # one rounding of the result; scores of size <= 32, mixed by rows of 1-norm <= 8, to a few units of fp32's last place in weights
    # and sums over values of size <= 5 (a score's error of 8 x 32 x 2^-23 x 16 is one of 2^-11 in its weight at the most)
    tol = want.abs() * torch.finfo(dt).eps / 2 + 5.0 * (2.0 ** -11 if "talk" in kind else 2.0 ** -14)
    assert ((out.float().cpu() - want).abs() <= tol).all()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind", ["plain", "window", "talk", "talk_window"])
@pytest.mark.parametrize("H,G", [(4, 2), (16, 4), (8, 1)])
def test_an_infinity_of_the_rows_own_value(H, G, kind, dt):
    """It is the row's result in that channel, as the keys that the row does not see add nothing."""
    if "talk" in kind and H // G > 4:
        pytest.skip("mixed heads: up to four a key head")
    g = torch.Generator().manual_seed(H)
    seg, nb = step(CTX, 16, g)
    k, v = (torch.randn(nb * 16, G, 128, generator=g).to(dt) for _ in range(2))
    at = torch.tensor([c - 1 for c in CTX])
    own = seg.tables[torch.arange(len(CTX)), at // 16].long() * 16 + at % 16
    v[own, :, 5], v[own, :, 77] = float("inf"), -float("inf")
    k, v = k.view(nb, 16, G, 128), v.view(nb, 16, G, 128)
    q = torch.randn(len(CTX), H, 128, generator=g).to(dt)
    kw = dict(window=21, keep_first=3) if "window" in kind else {}
    if "talk" in kind:
        kw["talk"] = torch.eye(H)
    want = row_attention_ref(q, None, k, v, 128, torch.empty(len(CTX), H, 128), seg, H, G, 0.05, **kw)
    assert (want[:, :, 5] == float("inf")).all() and (want[:, :, 77] == -float("inf")).all()
    out = torch.empty(len(CTX), H, 128, dtype=dt, device="cuda")
    kw = {n: x.cuda() if torch.is_tensor(x) else x for n, x in kw.items()}
    row_attention(q.cuda(), None, k.cuda(), v.cuda(), 128, out, on_gpu(seg), H, G, 0.05, **kw)
    assert torch.equal(out.cpu().isinf(), want.isinf()) and torch.equal(out.cpu().sign()[want.isinf()], want.sign()[want.isinf()])
    assert out.cpu().nan_to_num(0, 0, 0).allclose(want.nan_to_num(0, 0, 0).to(dt), rtol=2 * torch.finfo(dt).eps, atol=1e-3)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shaped,gated", [(False, False), (True, False), (True, True)])
@pytest.mark.parametrize("T,H,R,D2,bs", [(3, 16, 512, 64, 16), (33, 16, 512, 64, 16), (17, 20, 512, 0, 8), (11, 5, 256, 32, 32),
                                         (40, 16, 256, 64, 16), (11, 16, 384, 32, 16), (40, 3, 384, 0, 16), (40, 16, 512, 40, 16),
                                         (11, 16, 512, 72, 16), (40, 3, 512, 128, 8), (11, 20, 384, 104, 16), (33, 16, 256, 72, 16),
                                         (600, 16, 256, 96, 16), (11, 16, 192, 64, 16)])
def test_latent_rows(T, H, R, D2, bs, shaped, gated, dt):
    """Tiles of 64 keys (up to 32 rows x 16 heads) and of 128; with and without the expansion of the merged sums."""
    g = torch.Generator().manual_seed(T + R)
    ctx = [CTX[t % len(CTX)] for t in range(T)]
    seg, nb = step(ctx, bs, g)
    D = R + D2
    c = torch.full((nb * bs, D), float("nan")).to(dt)
    for t, n in enumerate(ctx):
        c[seg.tables[t].long()[torch.arange(n) // bs] * bs + torch.arange(n) % bs] = torch.randn(n, D, generator=g).to(dt)
    c = c.view(nb, bs, D)
    q = torch.randn(T, H, D, generator=g).to(dt)
    uv = (torch.randn(H, 64, R, generator=g) / R ** 0.5).to(dt)
    rnd = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    kw = dict(softcap=4.0, r1=rnd(H).abs(), r2=rnd(H).abs(), sink=rnd(H), q_temp=(0.4, 32)) if shaped else {}
    kw["gate"] = rnd(T, H).to(dt) if gated else None
    q1, q2 = q[:, :, :R], q[:, :, R:] if D2 else None
    want = row_attention_ref(q1, q2, c, c, R, torch.empty(T, H, R), seg, H, 1, 0.04, **kw)
    kw = {n: x.cuda() if torch.is_tensor(x) else x for n, x in kw.items()}
    qd, cd = q.cuda(), c.cuda()
    args = (qd[:, :, :R], qd[:, :, R:] if D2 else None, cd, cd, R)
    kw["vt"] = c[:, :, :R].transpose(1, 2).contiguous().cuda()
    out = torch.empty(T, H, R, dtype=dt, device="cuda")
    row_attention(*args, out, on_gpu(seg), H, 1, 0.04, **kw)
    # as above, weights in two 16-bit parts: 16 bits of them for bf16
    tol = want.abs() * torch.finfo(dt).eps / 2 + 5.0 * 2.0 ** -13
    assert ((out.float().cpu() - want).abs() <= tol).all()
    o = torch.empty(T, H, 64, dtype=dt, device="cuda")
    got = row_attention(*args, out.clone(), on_gpu(seg), H, 1, 0.04, expand=(uv.cuda(), o), **kw)
    if got is o:                                           # the expansion of the rounded rows, rounded once more
        w2 = torch.einsum("thr,hvr->thv", out.float().cpu(), uv.float())
        mag = torch.einsum("thr,hvr->thv", out.float().cpu().abs(), uv.float().abs())
        tol = w2.abs() * torch.finfo(dt).eps / 2 + mag * (2.0 ** -20 + torch.finfo(dt).eps / 8)
        assert ((o.float().cpu() - w2).abs() <= tol).all()
    assert (got is o) == (R in (256, 512) and T * H <= 4096)
