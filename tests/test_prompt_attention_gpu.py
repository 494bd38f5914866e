"""Attention of prompt portions in tiles of 128 rows and 64 keys (seqmix/window_attention.hip, seqmix/attention.hip)
where the tiles' edges, the block table and the moving reference of the weights can go wrong: portions around 32, 64
and 128 rows, cached context, blocks that are not a power of two, more blocks than the kernels hold in LDS, scores
that creep upwards, and unowned cache rows full of NaN."""
import pytest
import torch

from launches import launches
from lumen.ops.attention import chunk_sink_attention, chunk_sink_attention_ref, row_attention, row_attention_ref
from lumen.ops.segments import SegBatch, tile_list

pytestmark = pytest.mark.gpu
DTYPES = [(torch.bfloat16, 2.0 ** -8), (torch.float16, 2.0 ** -11)]


def portions(lens, starts, bs, g, *shapes):
    """Portions of whole tiles and their caches, one per (heads, size): scrambled blocks, NaN where no key is."""
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    total = [s + n for s, n in zip(starts, lens)]
    nb = [(t + bs - 1) // bs for t in total]
    order = torch.randperm(sum(nb) + 3, generator=g).tolist()
    tables = torch.zeros(len(lens), max(nb), dtype=torch.int32)
    caches = [torch.full((sum(nb) + 3, bs, *s), float("nan")) for s in shapes]
    for i, n in enumerate(nb):
        for b in range(n):
            tables[i, b] = order.pop()
            for c in caches:
                rows = min(bs, total[i] - b * bs)
                c[tables[i, b], :rows] = torch.randn(rows, *c.shape[2:], generator=g)
    i32 = dict(dtype=torch.int32, device="cuda")
    seg = SegBatch(torch.tensor(cu, **i32), torch.arange(len(lens), **i32), torch.tensor(starts, **i32),
                   torch.cat([torch.full((n,), i) for i, n in enumerate(lens)]).int().cuda(),
                   torch.cat([torch.arange(n) + s for s, n in zip(starts, lens)]).int().cuda(),
                   tables.cuda(), None, torch.tensor(tile_list(cu, len(lens)), **i32).view(-1, 2), cu[-1], 128)
    return cu[-1], seg, caches


def close(out, ref, ulp):
    # the output's rounding (half an ulp), the weights' ~16 bits and the products' fp32 sums, relative to the
    # largest entry: under two ulps of it
    assert torch.isfinite(out).all()
    err = (out.float() - ref.float()).abs().max() / ref.float().abs().max()
    assert err < 2 * ulp, err


@pytest.mark.parametrize("dtype,ulp", DTYPES)
@pytest.mark.parametrize("lens,starts,bs,window,keep", [
    ([31, 32, 33, 63, 64, 65, 1], [0, 0, 1, 0, 70, 3, 5], 16, 0, 0),
    ([127, 128, 129], [0, 64, 1], 12, 70, 5), ([130, 66], [200, 61], 16, 64, 130), ([40, 5], [560, 0], 1, 0, 0),
    ([33], [700], 1, 620, 7)])
@pytest.mark.parametrize("H,G,D,Dv", [(4, 2, 128, 128), (2, 2, 32, 64), (2, 1, 128, 256), (258, 2, 32, 32), (258, 6, 64, 128),
                                      (258, 2, 128, 128)])
def test_window_tiles(H, G, D, Dv, lens, starts, bs, window, keep, dtype, ulp):
    g = torch.Generator().manual_seed(D + bs + len(lens))
    T, seg, (k, v) = portions(lens, starts, bs, g, (G, D), (G, Dv))
    k, v = k.to(dtype).cuda(), v.to(dtype).cuda()
    q = torch.randn(T, H, D, generator=g).to(dtype).cuda()
    for cap, slopes in ((0.0, None), (3.0, torch.rand(H, generator=g).cuda() * 0.1)):
        out, ref = (torch.zeros(T, H, Dv, dtype=dt, device="cuda") for dt in (dtype, torch.float32))
        row_attention(q, None, k, v, Dv, out, seg, H, G, D ** -0.5, cap, slopes=slopes, window=window, keep_first=keep)
        row_attention_ref(q.float(), None, k.float(), v.float(), Dv, ref, seg, H, G, D ** -0.5, cap, slopes=slopes,
                          window=window, keep_first=keep)
        close(out, ref, ulp)


@pytest.mark.parametrize("dtype,ulp", DTYPES)
@pytest.mark.parametrize("lens,starts,bs,chunk", [
    ([31, 32, 33, 63, 64, 65, 1], [0, 0, 1, 0, 70, 3, 5], 16, 0), ([127, 128, 129], [0, 64, 1], 12, 75),
    ([40, 5], [560, 0], 1, 0)])
@pytest.mark.parametrize("H,G,D", [(4, 2, 128), (2, 1, 96), (2, 2, 256), (258, 2, 32)])
def test_chunk_tiles(H, G, D, lens, starts, bs, chunk, dtype, ulp):
    g = torch.Generator().manual_seed(D + bs + len(lens))
    T, seg, (k,) = portions(lens, starts, bs, g, (G, D))
    k = k.to(dtype).cuda()
    q = torch.randn(T, H * D, generator=g).to(dtype).cuda()
    out = chunk_sink_attention(q, k, seg, H, G, D, 0.3, chunk, 1e-6)
    close(out, chunk_sink_attention_ref(q.float(), k.float(), seg, H, G, D, 0.3, chunk, 1e-6), ulp)


@pytest.mark.parametrize("dtype,ulp", DTYPES)
@pytest.mark.parametrize("lens,starts,bs,chunk", [
    ([31, 32, 33, 63, 64, 65, 1], [0, 0, 1, 0, 70, 3, 5], 16, 0), ([127, 128, 129], [0, 64, 1], 12, 75)])
@pytest.mark.parametrize("H,G,D", [(258, 2, 128), (258, 3, 96)])
def test_chunk_tiles_of_many_workgroups(H, G, D, lens, starts, bs, chunk, dtype, ulp):
    """Whole tiles of keys a wave; the reference forms each key head's first and last query head."""
    g = torch.Generator().manual_seed(D + bs + len(lens))
    T, seg, (k,) = portions(lens, starts, bs, g, (G, D))
    k = k.to(dtype).cuda()
    q = torch.randn(T, H * D, generator=g).to(dtype).cuda()
    out = chunk_sink_attention(q, k, seg, H, G, D, 0.3, chunk, 1e-6).view(T, G, H // G, D)[:, :, [0, -1]].reshape(T, -1)
    some = q.view(T, G, H // G, D)[:, :, [0, -1]].reshape(T, -1)
    close(out, chunk_sink_attention_ref(some.float(), k.float(), seg, 2 * G, G, D, 0.3, chunk, 1e-6), ulp)


@pytest.mark.parametrize("dtype,ulp", DTYPES)
@pytest.mark.parametrize("rise", [0.01, 0.07, 0.5, -0.5])
def test_scores_that_creep(rise, dtype, ulp):
    """The score grows by ``rise`` per key: under and over what moves the reference within a tile."""
    T, H, G, D = 300, 1, 1, 64
    g = torch.Generator().manual_seed(7)
    _, seg, (k, v) = portions([T], [0], 16, g, (G, D), (G, D))
    k[:, :, :, 0] = 0.0
    for j in range(T):
        k[seg.tables[0, j // 16].item(), j % 16, 0, 0] = rise * j
    k, v = k.to(dtype).cuda(), v.to(dtype).cuda()
    q = torch.zeros(T, H, D)
    q[:, :, 0] = 1.0
    q = q.to(dtype).cuda()
    out, ref = (torch.zeros(T, H, D, dtype=dt, device="cuda") for dt in (dtype, torch.float32))
    row_attention(q, None, k, v, D, out, seg, H, G, 1.0)
    row_attention_ref(q.float(), None, k.float(), v.float(), D, ref, seg, H, G, 1.0)
    close(out, ref, ulp)


@pytest.mark.parametrize("dtype,ulp", DTYPES)
@pytest.mark.parametrize("lens,extra", [([31, 32, 33, 1, 65], 0), ([127, 128, 129, 260], 3)])
@pytest.mark.parametrize("H,tile", [(1, 128), (5, 128), (2, 64), (130, 128)])
def test_fresh_latent_rows(H, tile, lens, extra, dtype, ulp):
    """Prompts over their own rows against the reference, rows of wider buffers, decoded rows behind them."""
    from lumen.ops.attention import fresh_latent_attention, fresh_latent_attention_ref, fresh_latent_ok

    D, Dr, Dv = 128, 64, 128
    g = torch.Generator().manual_seed(H + len(lens))
    n, seg, _ = portions(lens + [1] * extra, [0] * len(lens) + [9] * extra, 16, g)
    n -= extra
    seg.q_tiles = torch.tensor(tile_list(seg.cu.tolist(), len(lens), tile), dtype=torch.int32, device="cuda").view(-1, 2)
    seg.tile_rows, seg.tile_size, seg.fresh = n, tile, True
    assert fresh_latent_ok(dtype, seg, D, Dr, Dv) and not fresh_latent_ok(dtype, seg, 64, Dr, Dv)
    f = lambda *s: torch.randn(*s, generator=g).to(dtype).cuda()  # noqa: E731
    q, kv, c = f(n + extra, H * (D + Dr) + 8), f(n, H * (D + Dv)), f(n, 24 + Dr)
    args = (q[:n, :H * (D + Dr)].view(n, H, D + Dr), kv[:, :H * D].view(n, H, D), c[:, 24:],
            kv[:, H * D:].view(n, H, Dv))
    out, ref = (torch.zeros(n, H, Dv, dtype=dt, device="cuda") for dt in (dtype, torch.float32))
    fresh_latent_attention(*args, out, seg, 0.07)
    fresh_latent_attention_ref(*args, ref, seg, 0.07)
    close(out, ref, ulp)
    seg.fresh = False
    with pytest.raises(ValueError):
        fresh_latent_attention(*args, out, seg, 0.07)


@pytest.mark.parametrize("dtype,ulp", DTYPES)
@pytest.mark.parametrize("lens,starts,bs,tile", [
    ([15, 16, 17, 1, 33], [0, 0, 3, 31, 64], 16, 128), ([130, 64], [0, 35], 12, 64), ([20, 3], [560, 0], 1, 128)])
@pytest.mark.parametrize("H,G,opts", [(1, 1, ()), (8, 2, ("cap", "r", "sink", "temp")), (12, 3, ("sink",)), (16, 4, ("r",)),
                                      (16, 8, ("cap",)), (24, 6, ("cap", "r", "sink", "temp")), (32, 8, ("temp", "r"))])
def test_mixed_head_tiles(H, G, opts, lens, starts, bs, tile, dtype, ulp):
    D = 128
    g = torch.Generator().manual_seed(H + bs)
    T, seg, (k, v) = portions(lens + [1], starts + [40], bs, g, (G, D), (G, D))
    seg.tile_rows, seg.tile_size = T - 1, tile             # (the last row is a decoded one)
    seg.keys = (T, 1)                                      # (the tiles' edges, also where they are not the faster kernel)
    seg.q_tiles = torch.tensor(tile_list(seg.cu.tolist(), len(lens), tile), dtype=torch.int32, device="cuda").view(-1, 2)
    k, v = k.to(dtype).cuda(), v.to(dtype).cuda()
    q = torch.randn(T, H * D + 8, generator=g).to(dtype).cuda()[:, :H * D].view(T, H, D)
    f = lambda *s: torch.rand(*s, generator=g).cuda()  # noqa: E731
    kw = dict(talk=torch.eye(H).cuda() + 0.3 * (f(H, H) - 0.5), softcap=4.0 if "cap" in opts else 0.0,
              q_temp=(0.3, 16) if "temp" in opts else None, r1=f(H) if "r" in opts else None,
              r2=f(H) if "r" in opts else None, sink=2 * f(H) - 1 if "sink" in opts else None)
    import lumen.ops._seqmix as sm
    calls, real = [], sm.call
    sm.call = lambda n, *a: (calls.append(n), real(n, *a))[1]
    try:
        out = torch.full((T, H, D), float("nan"), dtype=dtype, device="cuda")
        row_attention(q, None, k, v, D, out, seg, H, G, 0.1, **kw)
    finally:
        sm.call = real
    assert calls == ["sm_talk_tiles", "sm_row_attn"]
    ref = torch.zeros(T, H, D, device="cuda")
    row_attention_ref(q.float(), None, k.float(), v.float(), D, ref, seg, H, G, 0.1, **kw)
    close(out, ref, ulp)


@pytest.mark.parametrize("dtype,share", [(torch.bfloat16, 0.001), (torch.float16, 0.005)])
@pytest.mark.parametrize("H,G", [(8, 2), (16, 4), (32, 8)])
def test_mixed_head_tiles_hold_fp32_weights(H, G, dtype, share):
    """Scores, weights and sums in fp32: hardly a result but float64's rounded.  A relative error e of a result before
    it is rounded misses that for a share of ~ 2 e / (the type's half ulp): fp32's (a few 2^-24, over sums of 63 keys) 0.03
    and 0.2 %; weights of ~16 bits leave 0.25 and 1.2 %.  (Sizes whose shares were seen to be that.)"""
    T, D = 63, 128
    g = torch.Generator().manual_seed(H)
    _, seg, (k, v) = portions([T], [0], 16, g, (G, D), (G, D))
    k, v = k.to(dtype).cuda(), v.to(dtype).cuda()
    q, f = torch.randn(T, H, D, generator=g).to(dtype).cuda(), lambda *s: torch.rand(*s, generator=g).cuda()
    talk, r1, r2, sink = torch.eye(H).cuda() + 0.3 * (f(H, H) - 0.5), f(H), f(H), f(H)
    out = torch.empty(T, H, D, dtype=dtype, device="cuda")
    row_attention(q, None, k, v, D, out, seg, H, G, 0.088, 50.0, (0.3, 16), r1, r2, talk, sink)
    at = torch.arange(T, device="cuda")
    K, V = (x[seg.tables[0].long()[at // 16], at % 16].double().repeat_interleave(H // G, 1) for x in (k, v))
    s = torch.einsum("thd,jhd->htj", q.double(), K) * 0.088 * (1 + 0.3 * torch.log((at + 1) // 16 + 1.0).double())[:, None]
    s = 50 * torch.tanh(s / 50) - r1.double()[:, None, None] * torch.log(
        1 + r2.double()[:, None, None] * (at[:, None] - at).clamp(min=0))
    s = torch.einsum("ij,jtk->itk", talk.double(), s).masked_fill(at[:, None] < at, -float("inf"))
    e = torch.exp(s)
    ref = torch.einsum("htj,jhd->thd", e / (e.sum(-1, keepdim=True) + torch.exp(sink.double())[:, None, None]), V)
    assert (out != ref.to(dtype)).double().mean() < share


@pytest.mark.parametrize("kind,rows,H,halves", [("window", 128, 256, True), ("window", 129, 128, True), ("window", 128, 258, False), ("window", 129, 130, False),
                                                ("chunk", 128, 256, True), ("chunk", 129, 130, False), ("fresh", 128, 128, True), ("fresh", 65, 8, True),
                                                ("fresh", 64, 8, False), ("fresh", 128, 129, False)])
def test_few_workgroups_take_halves_of_the_keys(kind, rows, H, halves):
    """Two workgroups a tile of 128 rows, each with 64 of them, up to 256 (fresh: 128) tiles x heads: the tests above hold both forms."""
    from lumen.ops.attention import fresh_latent_attention

    g = torch.Generator().manual_seed(1)
    T, seg, (k, v) = portions([rows], [0], 16, g, (2, 128), (2, 128))
    seg.fresh = True
    k, v, out = k.bfloat16().cuda(), v.bfloat16().cuda(), torch.empty(T, H, 128, dtype=torch.bfloat16, device="cuda")
    f = lambda *s: torch.randn(*s, generator=g).bfloat16().cuda()  # noqa: E731
    if kind == "fresh":
        args = (f(T, H, 192), f(T, H, 128), f(T, 64), f(T, H, 128), out, seg, 0.07)
        (_, grid, _), = launches(lambda: fresh_latent_attention(*args))
    elif kind == "chunk":
        q = f(T, H * 128)
        (_, grid, _), = launches(lambda: chunk_sink_attention(q, k, seg, H, 2, 128, 0.3, 0, 1e-6))
    else:
        q = f(T, H, 128)
        (_, grid, _), = launches(lambda: row_attention(q, None, k, v, 128, out, seg, H, 2, 0.1))
    assert grid[0] == (2 if halves else 1) * -(-rows // 128) * H


ODD = {5: (0, float("inf")), 37: (9, float("-inf")), 100: (21, float("nan"))}     # position: channel, value


def odd_rows(run, v, seg, window=0):
    """``run`` before and after values of some tokens became infinite or NaN: the rows that see such a token are lost in
    its channel, the others keep what they had (formed again there), and other channels their bits."""
    before = run().clone()
    assert torch.isfinite(before).all()
    lost = torch.zeros_like(before, dtype=torch.bool)
    for j, (ch, x) in ODD.items():
        v(j)[..., ch] = x
        p = seg.positions[:before.shape[0]]
        lost[(p >= j) & ((window == 0) | (p - j < window)), :, ch] = True
    after, other = run(), ~lost.any(1).any(0)
    assert torch.equal(after[:, :, other], before[:, :, other]) and not torch.isfinite(after[lost]).any()
    close(after[~lost], before[~lost], 2.0 ** -8 if before.dtype == torch.bfloat16 else 2.0 ** -11)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind,H,G,D,Dv,window", [
    ("window", 4, 2, 128, 128, 0), ("window", 2, 2, 64, 128, 20), ("window", 2, 1, 128, 256, 0), ("talk", 8, 2, 128, 128, 0),
    ("talk", 16, 4, 128, 128, 0), ("talk", 24, 6, 128, 128, 0), ("fresh", 3, 3, 128, 128, 0), ("window", 130, 2, 128, 128, 0),
    ("window", 130, 2, 64, 128, 20), ("fresh", 66, 66, 128, 128, 0)])
def test_infinite_values_of_hidden_tokens(kind, H, G, D, Dv, window, dtype):
    g = torch.Generator().manual_seed(H)
    T, seg, (k, v) = portions([131], [0], 16, g, (G, D), (G, Dv))
    seg.keys = (T, 1)                                      # (mixed heads: the tiles)
    f = lambda *s: torch.randn(*s, generator=g).to(dtype).cuda()  # noqa: E731
    k, v, out = k.to(dtype).cuda(), v.to(dtype).cuda(), torch.zeros(T, H, Dv, dtype=dtype, device="cuda")
    if kind == "fresh":
        from lumen.ops.attention import fresh_latent_attention
        seg.fresh = True
        q, k, kr, v = f(T, H, D + 64), f(T, H, D), f(T, 64), f(T, H, Dv)
        return odd_rows(lambda: fresh_latent_attention(q, k, kr, v, out, seg, 0.07), lambda j: v[j], seg)
    q, talk = f(T, H, D), torch.eye(H).cuda() + 0.1 if kind == "talk" else None
    odd_rows(lambda: row_attention(q, None, k, v, Dv, out, seg, H, G, 0.1, talk=talk, window=window),
             lambda j: v[seg.tables[0, j // 16].item(), j % 16], seg, window)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,G,D,chunk", [(4, 2, 128, 0), (2, 1, 96, 50), (2, 2, 256, 0), (2, 2, 64, 128), (130, 2, 128, 0), (130, 1, 96, 50),
                                           (130, 2, 64, 128)])
def test_infinite_keys_of_hidden_tokens(H, G, D, chunk, dtype):
    """Keys that are their own values: whole rows that see such a token are lost, the others keep what they had."""
    g = torch.Generator().manual_seed(H)
    T, seg, (k,) = portions([131], [0], 16, g, (G, D))
    k, q = k.to(dtype).cuda(), torch.randn(T, H * D, generator=g).to(dtype).cuda()
    run = lambda: chunk_sink_attention(q, k, seg, H, G, D, 0.3, chunk, 1e-6).view(T, -1)  # noqa: E731
    before = run()
    lost = torch.zeros(T, dtype=torch.bool, device="cuda")
    for j, x in ((37, float("inf")), (70, float("nan"))):
        k[seg.tables[0, j // 16].item(), j % 16] = x
        p = seg.positions
        lost |= (p >= j) & ((chunk == 0) | (p // max(chunk, 1) == j // max(chunk, 1)))
    after = run()
    assert torch.isnan(after[lost]).all() and 0 < int(lost.sum()) < T
    close(after[~lost], before[~lost], 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_fresh_and_cached_prompts_agree(dtype):
    """One engine step of whole prompts (expanded keys) against the same prompts in two portions (the cached latent):
    logits of the same rows, with a decoded sequence beside them."""
    import lumen.serve.hybrid_runner as R
    from lumen.bench.hybrid_bench import dalavik_config
    from lumen.models import build_model
    from lumen.ops.segments import whole_sequences
    from lumen.serve.model_runner import StepInput

    cfg = dalavik_config(1024)
    cfg.vocab_size = 512
    torch.manual_seed(3)
    model = build_model(cfg, dtype=dtype, device=torch.device("cuda"), init="random")
    lens = [70, 1, 133]
    tok = torch.randint(3, 500, (sum(lens),), device="cuda")
    routes = []
    real, R.fresh_latent_attention = R.fresh_latent_attention, lambda *a: (routes.append(1), real(*a))[1]
    try:
        out = []
        for cut in (False, True):
            run = R.HybridRunner(R.WEIGHTS["dalavik"](model), 64, 16, torch.device("cuda"), 256, 4, use_graphs=False)
            whole = whole_sequences(lens, "cuda")
            pos, cu = whole.positions, [0, 70, 71, 204]
            parts = [[(0, 0, 40), (1, 0, 1), (2, 0, 90)], [(0, 40, 70), (2, 90, 133)]] if cut else \
                [[(i, 0, n) for i, n in enumerate(lens)]]
            x = None
            for part in parts:
                rows = torch.cat([torch.arange(cu[i] + a, cu[i] + b) for i, a, b in part]).cuda()
                c = [0]
                for _, a, b in part:
                    c.append(c[-1] + b - a)
                ids = torch.tensor([i for i, _, _ in part])
                i32 = dict(dtype=torch.int32, device="cuda")
                seg = SegBatch(torch.tensor(c, **i32), ids.int().cuda(), torch.tensor([a for _, a, _ in part], **i32),
                               torch.cat([torch.full((b - a,), k) for k, (_, a, b) in enumerate(part)]).int().cuda(),
                               pos[rows], whole.tables[ids.cuda()], whole.cache_slots[rows],
                               torch.tensor(tile_list(c, len(part)), **i32).view(-1, 2), c[-1], 128)
                inp = StepInput("mixed", tok[rows], pos[rows], seg.cache_slots, c, kv_lens=[b for _, _, b in part],
                                sample_rows=torch.tensor(c[1:], device="cuda") - 1, seg=seg)
                x = run.execute(inp)
            out.append(x[[0, -1]].float())
    finally:
        R.fresh_latent_attention = real
    assert len(routes) == 6                              # the whole prompts and the first portions, 3 layers
    err = (out[0] - out[1]).norm() / out[1].norm()
    assert err < (0.02 if dtype == torch.bfloat16 else 0.003), err       # 4 layers of 16-bit roundings
