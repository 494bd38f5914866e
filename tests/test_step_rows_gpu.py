"""Row kernels that hold a row in registers -- norms of the stream, of groups and of heads, and the routing of up to 64
experts by counting -- at the edges of the widths and row counts that they take, against float64."""
import pytest
import torch

from launches import launches
from lumen.ops import attention as A
from lumen.ops import moe, norm

pytestmark = pytest.mark.gpu
HALF = {torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12, torch.float32: 2.0 ** -24}
BF16 = torch.bfloat16


def gen(seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return lambda *s: torch.randn(*s, device="cuda", generator=g)


def near(got, want, sums=4e-6):
    """One rounding of the stored type, beside fp32 sums and products (relative to the row's largest value)."""
    want = want.double()
    err = (got.double() - want).abs()
    assert (err <= 2.01 * HALF[got.dtype] * want.abs() + sums * want.abs().amax(-1, keepdim=True)).all(), err.max()


@pytest.mark.parametrize("dt", [BF16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,W", [(1, 4), (3, 1020), (2, 1024), (5, 1028), (1, 2048), (9, 2052), (2, 4096), (3, 4100), (2, 1023)])
def test_stream(T, W, dt):
    r = gen(W)
    x, y, w, table = r(T, W), r(T, W).to(dt), r(W), r(7, W).to(dt)
    want = x.double() + y.double()
    rms = lambda v: v / torch.sqrt((v * v).mean(-1, keepdim=True) + 1e-6) * w.double()  # noqa: E731
    h = norm.residual_rms(x, y, w, 1e-6)
    near(x, want)
    near(h, rms(want))
    tokens = torch.arange(T, device="cuda") % 7
    x, h, e = norm.embed_rms(tokens, table, 1.5, w, 1e-6, rows=True)
    near(h, rms(table[tokens].double() * 1.5))
    assert torch.equal(e, table[tokens])
    parts, base = r(2 * T, W), r(T, W)
    x, h = norm.parts_rms(parts, base, 0.25, w, 1e-6, dt)
    near(h, rms(parts[:T].double() + parts[T:].double() + 0.25 * base.double()), 2e-5)      # (three terms may cancel)


@pytest.mark.parametrize("off", [4, 8])
@pytest.mark.parametrize("dt", [BF16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,W,groups", [(1, 256, 1), (2, 2048, 1), (1, 2052, 1), (3, 4096, 1), (2, 4100, 1), (2, 1032, 2), (4, 1536, 3),
                                        (1, 4096, 4), (2, 4112, 4), (3, 640, 5), (2, 4096, 32), (2, 66, 3), (1030, 512, 1)])
def test_groups(T, W, groups, dt, off):
    """Columns of a wider projection: from the eighth on in registers (16 bytes), from the fourth by passes in 16 bits."""
    r = gen(W + groups)
    z, w, x = r(T, W + 16).to(dt)[:, off:off + W], r(W), r(T, W)
    ref = norm.group_rms_norm_ref(z.double(), w, groups, 1e-6, torch.float64)
    ref64 = (z.double().reshape(T, groups, -1) / torch.sqrt((z.double().reshape(T, groups, -1) ** 2).mean(-1, keepdim=True) + 1e-6)
             ).reshape(T, W) * w.double()
    near(ref.float(), ref64, 1e-6)
    near(norm.group_rms_norm(z, w, groups, 1e-6), ref64)
    (name, _, _), = launches(lambda: norm.group_rms_norm(z, w, groups, 1e-6))
    waves = 1 if groups >= 3 else 4 // groups
    parts = -(-W // groups // (256 * waves))
    held = off * z.element_size() % 16 == 0 and W // groups % 4 == 0 and (W + 16) % 4 == 0 and parts <= 4
    assert (f", {1 if parts <= 1 else 2 if parts <= 2 else 4}>" in name and "group_rms_held<" in name) if held else "group_rms_kernel<" in name
    want = x.double() + ref64
    x, xb = norm.group_rms_residual(x, z, w, groups, 1e-6, dt)
    near(x, want)
    if xb is not None:
        near(xb, want)
    o = r(T, W)
    for gate, first in (("silu", True), ("sigmoid", False)):
        a = torch.sigmoid(z.double()) * (z.double() if gate == "silu" else 1)
        p = (o.double() * a if first else o.double()).reshape(T, groups, -1)
        p = (p / torch.sqrt((p * p).mean(-1, keepdim=True) + 1e-6)).reshape(T, W) * w.double()
        near(norm.gated_rms_norm(o, z, w, groups, 1e-6, gate, first), p if first else p * a)


@pytest.mark.parametrize("dt", [BF16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,H,G,D,dims,off", [(1, 16, 4, 128, 128, 0), (5, 16, 16, 128, 128, 0), (3, 30, 2, 128, 0, 0), (2, 31, 2, 128, 0, 0),
                                              (4, 62, 2, 64, 16, 0), (2, 64, 2, 128, 128, 0), (3, 2, 1, 64, 64, 2), (1, 1, 1, 8, 0, 0),
                                              (1025, 4, 2, 64, 64, 0), (2, 8, 8, 512, 64, 0), (3, 5, 1, 24, 8, 0)])
def test_heads(T, H, G, D, dims, off, dt):
    """16-bit rows of up to 256 and 512 items of eight, and past both; head_norm_write with 8 to 64 lanes a head."""
    r = gen(H * D + dims)
    n = (H + 2 * G) * D
    z = r(T, n + 8).to(dt)[:, off:off + n]
    if off:
        z = r(T * n + off).to(dt)[off:].view(T, n)
    f = 1.0 / 100 ** torch.linspace(0, 1, max(1, dims // 2), device="cuda")
    pos = torch.arange(T, device="cuda", dtype=torch.int32) % 90
    slots = torch.randperm(T + 9, generator=torch.Generator().manual_seed(T))[:T].cuda()
    if T > 2:
        slots[1] = -1
    cache = lambda t: [torch.zeros(T + 9, 1, G, D, device="cuda", dtype=t) for _ in range(2)]  # noqa: E731
    for kind in ("row", "turned", "plain"):
        wq, wk = r(H * D if kind == "row" else D), r(G * D if kind == "row" else D)
        got, want, c1, c2 = z.clone(), z.double(), cache(dt), cache(torch.float64)
        if kind == "plain":
            A.head_norm_write(got, wq, wk, slots, *c1, H, G, D, D, 1e-6)
            q, k, v = (want[:, a * D:b * D].reshape(T, -1, D) for a, b in ((0, H), (H, H + G), (H + G, H + 2 * G)))
            unit = lambda x: x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6)  # noqa: E731
            q, k = unit(q) * wq.double(), unit(k) * wk.double()
        else:
            if kind == "row":
                A.row_norm_rotary_write(got, wq, wk, pos, slots, *c1, H, G, D, D, dims, f, 1.0, 1e-6)
            else:
                A.head_norm_rotary_write(got, wq, wk, pos, slots, *c1, H, G, D, D, dims, f, 1e-6)
            parts = [want[:, :H * D], want[:, H * D:(H + G) * D]]
            shape = [(T, -1)] * 2 if kind == "row" else [(T, H, D), (T, G, D)]
            q, k = ((lambda x: x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6))(p.reshape(s)) * w.double()
                    for p, s, w in zip(parts, shape, (wq, wk)))
            a = (pos.float().view(T, 1, 1) * f.view(1, 1, -1)).double()           # (the angle is an fp32 product)

            def turn(x, n):
                x = x.reshape(T, n, D)
                if not dims:
                    return x
                u, v = x[..., :dims // 2], x[..., dims // 2:dims]
                return torch.cat([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin(), x[..., dims:]], -1)

            q, k = turn(q, H), turn(k, G)
            v = want[:, (H + G) * D:].reshape(T, G, D)
        near(got[:, :H * D], q.reshape(T, -1), 1e-5)
        assert torch.equal(got[:, H * D:], z[:, H * D:])
        ok = slots >= 0
        c2[0][slots[ok], 0], c2[1][slots[ok], 0] = k[ok], v[ok]
        near(c1[0].flatten(1), c2[0].flatten(1), 1e-5)
        assert torch.equal(c1[1].double(), c2[1])


@pytest.mark.parametrize("E,top", [(1, 1), (2, 2), (8, 2), (40, 2), (41, 2), (60, 3), (61, 3), (63, 63), (64, 4), (65, 4), (64, 3)])
def test_routes(E, top):
    """Counting up to 64 experts and 20 a choice, rounds of arg-max past that; equal logits, infinities and rows that are all -inf
    take the lowest index, NaN is never chosen."""
    r = gen(E)
    z = r(40, E)
    z[::3] = (2 * z[::3]).round() / 2                       # ties
    z[5] = 1.0
    near(moe.route_topk(z, top), moe.route_topk_ref(z, top), 1e-5)
    z[7, E // 2], z[8, 0] = float("nan"), -float("inf")
    got = moe.route_topk(z, top)
    assert got[7, E // 2] == 0 and got[8].isfinite().all() == (E > 1)
    live = z.clone()
    live[7, E // 2] = -1e30
    if top < E:                                             # (with every expert chosen the stand-in is chosen too, at weight 0)
        near(got[7], moe.route_topk_ref(live, top)[7], 1e-5)
    z = r(40, E)
    z[::3] = (2 * z[::3]).round() / 2
    corr = 0.1 * r(E)
    for groups in {1, 4 if E % 4 == 0 and top <= E // 2 else 1}:
        keep = max(1, groups // 2)
        for score, normalize in (("sigmoid", True), ("softmax", False)):
            got = moe.route_groups(z, None, top, groups, keep, 1.5, 1e-20, 1, score, normalize)
            near(got, moe.route_groups_ref(z, None, top, groups, keep, 1.5, 1e-20, 1, score, normalize), 1e-5)
            got = moe.route_groups(z, corr, top, groups, keep, 1.5, 1e-20, 1, score, normalize)
            near(got, moe.route_groups_ref(z, corr, top, groups, keep, 1.5, 1e-20, 1, score, normalize), 1e-5)


@pytest.mark.parametrize("T,W,S,groups", [(2, 1024, 1, 1), (3, 2048, 2, 1), (1, 2048, 4, 2), (5, 2304, 5, 1), (2, 4096, 8, 4), (64, 4352, 9, 1),
                                          (2, 8192, 3, 1), (3, 256, 13, 1), (2, 2048, 16, 8)])
def test_slabs(T, W, S, groups):
    from lumen.ops._seqmix import DT, call

    r = gen(W + S)
    y, w, x = r(S, T, W), r(W), r(T, W)
    out = torch.empty(T, W, device="cuda", dtype=BF16)
    g = y.double().sum(0).reshape(T, groups, -1)
    want = x.double() + (g / torch.sqrt((g * g).mean(-1, keepdim=True) + 1e-6)).reshape(T, W) * w.double()
    call("sm_slab_rms", DT[BF16], y, S, w, x, out, T, W, groups, 1e-6)
    near(x, want, 1e-5)
    near(out, want, 1e-5)
