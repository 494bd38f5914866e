"""Which calls the kernels of few rows and of decode steps take, and what happens to the ones they cannot."""
from contextlib import nullcontext

import pytest
import torch

from lumen.ops import _seqmix, gemm
from lumen.ops import moe as M


@pytest.fixture
def launched(monkeypatch):
    """The few-row kernels' launches, recorded instead of run (CPU tensors)."""
    calls = []
    monkeypatch.setattr(_seqmix, "use_seqmix", lambda t: True)
    monkeypatch.setattr(_seqmix, "call", lambda name, *a: calls.append((name, a)))
    return calls


BF = dict(dtype=torch.bfloat16)


def test_few_row_kernel_refuses_operands_it_would_misread(launched):
    x, w = torch.zeros(3, 128, **BF), torch.zeros(8, 128, **BF)
    wts = torch.zeros(3, 1)
    bad = [dict(w=torch.zeros(8, 64, **BF)), dict(w=torch.zeros(8, 256, **BF)[:, ::2]),
           dict(w=torch.zeros(8, 128, device="meta", **BF)), dict(w=w.half()), dict(x=torch.zeros(128, 3, **BF).t()),
           dict(bias=torch.zeros(4, **BF)), dict(bias=torch.zeros(16, **BF)[::2]),
           dict(bias=torch.zeros(8, device="meta", **BF)), dict(bias=torch.zeros(8)),
           dict(blocks=(wts[:2], 1, 64, 64)), dict(blocks=(wts.half(), 1, 64, 64)),
           dict(blocks=(wts.to("meta"), 1, 64, 64)), dict(blocks=(torch.zeros(3, 2), 1, 64, 64))]
    for kw in bad:
        with pytest.raises(ValueError):
            gemm.thin_linear(kw.pop("x", x), kw.pop("w", w), **kw)
    assert not launched
    gemm.thin_linear(x, w, torch.zeros(8, **BF), blocks=(wts, 1, 64, 64))
    assert [n for n, _ in launched] == ["sm_thin_gemm"]


def test_activation_form_refuses_operands_it_would_misread(launched):
    h, gu, wts = torch.zeros(3, 128, **BF), torch.zeros(2 * (2 * 64 + 64), 128, **BF), torch.zeros(3, 2)
    args = (2, 64, 64)
    for a in ((h, gu[:-1], wts), (h, gu[:, :64].contiguous(), wts), (h, gu.half(), wts), (h, gu, None),
              (h, gu, wts[:2]), (h, gu, torch.zeros(3, 4)[:, :2]), (h, gu, wts.half()),
              (h, gu.to("meta"), wts), (h, gu, wts.to("meta"))):
        with pytest.raises(ValueError):
            M.thin_act(*a, *args)
    assert not launched
    M.thin_act(h, gu, wts, *args)
    assert [n for n, _ in launched] == ["sm_thin_act"]


@pytest.mark.parametrize("down", [(96, 128), (96, 256), (94, 192)])
def test_second_projection_of_another_shape_is_not_read(launched, monkeypatch, down):
    """A [W, K] that does not fit the activation goes to the library, whose error it always was; one
    of a width the kernel does not have (94) is multiplied there."""
    monkeypatch.setattr(M, "thin_act_ok", lambda *a, **k: True)
    monkeypatch.setattr(M, "_thin_act", lambda h, gu, wts, E, ff, ffs, *a: torch.zeros(
        h.shape[0], E * ff + ffs, **BF))
    h, gu, wts = torch.zeros(3, 128, **BF), torch.zeros(384, 128, **BF), torch.zeros(3, 2)
    run = lambda: M.moe_dense(h, wts, gu, torch.zeros(*down, **BF), 2, 64, 64, top=1)  # noqa: E731
    if down[1] == 192:
        assert run().shape == (3, 94)
    else:
        with pytest.raises(RuntimeError):
            run()
    assert not launched


class OnGpu(torch.Tensor):
    """A CPU tensor that a dispatch takes for the GPU's."""
    is_cuda = True


@pytest.mark.parametrize("n,bucket,have,table_rows", [(3, 8, 8, 8), (3, 8, 5, 8), (3, 8, 16, 8), (3, 8, 8, 4),
                                                      (8, 4, 8, 8)])
def test_step_inputs_never_pass_the_buffers_end(launched, n, bucket, have, table_rows):
    """The one-launch form writes ``bucket`` entries: buffers of another length are filled by copies."""
    from lumen.serve.model_runner import fill_step

    i32 = dict(dtype=torch.int32)
    tok, slots = torch.arange(n).as_subclass(OnGpu), torch.arange(n)
    pos, tables = torch.arange(n, **i32), torch.ones(n, 2, **i32)
    td, sd, pd = torch.full((have,), 9), torch.full((have,), 9), torch.full((have,), 9, **i32)
    tab = torch.zeros(table_rows, 4, **i32)
    fill_step([(pos, pd, 0)], tok, td, slots, sd, tables, tab, n, bucket)
    if (n, bucket, have, table_rows) == (3, 8, 8, 8):
        assert [c for c, _ in launched] == ["sm_fill_step"]
        return
    assert not launched
    assert pd[:n].tolist() == list(range(n)) and tab[:n, :2].eq(1).all()
    if n < bucket:
        assert pd[n:].eq(0).all() and sd[n:].eq(-1).all() and td[n:].eq(9).all()


@pytest.mark.gpu
def test_operands_of_two_devices_stay_with_the_library():
    x, w = torch.zeros(3, 128, device="cuda", **BF), torch.zeros(8, 128, **BF)
    assert not gemm.thin_ok(x, w) and gemm.thin_ok(x, w.cuda())
    with pytest.raises(RuntimeError):
        gemm.project(x, w)
    with pytest.raises(RuntimeError):
        gemm.project(x, w.cuda(), torch.zeros(8, **BF))
    gu, wts = torch.zeros(384, 128, device="cuda", **BF), torch.zeros(3, 2, device="cuda")
    assert M.thin_act_ok(x, wts, gu, 2, 64, 64)
    for t in (wts.cpu(), wts[:2], torch.zeros(3, 3, device="cuda")):
        assert not M.thin_act_ok(x, t, gu, 2, 64, 64)


def test_a_plain_call_has_nothing_to_differentiate_batch_or_trace():
    """Of each kind of tensor, and inside each transform, the rule that sends products past autograd."""
    import torch.autograd.forward_ad as fwd
    from torch.utils.flop_counter import FlopCounterMode

    x, w, seen = torch.randn(3, 8), torch.randn(4, 8), []

    def probe(v):
        seen.append(gemm._plain(v, w))
        return v @ w.t()

    assert gemm._plain(x, w) and gemm._plain(torch.nn.Parameter(w, requires_grad=False), x)
    xr = x.clone().requires_grad_()
    assert not gemm._plain(xr, w) and not gemm._plain(w, x, xr)
    with torch.no_grad():
        assert gemm._plain(xr, w)
    assert not gemm._plain(x.as_subclass(OnGpu), w) and not gemm._plain(x.to_sparse(), w)
    with fwd.dual_level():
        assert gemm._plain(x, w)
        dual = fwd.make_dual(x, torch.ones_like(x))
        assert not gemm._plain(dual, w) and not gemm._plain(w, dual)
    torch.func.vmap(probe)(x[None])
    torch.func.jvp(probe, (x,), (x,))
    torch.func.grad(lambda v: probe(v).sum())(x)
    torch.jit.trace(probe, x, check_trace=False)
    with FlopCounterMode(display=False):
        probe(x)
    assert seen and not any(seen)


@pytest.mark.gpu
def test_long_contractions_and_cut_products_keep_tangents_and_transforms():
    import torch.autograd.forward_ad as fwd

    g = torch.Generator(device="cuda").manual_seed(1)
    for M_, N, K in ((512, 4096, 8192), (1900, 22016, 2048)):
        x, t = (torch.randn(M_, K, device="cuda", generator=g).bfloat16() for _ in range(2))
        w = torch.randn(N, K, device="cuda", generator=g).bfloat16()
        assert gemm.split_slices(x, w) or gemm._split_plan(x, w)
        with fwd.dual_level():
            y = fwd.unpack_dual(gemm.mm_nt(fwd.make_dual(x, t), w))
        want = torch.matmul(t, w.t())
        assert y.tangent is not None and ((y.tangent - want).norm() <= 2.0 ** -7 * want.norm())
        with torch.autocast("cuda", torch.float16):
            assert gemm.mm_nt(x, w).dtype == torch.float16


def test_few_row_rule_asks_for_a_plain_call(monkeypatch):
    x, w = torch.zeros(3, 128, **BF), torch.zeros(8, 128, **BF)
    wts, gu = torch.zeros(3, 2), torch.zeros(384, 128, **BF)
    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    assert gemm.thin_ok(x, w) and M.thin_act_ok(x, wts, gu, 2, 64, 64)
    for a, b, c in ((x.clone().requires_grad_(), wts, gu), (x, wts, gu.clone().requires_grad_()),
                    (x, wts.clone().requires_grad_(), gu)):
        assert not M.thin_act_ok(a, b, c, 2, 64, 64)
    assert not gemm.thin_ok(x.clone().requires_grad_(), w)
    assert not gemm.thin_ok(x, w.clone().requires_grad_())
    seen = []
    torch.func.vmap(lambda v: (seen.append(gemm.thin_ok(v, w)), v)[1])(x[None])
    assert seen == [False]


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 8])
def test_few_row_products_keep_gradients_tangents_and_batching(rows):
    """What the library answered before the few-row kernels: history, tangents, vmap."""
    import torch.autograd.forward_ad as fwd

    g = torch.Generator(device="cuda").manual_seed(rows)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g).bfloat16()  # noqa: E731
    x, t, w, b = r(rows, 4096), r(rows, 4096), r(256, 4096), r(256)
    near = lambda a, e: ((a - e).norm() <= 2.0 ** -7 * e.norm())  # noqa: E731
    for f, ref in ((lambda v: gemm.project(v, w), lambda v: v @ w.t()),
                   (lambda v: gemm.project(v, w, b), lambda v: v @ w.t() + b)) + (
                       ((lambda v: gemm.linear_nt(v, w), lambda v: v @ w.t()),) if rows > 4 else ()):
        xr = x.clone().requires_grad_()
        y = f(xr)
        assert y.requires_grad and near(y.detach(), ref(x))
        y.sum().backward()
        assert near(xr.grad, w.sum(0, keepdim=True).expand_as(x))
        assert near(torch.func.vmap(f)(x[None])[0], ref(x))
        with fwd.dual_level():
            tan = fwd.unpack_dual(f(fwd.make_dual(x, t))).tangent
        assert tan is not None and near(tan.float(), (t @ w.t()).float())
    xr = x.clone().requires_grad_()
    assert M.router_logits(xr, w).requires_grad == torch.mm(xr, w.t(), out_dtype=torch.float32).requires_grad


@pytest.mark.parametrize("M_,K,top,ff,kernels", [(1, 4096, 3, 64, 2), (2, 4096, 3, 64, 2), (1, 2048, 3, 64, 2),
                                                 (1, 4096, 3, 48, 0), (1, 4096, None, 64, 0)])
def test_one_row_skips_experts_at_any_width(launched, monkeypatch, M_, K, top, ff, kernels):
    """The GEMV's limit on K is one of a matrix that is read whole: it holds where no expert is skipped."""
    E = 16
    h, wts = torch.zeros(M_, K, **BF), torch.zeros(M_, E)
    gu, down = torch.zeros(2 * (E + 1) * ff, K, **BF), torch.zeros(64, (E + 1) * ff, **BF)
    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    monkeypatch.setattr(M, "project", lambda x, w, bias=None: torch.zeros(x.shape[0], w.shape[0], **BF))
    monkeypatch.setattr(M, "_act", lambda z, wts, E, ff, ffs, *a: torch.zeros(z.shape[0], E * ff + ffs, **BF))
    M.moe_dense(h, wts, gu, down, E, ff, ff, top=top)
    assert [n for n, _ in launched] == ["sm_thin_act", "sm_thin_gemm"][:kernels]


@pytest.mark.parametrize("M_", [1, 3])
def test_rows_too_far_apart_for_the_kernels_offsets_stay_with_the_library(launched, monkeypatch, M_):
    """The last rows of long sequences (hidden[:, -1]): 64 rows at the stride have to lie within 2^32 bytes."""
    w = torch.zeros(8, 128, **BF)
    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    for ld, ok in (((1 << 25) - 8, True), (1 << 25, False)):
        x = torch.empty(2 * ld + 128 if M_ > 1 else 128, device="meta", **BF).as_strided((M_, 128), (ld, 1))
        assert gemm.thin_ok(x, w.to("meta")) == ok
    h, wts = torch.empty(M_, 128, device="meta", **BF), torch.empty(M_, 1, device="meta")
    for ffs, ok in ((0, True), (64, False)):             # the second projection's K
        ff = (1 << 24) - 64
        gu = torch.empty(2 * (ff + ffs), 128, device="meta", **BF)
        assert M.thin_act_ok(h, wts, gu, 1, ff, ffs, sparse=True) == ok


@pytest.mark.parametrize("current,taken", [(1, True), (0, False)])
def test_products_of_another_device_follow_the_library(launched, monkeypatch, current, taken):
    """The kernels launch on the current device; the library goes where its operands are."""
    class Second(torch.Tensor):
        device = torch.device("cuda", 1)

    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: current, raising=False)
    for name in ("_plain", "use_native"):
        monkeypatch.setattr(gemm, name, lambda *a: True)
    on = lambda *s: torch.empty(*s, device="meta", **BF).as_subclass(Second)  # noqa: E731
    assert gemm.thin_ok(on(3, 128), on(8, 128)) == taken
    assert bool(gemm.split_slices(on(512, 8192), on(4096, 8192))) == taken
    asked = []
    monkeypatch.setattr(gemm, "skinny_ok", lambda *a: asked.append(a))
    monkeypatch.setattr(gemm.F, "linear", lambda *a: None)
    gemm.project(on(1, 4096), on(64, 4096))
    assert bool(asked) == taken


def test_decode_plans_are_read_for_calls_that_can_use_one(monkeypatch, tmp_path):
    """Neither with the plans switched off nor for CPU tensors (a file that is no table)."""
    bad = tmp_path / "plans.json"
    bad.write_text("{")
    monkeypatch.setenv("LUMEN_DGEMM_PLANS", str(bad))
    monkeypatch.setattr(gemm, "_dg_plans", None)
    x, w = torch.zeros(70, 64, **BF), torch.zeros(8, 64, **BF)
    assert gemm.dg_plan(x, w) is None and gemm.linear_nt(x, w).shape == (70, 8)
    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    monkeypatch.setattr(gemm, "DGEMM", False)
    assert gemm.dg_plan(x, w) is None


@pytest.mark.parametrize("E,W,ff,most", [(8, 1024, 704, 160), (8, 2048, 1408, 160), (4, 2048, 1408, 512), (4, 4096, 2816, 256),
                                         (8, 4096, 2816, 32), (16, 1024, 704, 64), (16, 2048, 1408, 32), (8, 256, 128, 64)])
def test_experts_own_rows_from_where_they_pay(E, W, ff, most):
    """``most``: the most rows that all experts serve; a few experts of a narrow layer serve more of them."""
    gu = torch.empty(2 * E * ff, W, device="meta")
    assert not M.chosen_pays(most, gu, E) and M.chosen_pays(most + 1, gu, E)


@pytest.mark.parametrize("lens,starts,width,tiles", [
    ([2], [510], 32, False), ([128] * 2, [1000] * 2, 71, False), ([256], [0], 16, False), ([320], [0], 20, True), ([80] * 3, [0] * 3, 5, True),
    ([5] * 64, [1000] * 64, 63, True), ([5] * 64, [200] * 63 + [8000], 501, False), ([300] * 2, [0] * 2, 600, True), ([16], [0], 600, True)])
def test_mixed_heads_of_few_rows_behind_many_keys(launched, monkeypatch, lens, starts, width, tiles):
    """A tile's chain is as long as the longest portion: short portions behind long contexts keep the row kernel."""
    from lumen.ops.attention import row_attention
    from lumen.ops.segments import SegBatch, portion_keys, tile_list

    monkeypatch.setattr(_seqmix, "talk_tiles_ok", lambda *a: True)
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    T, S, H, D = cu[-1], len(lens), 2, 128
    i32 = dict(dtype=torch.int32)
    row = torch.repeat_interleave(torch.arange(S), torch.tensor(lens)).int()
    seg = SegBatch(torch.tensor(cu, **i32), torch.arange(S, **i32), torch.tensor(starts, **i32), row, torch.zeros(T, **i32),
                   torch.zeros(S, width, **i32), None, torch.tensor(tile_list(cu, S), **i32).view(-1, 2), T, 128)
    q, k, v = torch.zeros(T, H, D, **BF), torch.zeros(1, 16, H, D, **BF), torch.zeros(1, 16, H, D, **BF)
    kv = [a + b for a, b in zip(lens, starts)]
    name = "sm_talk_tiles" if tiles else "sm_row_attn"
    for keys in (portion_keys(cu, kv, T), None):                # (without the host's count: by the tables' width)
        seg.keys, uneven = keys, width * 16 > 2 * max(kv) or max(kv) > 2 * min(kv)
        row_attention(q, None, k, v, D, torch.zeros(T, H, D, **BF), seg, H, H, 0.1, talk=torch.eye(H))
        if keys is not None or not uneven:
            assert [n for n, _ in launched] == [name]
        launched.clear()
    assert portion_keys(cu, kv, T + 1) is None and portion_keys(None, kv, T) is None and portion_keys(cu, None, T) is None


def test_latent_products_of_many_rows_keep_the_library(launched, monkeypatch):
    from lumen.ops import attention as A

    def run(T, H, D, R):
        launched.clear()
        q, uk = torch.zeros(T, H, D + 64, **BF), torch.zeros(H, D, R, **BF)
        assert A.latent_query(q, uk, uk.transpose(1, 2).contiguous(), D, torch.zeros(T, **i32)).shape == (H, T, R)
        return len(launched)

    i32 = dict(dtype=torch.int32)
    assert [run(*s) for s in ((1, 64, 128, 512), (128, 16, 128, 512), (129, 16, 128, 512), (64, 64, 128, 512), (512, 4, 128, 512),
                              (512, 16, 64, 128))] == [1, 1, 0, 0, 1, 1]
    monkeypatch.setattr(gemm, "_here", lambda *a: True)

    def expand(T, H, R, Dv):
        uv, o = torch.zeros(H, Dv, R, **BF), torch.zeros(T, H, Dv, **BF)
        return A._expand_ok((uv, o), torch.zeros(1, **BF), T, H, R)

    assert [expand(*s) for s in ((1, 64, 512, 128), (256, 16, 512, 128), (257, 16, 512, 128), (64, 64, 512, 128), (65, 64, 512, 128),
                                 (512, 4, 512, 128))] == [True, True, False, True, False, True]


@pytest.mark.parametrize("normed,sizes", [
    (False, ((1, 2048, 64, 1), (47, 3072, 64, 0), (48, 3072, 64, 1), (1, 8192, 64, 0), (1, 8192, 16, 1), (15, 6144, 32, 0),
             (16, 6144, 32, 1), (7, 4096, 33, 1))),
    (True, ((1, 4096, 64, 1), (31, 8192, 64, 0), (32, 8192, 64, 1), (1, 8192, 32, 1)))])
def test_large_routers_of_few_rows_keep_the_thin_gemm(normed, sizes):
    assert [M._route_rows_pay(T, W, E, normed) for T, W, E, _ in sizes] == [bool(s[3]) for s in sizes]


@pytest.mark.parametrize("lead", [(), (2,), (2, 3), (300, 2), (100, 2), (2, 3, 4)])
def test_products_of_rows_in_any_number_of_dimensions(lead):
    x, w = torch.randn(*lead, 8), torch.randn(5, 8)
    for f in (gemm.linear_nt, gemm.matmul_nt, gemm.mm_nt, gemm.project):
        assert torch.allclose(f(x, w), x @ w.t(), atol=1e-5)


def test_decoded_rows_take_the_same_products_eager_warmed_up_and_captured(monkeypatch):
    """The caller says that a step's rows are decoded; whether the stream is being captured is not asked."""
    from types import SimpleNamespace

    from lumen.serve.model_runner import ModelRunner

    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    for name in ("_plain", "_here", "use_native"):
        monkeypatch.setattr(gemm, name, lambda *a: True)
    x, w, down = (torch.empty(*s, device="meta", **BF) for s in ((100, 1024), (2048, 1024), (1024, 3200)))
    long, most = torch.empty(100, 3200, device="meta", **BF), torch.empty(300, 1024, device="meta", **BF)
    seen = []

    def routes(*a, **k):
        seen.append((gemm.tile_ok(x, w), gemm.split_slices(long, down), gemm.tile_ok(most, w)))

    for capturing in (False, True):
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing)
        routes()
        with gemm.decoded_rows():
            routes()
    routes()
    prompt, decoded = seen[0], seen[1]
    assert all(prompt) and decoded == (0, 0, prompt[2]) and seen == [prompt, decoded] * 2 + [prompt]

    seen.clear()
    run = SimpleNamespace(use_graphs=False, _decode_input=routes)
    ModelRunner.decode(run, SimpleNamespace(tokens=x))
    within = lambda *a, **k: nullcontext()  # noqa: E731
    stream = SimpleNamespace(wait_stream=lambda s: None)
    for name, v in (("stream", within), ("graph", within), ("Stream", lambda: stream), ("current_stream", lambda: stream),
                    ("CUDAGraph", object), ("graph_pool_handle", object)):
        monkeypatch.setattr(torch.cuda, name, v)
    run = SimpleNamespace(_static_inputs=lambda b: {}, _decode_static=routes, _graph_pool=None, _graphs={})
    ModelRunner._capture(run, 128)
    assert len(seen) == 4 and set(seen) == {decoded}


@pytest.mark.gpu
@pytest.mark.parametrize("M_,N,K", [(100, 2048, 1024), (128, 1024, 3200)])
def test_captured_products_are_the_warm_ups(M_, N, K):
    x, w = torch.randn(M_, K, device="cuda").bfloat16(), torch.randn(N, K, device="cuda").bfloat16()
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side), gemm.decoded_rows():
        want = [f(x, w) for f in (gemm.project, gemm.linear_nt)]
    torch.cuda.current_stream().wait_stream(side)
    with torch.cuda.graph(graph), gemm.decoded_rows():
        got = [f(x, w) for f in (gemm.project, gemm.linear_nt)]
    for _ in range(3):
        for y in got:
            y.zero_()
        graph.replay()
        assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("scan", ["wkv", "delta"])
def test_low_rank_decay_of_another_shape_is_not_read(launched, scan):
    """The scan reads row c of the second factor for channel c: one with fewer rows would be read past its end."""
    from lumen.ops import recurrent as R
    from lumen.ops.segments import SegBatch

    T, H, D = 3, 2, 64
    i32 = dict(dtype=torch.int32)
    at = torch.arange(T, **i32)
    seg = SegBatch(torch.arange(T + 1, **i32), at, at, at, at, None, None)
    x, w0, state = torch.zeros(T, H * D, **BF), torch.zeros(H * D), torch.zeros(T, H, D, D)

    def run(wl, w2):
        if scan == "wkv":
            return R.wkv_scan(x, x, x, wl, x, w0, w0, w0, state, seg, H, D, 1e-5, w2)
        return R.delta_scan(x, x, x, wl, x, x, w0, w0, w0, state, seg, H, D, 1e-5, 1.0, 1e-5, w2)

    wl, w2 = torch.zeros(T, 16, **BF), torch.zeros(H * D, 16, **BF)
    for a, b in ((wl, w2[:-1]), (wl, w2[:64]), (wl[:2], w2), (wl[:, :8], w2), (wl, w2.flatten())):
        with pytest.raises(ValueError):
            run(a, b)
    assert not launched
    assert run(wl, w2).shape == (T, H * D) and len(launched) == 1


@pytest.mark.parametrize("rows,K,apart", [(4096, 4096, True), (4096, 2048, True), (4096, 1024, True), (2176, 2048, False), (3072, 2048, False),
                                          (4224, 4096, False), (2048, 1088, True)])
def test_walks_apart_follow_the_distance_of_rows(monkeypatch, rows, K, apart):
    """Rows a multiple of 4 KiB apart meet in the same memory channels, however many of their columns are read."""
    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    for name in ("_plain", "_here", "use_native"):
        monkeypatch.setattr(gemm, name, lambda *a: True)
    x, w = torch.empty(40, K, device="meta", **BF), torch.empty(24576, rows, device="meta", **BF)[:, :K]
    code = gemm.tile_ok(x, w)
    assert code and (code > 255) == apart


def test_served_stacks_and_llama_take_the_same_products(monkeypatch):
    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    for name in ("_plain", "_here", "use_native", "thin_ok"):
        monkeypatch.setattr(gemm, name, lambda *a: True)
    for name in ("split_linear", "tile_linear", "_thin"):
        monkeypatch.setattr(gemm, name, lambda x, w, *a, name=name: (name, a[0] if a else None))
    split = 0
    for M_ in (17, 32, 33, 40, 64):
        x = {K: torch.empty(M_, K, device="meta", **BF) for K in (1024, 3072, 4096, 5632, 8192, 11008, 16384)}
        for K in x:
            for N in (2048, 4096, 5120, 7168, 7680, 8192, 12288, 32000):
                w = torch.empty(N, K, device="meta", **BF)
                got, want = gemm.project(x[K], w), gemm.linear_nt(x[K], w)
                assert got[0] == want[0] and (got[1] or 0) == (want[1] or 0), (M_, N, K)
                split += got[0] == "split_linear" and N >= gemm.FEW_MIN_N
    assert split


@pytest.mark.parametrize("T,H,heads,splits", [(16, 8, 4, 32), (16, 16, 8, 32), (8, 16, 4, 32), (14, 16, 8, 32), (1, 16, 4, 32), (32, 16, 16, 16),
                                              (64, 16, 16, 8), (64, 8, 8, 8)])
def test_halved_heads_of_few_rows_keep_as_many_splits(launched, T, H, heads, splits):
    """Behind a server's tables: rows of 4000 tokens on half the heads and half the splits took longer than before either."""
    from lumen.ops.attention import row_attention
    from lumen.ops.segments import SegBatch

    i32 = dict(dtype=torch.int32)
    at = torch.arange(T, **i32)
    seg = SegBatch(torch.arange(T + 1, **i32), at, at, at, at, torch.zeros(T, 256, **i32), None)
    q, kv = torch.zeros(T, H, 128, **BF), torch.zeros(1, 16, H, 128, **BF)
    row_attention(q, None, kv, kv.clone(), 128, torch.zeros(T, H, 128, **BF), seg, H, H, 0.1)
    (name, a), = launched
    assert name == "sm_row_attn" and a[-3] == splits and a[24] == heads


@pytest.mark.parametrize("T,H,G,bs,talk,offset,step", [
    (64, 16, 4, 16, False, 0, True), (64, 16, 8, 16, False, 0, True), (64, 32, 8, 64, False, 0, True), (8, 16, 4, 16, True, 0, True),
    (8, 32, 8, 8, True, 0, True), (64, 16, 4, 12, False, 0, False), (64, 16, 8, 24, False, 0, False), (8, 16, 4, 20, True, 0, False),
    (64, 16, 8, 16, False, 4, False), (8, 16, 4, 16, True, 4, False), (64, 16, 16, 16, False, 0, False), (64, 32, 2, 16, False, 0, False),
    (8, 32, 4, 16, True, 0, False), (8, 18, 9, 16, True, 0, False)])
def test_splits_of_the_keys_are_those_of_the_kernel_that_runs(launched, T, H, G, bs, talk, offset, step):
    """Behind tables of 4096 keys.  The kernels of decode steps deal keys out otherwise than the general one, which takes
    blocks of no power of two, heads one or 16 a key head, mixed heads eight a key head, and rows off 16 bytes."""
    from lumen.ops.attention import row_attention
    from lumen.ops.segments import SegBatch

    i32 = dict(dtype=torch.int32)
    at = torch.arange(T, **i32)
    seg = SegBatch(torch.arange(T + 1, **i32), at, at, at, at, torch.zeros(T, -(-4096 // bs), **i32), None)
    q, kv = torch.zeros(T, H * 128 + 8, **BF)[:, offset:offset + H * 128], torch.zeros(1, bs, G, 128, **BF)
    row_attention(q.view(T, H, 128), None, kv, kv.clone(), 128, torch.zeros(T, H, 128, **BF), seg, H, G, 0.1,
                  talk=torch.eye(H) if talk else None)
    (name, a), = launched
    blocks = T * -(-H // a[24])
    general = min(32, (1024 if not talk and a[24] <= 8 and blocks <= 32 else 512) // blocks)
    deep = min(64, 512 // T if talk else 1024 // (T * G))
    assert general != deep
    assert name == "sm_row_attn" and a[-3] == (deep if step else general)


@pytest.mark.parametrize("form", ["window", "talk", "latent", "decoded"])
@pytest.mark.parametrize("rows", [[1] * 5, [2100, 1, 1, 1], [2100, 1]])
def test_decoded_rows_behind_portions_are_dealt_out_as_decoded_rows(launched, monkeypatch, form, rows):
    """The portions' rows are another kernel's, so every row that is left is a sequence of its own."""
    from lumen.ops.attention import row_attention
    from lumen.ops.segments import SegBatch, tile_list

    monkeypatch.setattr(_seqmix, "talk_tiles_ok", lambda *a: True)
    i32, S, T = dict(dtype=torch.int32), len(rows), sum(rows)
    cu = [sum(rows[:i]) for i in range(S + 1)]
    P = rows.count(2100)
    seg = SegBatch(torch.tensor(cu, **i32), torch.arange(S, **i32), torch.zeros(S, **i32),
                   torch.repeat_interleave(torch.arange(S), torch.tensor(rows)).int(), torch.zeros(T, **i32), torch.zeros(S, 160, **i32),
                   None, torch.tensor(tile_list(cu, P), **i32).view(-1, 2) if P else None, cu[P], 128)
    H, n = 16, T
    if form == "decoded":
        seg, n = seg.decoded(), T - cu[P]
    if form in ("latent", "decoded"):
        q, c = torch.zeros(n, H, 576, **BF), torch.zeros(1, 16, 576, **BF)
        row_attention(q[:, :, :512], q[:, :, 512:], c, c, 512, torch.zeros(n, H, 512, **BF), seg, H, 1, 0.1, vt=torch.zeros(1, 512, 16, **BF))
        want = ["sm_latent_tiles"] * (P > 0 and form == "latent") + ["sm_latent_attn"]
    else:
        q, k = torch.zeros(n, H, 128, **BF), torch.zeros(1, 16, 4, 128, **BF)
        row_attention(q, None, k, k.clone(), 128, torch.zeros(n, H, 128, **BF), seg, H, 4, 0.1, talk=torch.eye(H) if form == "talk" else None)
        want = [{"window": "sm_win_attn_tiles", "talk": "sm_talk_tiles"}[form]] * (P > 0) + ["sm_row_attn"]
    assert [n for n, _ in launched] == want
    assert launched[-1][1][-4] == 1


def test_rows_of_one_portion_are_not_dealt_out_as_decoded_rows(launched):
    from lumen.ops.attention import row_attention
    from lumen.ops.segments import SegBatch

    i32 = dict(dtype=torch.int32)
    seg = SegBatch(torch.tensor([0, 40], **i32), torch.zeros(1, **i32), torch.zeros(1, **i32), torch.zeros(40, **i32), torch.arange(40, **i32),
                   torch.zeros(1, 160, **i32))
    q, k = torch.zeros(40, 16, 128, **BF), torch.zeros(1, 16, 4, 128, **BF)
    row_attention(q, None, k, k.clone(), 128, torch.zeros(40, 16, 128, **BF), seg, 16, 4, 0.1)
    assert launched[0][0] == "sm_row_attn" and launched[0][1][-4] == 0


@pytest.mark.parametrize("T,R,D2,splits", [(1, 512, 64, 64), (32, 512, 64, 16), (33, 512, 64, 15), (1, 384, 0, 64), (1, 256, 64, 64), (1, 512, 96, 32),
                                           (1, 384, 128, 32), (1, 256, 96, 32), (32, 512, 72, 16), (1, 192, 64, 32), (1, 64, 0, 32)])
def test_splits_of_latent_keys_are_of_the_tile_that_the_kernel_takes(launched, T, R, D2, splits):
    """Behind tables of 4096 keys: 64 splits of tiles of 128 keys would leave half of the workgroups without a key."""
    from lumen.ops.attention import row_attention
    from lumen.ops.segments import SegBatch

    i32 = dict(dtype=torch.int32)
    at = torch.arange(T, **i32)
    seg = SegBatch(torch.arange(T + 1, **i32), at, at, at, at, torch.zeros(T, 256, **i32), None)
    q, c = torch.zeros(T, 16, R + D2, **BF), torch.zeros(1, 16, R + D2, **BF)
    row_attention(q[:, :, :R], q[:, :, R:] if D2 else None, c, c, R, torch.zeros(T, 16, R, **BF), seg, 16, 1, 0.1,
                  vt=torch.zeros(1, R, 16, **BF))
    (name, a), = launched
    assert name == "sm_latent_attn" and a[-3] == splits


def test_scans_of_portions_without_rows(launched):
    from lumen.ops.recurrent import head_scan
    from lumen.ops.segments import SegBatch

    i32 = dict(dtype=torch.int32)
    seg = SegBatch(torch.zeros(3, **i32), torch.arange(2, **i32), torch.zeros(2, **i32), torch.zeros(0, **i32), torch.zeros(0, **i32))
    x = torch.zeros(0, 4 * 32, **BF)
    assert head_scan(x, x, x, torch.zeros(2, 4, 32, 32), seg, 4, 32, 32, torch.zeros(4)).shape == (0, 128)
    assert [n for n, _ in launched] == ["sm_head_scan_chunk"]


@pytest.mark.parametrize("R,Dr,T,H,keys,joined,plan", [
    (512, 64, 8, 16, 2048, False, (64, 32)), (512, 64, 8, 16, 2049, True, (128, 17)), (384, 64, 8, 16, 4096, False, (128, 32)),
    (512, 64, 16, 16, 2048, True, (128, 16)), (512, 64, 16, 16, 2560, True, (64, 32)), (256, 32, 32, 16, 1025, False, (64, 16)),
    (256, 32, 1, 16, 64, False, (64, 1)), (256, 32, 1, 16, 65, False, (128, 1)), (384, 64, 32, 4, 128, False, (128, 1)),
    (512, 64, 1, 16, 128, True, (64, 2)), (512, 64, 1, 16, 129, False, (64, 3)),
    (384, 64, 129, 32, 1024, True, (128, 4)), (384, 64, 129, 32, 896, True, (128, 1)), (512, 64, 258, 16, 1900, True, (128, 1)),
    (512, 64, 224, 32, 1900, False, (128, 4)), (512, 64, 225, 32, 1900, False, (128, 1)), (512, 64, 256, 32, 1900, False, (128, 1)),
    (512, 64, 257, 32, 1900, False, (128, 4)), (512, 64, 321, 32, 1900, False, (128, 1)), (256, 32, 140, 32, 1900, True, (128, 1)),
    (512, 96, 140, 32, 1900, True, (128, 1)), (512, 64, 64, 16, 1, False, (128, 1)), (512, 64, 64, 16, 4096, False, (128, 8))])
def test_tiles_and_splits_of_latent_keys(R, Dr, T, H, keys, joined, plan):
    """Tiles of 64 keys for few rows, of 128 where those are one round of the CUs or one split; four splits where blocks of heads of
    long contexts leave much of the last round idle."""
    assert _seqmix.latent_plan(R, R + Dr, T, H, keys, joined) == plan
