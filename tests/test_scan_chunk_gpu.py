"""The chunked prompt scans (seqmix/recurrent_chunk.hip) against float64 token loops: portions around the
chunk length, state carried over, head sizes on and off the blocks, decays from none to total, and rows
that are not finite."""
import math

import pytest
import torch

from _ref_gedatar import ref_unit_rms
from lumen.ops.recurrent import delta_scan, wkv_scan
from lumen.ops.segments import SegBatch, tile_list

pytestmark = pytest.mark.gpu
KEY_EPS, SCALE, EPS = 1e-6, math.exp(-0.5), 1e-6


def batch(pieces, decoded, starts):
    """Portions of ``pieces`` rows, then ``decoded`` one-row segments; slots in reverse."""
    cu = [0]
    for n in list(pieces) + [1] * decoded:
        cu.append(cu[-1] + n)
    S, i32 = len(cu) - 1, dict(dtype=torch.int32, device="cuda")
    t = torch.tensor
    rows = sum(pieces)
    row_seg = torch.cat([torch.full((b - a,), i) for i, (a, b) in enumerate(zip(cu, cu[1:]))])
    pos = torch.cat([torch.arange(b - a) + s for (a, b), s in zip(zip(cu, cu[1:]), starts)])
    return cu, SegBatch(t(cu, **i32), t(list(range(S))[::-1], **i32), t(starts, **i32),
                        row_seg.int().cuda(), pos.int().cuda(), None, None,
                        t(tile_list(cu, len(pieces)), **i32).view(-1, 2), rows, 128)


def rows(T, H, D, dtype, g, pad):
    return [torch.randn(T, H * D + pad, generator=g).to(dtype).cuda()[:, pad:] for _ in range(6)]


def exact(kind, x, w0, ub, nw, S0, H, D):
    """One segment from the state S0 in float64: (normed, gated rows; last state)."""
    f = lambda t: t.detach().cpu().double()  # noqa: E731
    r, k, v, wl, al, g = (f(t).reshape(-1, H, D) for t in x)
    z = wl + f(w0).view(H, D)
    S = S0.clone()
    out = []
    for t in range(r.shape[0]):
        kv = k[t][:, :, None] * v[t][:, None, :]
        if kind == "wkv":
            w = torch.exp(-torch.exp(z[t]))
            out.append(torch.einsum("hkv,hk->hv", S + f(ub).view(H, D)[:, :, None] * kv, r[t]))
            S = w[:, :, None] * S + kv
        else:
            w = torch.exp(-SCALE * torch.sigmoid(z[t]))
            un = k[t] / torch.sqrt(k[t].square().sum(-1, keepdim=True) + KEY_EPS)
            b = torch.sigmoid(al[t] + f(ub).view(H, D)) * un
            S = w[:, :, None] * S - b[:, :, None] * torch.einsum("hk,hkv->hv", un, S)[:, None] + kv
            out.append(torch.einsum("hkv,hk->hv", S, r[t]))
    gate = torch.sigmoid(g) * (g if kind == "wkv" else 1.0)
    y = ref_unit_rms(torch.stack(out), EPS) * f(nw).view(H, D) * gate
    return y.reshape(-1, H * D), S


def run(kind, x, w0, ub, nw, state, seg, H, D):
    r, k, v, wl, al, g = x
    if kind == "wkv":
        return wkv_scan(r, k, v, wl, g, w0, ub, nw, state, seg, H, D, EPS)
    return delta_scan(r, k, v, wl, al, g, w0, ub, nw, state, seg, H, D, EPS, SCALE, KEY_EPS)


@pytest.mark.parametrize("kind", ["wkv", "delta"])
@pytest.mark.parametrize("dtype,ulp", [(torch.bfloat16, 2.0 ** -8), (torch.float16, 2.0 ** -11)])
@pytest.mark.parametrize("H,D,pad", [(2, 128, 0), (3, 64, 8), (2, 32, 3), (1, 20, 0), (1, 256, 0),
                                     (2, 100, 4), (1, 136, 8)])
def test_portions_and_decoded_rows(kind, dtype, ulp, H, D, pad):
    g = torch.Generator().manual_seed(D + H)
    pieces, decoded = [1, 15, 16, 17, 33, 50], 2
    starts = [0, 3, 0, 40, 7, 0, 9, 0]
    cu, seg = batch(pieces, decoded, starts)
    x = rows(cu[-1], H, D, dtype, g, pad)
    w0 = torch.linspace(-3, 1, H * D).cuda()
    ub, nw = torch.randn(H * D, generator=g).cuda(), (1 + 0.1 * torch.randn(H * D, generator=g)).cuda()
    state = torch.randn(len(starts), H, D, D, generator=g).cuda()
    before = state.clone()
    y = run(kind, x, w0, ub, nw, state, seg, H, D)
    for s, (a, b) in enumerate(zip(cu, cu[1:])):
        slot = len(starts) - 1 - s
        S0 = before[slot].cpu().double() * (starts[s] > 0)
        want, S = exact(kind, [t[a:b] for t in x], w0, ub, nw, S0, H, D)
        # one rounding of the result; fp32 sums over <= 50 tokens and 256 channels: 2e-5 of a row's size
        err = (y[a:b].cpu().double() - want).abs()
        assert (err <= want.abs() * ulp + 2e-5 * want.abs().max()).all(), (s, err.max())
        assert (state[slot].cpu().double() - S).norm() <= 2e-6 * S.norm()


@pytest.mark.parametrize("H,D", [(2, 64), (1, 128)])
def test_wkv_decays_from_none_to_total(H, D):
    """exp(-exp(z)) for z from -20 (keeps everything) to 8 (keeps nothing), channel by channel and token
    by token: products over a chunk leave fp32's range many times over."""
    g = torch.Generator().manual_seed(5)
    cu, seg = batch([70], 0, [4])
    x = rows(70, H, D, torch.bfloat16, g, 0)
    x[3] = (torch.rand(70, H * D, generator=g) * 28 - 20).bfloat16().cuda()
    x[3][:, ::3] = 3.0                         # e^-20 a token: four of them pass 2^-80
    w0, ub, nw = torch.zeros(H * D).cuda(), torch.randn(H * D, generator=g).cuda(), torch.ones(H * D).cuda()
    state = torch.randn(1, H, D, D, generator=g).cuda()
    S0 = state[0].cpu().double()
    y = run("wkv", x, w0, ub, nw, state, seg, H, D)
    want, S = exact("wkv", x, w0, ub, nw, S0, H, D)
    err = (y.cpu().double() - want).abs()
    assert (err <= want.abs() * 2.0 ** -8 + 2e-5 * want.abs().max()).all()
    assert (state[0].cpu().double() - S).norm() <= 2e-6 * S.norm()


@pytest.mark.parametrize("H,D", [(2, 64), (1, 32), (1, 200)])
@pytest.mark.parametrize("T", [160, 161, 175])
def test_wkv_runs_of_cut_chunks(H, D, T):
    """Stretches whose chunks stay in range, whose every chunk is cut, and with single cuts; rows of one token and the end
    within a cut stretch; a row that is not finite among them."""
    g = torch.Generator().manual_seed(T + D)
    cu, seg = batch([T, 1, 2], 0, [0, 5, 0])
    x = rows(T + 3, H, D, torch.bfloat16, g, 0)
    z = torch.full((T + 3, H * D), -4.0)
    z[30:75, 7::16] = 2.0                      # e^-7.4 a token: 9 of them to a chunk
    z[95, 1] = z[97, 9] = z[120, 3] = 4.5      # one total decay in a chunk
    z[T - 25:, ::8] = 3.0                      # 3 to a chunk, up to the end and in the short portions
    x[3] = z.bfloat16().cuda()
    w0, ub, nw = torch.zeros(H * D).cuda(), torch.randn(H * D, generator=g).cuda(), torch.ones(H * D).cuda()
    state = torch.randn(3, H, D, D, generator=g).cuda()
    before = state.clone()
    y = run("wkv", x, w0, ub, nw, state, seg, H, D)
    for s, (a, b) in enumerate(zip(cu, cu[1:])):
        S0 = before[2 - s].cpu().double() * (s == 1)
        want, S = exact("wkv", [t[a:b] for t in x], w0, ub, nw, S0, H, D)
        err = (y[a:b].cpu().double() - want).abs()
        assert (err <= want.abs() * 2.0 ** -8 + 2e-5 * want.abs().max()).all()
        assert (state[2 - s].cpu().double() - S).norm() <= 2e-6 * S.norm()
    clean, at = y.clone(), 50
    x[2][at, 3] = float("inf")
    y = run("wkv", x, w0, ub, nw, before.clone(), seg, H, D)
    torch.testing.assert_close(y[:at], clean[:at], rtol=2.0 ** -7, atol=1e-4)
    torch.testing.assert_close(y[:T, D:], clean[:T, D:], rtol=2.0 ** -7, atol=1e-4)
    assert not torch.isfinite(y[at + 1, :D]).all()


@pytest.mark.parametrize("kind", ["wkv", "delta"])
def test_a_row_that_is_not_finite_spoils_no_earlier_row(kind):
    H, D = 2, 64
    g = torch.Generator().manual_seed(9)
    cu, seg = batch([40, 21], 0, [0, 0])
    x = rows(61, H, D, torch.bfloat16, g, 0)
    w0, ub, nw = torch.zeros(H * D).cuda(), torch.zeros(H * D).cuda(), torch.ones(H * D).cuda()
    clean = run(kind, x, w0, ub, nw, torch.zeros(2, H, D, D).cuda(), seg, H, D)
    x[2][21, 5] = float("nan")                 # a value of head 0
    x[1][50, 70] = float("inf")                # a key of head 1
    y = run(kind, x, w0, ub, nw, torch.zeros(2, H, D, D).cuda(), seg, H, D)
    tol = dict(rtol=2.0 ** -7, atol=1e-4)
    torch.testing.assert_close(y[:21], clean[:21], **tol)
    torch.testing.assert_close(y[40:50], clean[40:50], **tol)
    torch.testing.assert_close(y[21:40, D:], clean[21:40, D:], **tol)
    torch.testing.assert_close(y[50:, :D], clean[50:, :D], **tol)
    assert torch.isnan(y[21, :D]).any() and not torch.isfinite(y[51, D:]).all()


@pytest.mark.parametrize("kind", ["wkv", "delta"])
@pytest.mark.parametrize("what,by", [(1, 58), (0, 50), (0, -50), (1, -100), (2, 50), (1, 30)])
def test_large_and_small_values_of_a_range_without_end(kind, what, by):
    """bf16 reaches 2^127 (and the norm of a read-out 2^63): rows of r, k or v far from 1, under decays whose products over a chunk leave
    the range of the scaled rows, as the token-by-token walk takes them."""
    H, D, T = 2, 64, 50
    g = torch.Generator().manual_seed(7)
    cu, seg = batch([T], 0, [4])
    x = rows(T, H, D, torch.bfloat16, g, 0)
    scale = torch.ones(T, 1)
    scale[[3, 9, 10, 30]] = 2.0 ** by
    x[what] = (x[what].float().cpu() * scale).bfloat16().cuda()
    if what == 1 and by > 0:                    # products k v of ordinary size
        x[2] = (x[2].float().cpu() / scale).bfloat16().cuda()
    x[3][:, ::5] = 1.6                          # wkv: e^-5 a token
    w0, ub = torch.zeros(H * D).cuda(), torch.randn(H * D, generator=g).cuda()
    nw = torch.ones(H * D).cuda()
    state = torch.randn(1, H, D, D, generator=g).cuda()
    S0 = state[0].cpu().double()
    y = run(kind, x, w0, ub, nw, state, seg, H, D)
    want, S = exact(kind, x, w0, ub, nw, S0, H, D)
    err = (y.cpu().double() - want).abs()
    assert torch.isfinite(y).all() and torch.isfinite(state).all()
    # of each row's own size: one rounding of the result; fp32 sums over <= 50 tokens and 64 channels
    assert (err <= want.abs() * 2.0 ** -8 + 2e-5 * want.abs().amax(1, keepdim=True) + 1e-30).all()
    assert (state[0].cpu().double() - S).norm() <= 2e-6 * S.norm()


@pytest.mark.parametrize("kind", ["wkv", "delta"])
def test_rows_that_are_left_may_pass_32_bits(kind):
    """Rows left x row stride over 2^32 elements (a prompt of 105 k tokens in a fused projection of 41 k
    columns; here 70 rows at the largest stride): the chunk's own offsets stay in range."""
    H, D, T, ld = 1, 64, 70, (1 << 26) - 8
    g = torch.Generator().manual_seed(2)
    cu, seg = batch([T], 0, [0])
    x = rows(T, H, D, torch.bfloat16, g, 0)
    w0, ub, nw = torch.zeros(D).cuda(), torch.randn(D, generator=g).cuda(), torch.ones(D).cuda()
    s1, s2 = (torch.zeros(1, H, D, D).cuda() for _ in range(2))
    y = run(kind, x, w0, ub, nw, s1, seg, H, D)
    far = torch.empty((T - 1) * ld + D, dtype=torch.bfloat16, device="cuda").as_strided((T, D), (ld, 1))
    far.copy_(x[1])
    assert torch.equal(run(kind, [x[0], far, *x[2:]], w0, ub, nw, s2, seg, H, D), y) and torch.equal(s1, s2)


def test_a_total_decay_leaves_nothing():
    H, D = 1, 64
    g = torch.Generator().manual_seed(3)
    cu, seg = batch([20], 0, [4])
    x = rows(20, H, D, torch.bfloat16, g, 0)
    x[3].fill_(-3.0)
    x[3][5] = 5.0                               # exp(-e^5) = 0 in fp32
    w0, ub, nw = torch.zeros(D).cuda(), torch.zeros(D).cuda(), torch.ones(D).cuda()
    state = 2.0 ** 100 * torch.randn(1, H, D, D, generator=g).cuda()
    run("wkv", x, w0, ub, nw, state, seg, H, D)
    _, S = exact("wkv", x, w0, ub, nw, torch.zeros(H, D, D).double(), H, D)
    assert (state[0].cpu().double() - S).norm() <= 2e-6 * S.norm()


@pytest.mark.parametrize("kind,D", [("wkv", 64), ("delta", 64), ("delta", 128)])
def test_state_is_no_further_from_float64_than_the_serial_walk(kind, D, monkeypatch):
    import lumen.ops.recurrent as R

    H, err = 2, []
    g = torch.Generator().manual_seed(D)
    cu, seg = batch([400, 300], 0, [0, 5])
    x = rows(cu[-1], H, D, torch.bfloat16, g, 0)
    w0 = torch.linspace(-3, 1, H * D).cuda()
    ub, nw = 0.5 * torch.randn(H * D, generator=g).cuda(), torch.ones(H * D).cuda()
    before = torch.randn(2, H, D, D, generator=g).cuda()
    want = [exact(kind, [t[a:b] for t in x], w0, ub, nw, before[1 - i].cpu().double() * i, H, D)[1]
            for i, (a, b) in enumerate(zip(cu, cu[1:]))]
    for portions in (R._chunk_portions, lambda *a, **k: 0):          # the chunked kernel, the serial one
        monkeypatch.setattr(R, "_chunk_portions", portions)
        state = before.clone()
        run(kind, x, w0, ub, nw, state, seg, H, D)
        err.append(sum(((state[1 - i].cpu().double() - S).norm() / S.norm()).item()
                       for i, S in enumerate(want)))
    # measured over 36 portions: 0.94 - 1.0 of the serial walk's on average, +- 0.05 for one draw
    assert err[0] <= 1.1 * err[1], err


@pytest.mark.parametrize("kind", ["wkv", "delta"])
@pytest.mark.parametrize("H,D,n", [(9, 64, 30), (5, 20, 60), (3, 128, 90), (2, 256, 3)])
def test_more_workgroups_than_compute_units_and_one_key_for_all_rows(kind, H, D, n):
    """Grids of over 256 workgroups (fewer producer waves for the smaller heads), and rows that all carry one key with
    nearly whole removal: the chunk's triangular matrix is full, its powers grow though its inverse does not."""
    g = torch.Generator().manual_seed(D)
    pieces = [15 + 7 * (i % 3) for i in range(n)]
    starts = [i % 2 for i in range(n)]
    cu, seg = batch(pieces, 0, starts)
    x = rows(cu[-1], H, D, torch.bfloat16, g, 0)
    x[1][:] = x[1][:1].clone()
    x[4][:] = 4.0
    w0 = torch.full((H * D,), -6.0).cuda()
    ub, nw = torch.zeros(H * D).cuda(), torch.ones(H * D).cuda()
    state = torch.randn(n, H, D, D, generator=g).cuda()
    before = state.clone()
    y = run(kind, x, w0, ub, nw, state, seg, H, D)
    for s in list(range(0, n, 7)) + [n - 1]:
        a, b, slot = cu[s], cu[s + 1], n - 1 - s
        want, S = exact(kind, [t[a:b] for t in x], w0, ub, nw, before[slot].cpu().double() * (starts[s] > 0), H, D)
        # as above: one rounding of the result, fp32 sums
        err = (y[a:b].cpu().double() - want).abs()
        assert (err <= want.abs() * 2.0 ** -8 + 2e-5 * want.abs().max()).all(), (s, err.max())
        assert (state[slot].cpu().double() - S).norm() <= 2e-6 * S.norm()
