"""The few-row GEMM (seqmix/thin_gemm.hip) against float64 at the edges of its tiles: rows 1 .. 64
around every row class, columns that end inside a tile, k ranges with fewer stages than waves, strided
rows, bias, fp32 results; and the rule that sends a projection to it."""
import pytest
import torch

from lumen.ops.gemm import project, thin_linear, thin_ok

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
