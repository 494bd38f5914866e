"""Few-row projections whose last columns go through tanh or into a key cache in the epilogue."""
import pytest
import torch

from lumen.ops.gemm import project_tanh, project_write_keys

pytestmark = pytest.mark.gpu
ULP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}
SHAPES = [(1, 64, 64), (8, 100, 2048), (9, 2048, 128), (16, 8192, 4096), (17, 36, 5632), (33, 260, 1024), (64, 8196, 512),
          (65, 64, 64), (3, 64, 100)]


def near(got, want, dt):
    # one rounding; the separate launches round the product before its tanh as well
    err = (got.double() - want).abs()
    assert (err <= 2 * ULP[dt] * want.abs() + 1e-5 * want.abs().max() + ULP[dt] * (want.abs() < 1)).all(), err.max()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_tanh(M, N, K, dt):
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, K + 8, device="cuda", generator=g).to(dt)[:, :K]
    w = (torch.randn(N, K, device="cuda", generator=g) / K ** 0.5).to(dt)
    y = x.double() @ w.double().t()
    for start in (0, 5, N - 4, N - 1):
        head, tail = project_tanh(x, w, start)
        assert head.shape == (M, start) and tail.shape == (M, N - start)
        if start:
            near(head, y[:, :start], dt)
        near(tail, torch.tanh(y[:, start:]), dt)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_keys(M, N, K, dt):
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, K, device="cuda", generator=g).to(dt)
    w = (torch.randn(N, K, device="cuda", generator=g) / K ** 0.5).to(dt)
    for GD in (N, 16, 18):                                 # 18: columns that keep the separate launch
        G, D = (2, GD // 2) if GD % 2 == 0 else (1, GD)
        cache = torch.zeros(9, 8, G, D, device="cuda", dtype=dt)
        slots = torch.randperm(72, generator=torch.Generator().manual_seed(M))[:M].cuda()
        slots[M // 2] = -1
        y = project_write_keys(x, w, cache, slots, N - GD)
        near(y, x.double() @ w.double().t(), dt)
        want = torch.zeros(72, GD, device="cuda", dtype=dt)
        want[slots[slots >= 0]] = y[slots >= 0, N - GD:]
        assert torch.equal(cache.view(72, GD), want)
