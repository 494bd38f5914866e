"""Where a wide product is cut into whole waves of 256 x 256 tiles."""
import torch

from lumen.ops import gemm


def test_wave_cols():
    for M in (1, 255, 256, 1900, 2048, 4010, 4096, 8000, 65536, 65537, 1 << 20):
        for N in (8, 1000, 2048, 4096, 11008, 11264, 12288, 22016, 22020, 32000):
            n1 = gemm.wave_cols(M, N, 4096)
            tm, tn = -(-M // 256), -(-N // 256)
            assert n1 % 256 == 0 and 0 <= n1 < N
            if n1 or gemm.split_cols(M, N):
                assert M * N >= gemm.MIN_CUT
            if n1:
                assert N % 8 == 0 and tm * tn % 256 and n1 // 256 * tm >= 2 * (256 // tm) * tm
            assert gemm.wave_cols(M, N, 1024) == 0
    assert gemm.wave_cols(4010, 22016, 4096) == 20480
    assert gemm.wave_cols(4096, 4096, 4096) == 0                # whole waves already


def test_cpu_and_tracked_calls_keep_one_product():
    x, w = torch.randn(300, 64, requires_grad=True), torch.randn(32, 64)
    y = gemm.mm_nt(x, w)
    y.sum().backward()
    assert torch.allclose(y, x @ w.t()) and x.grad is not None
    assert gemm.split_slices(x, w) == 0 and gemm._split_plan(x, w) == 0
