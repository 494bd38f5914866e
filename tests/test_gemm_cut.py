"""Where a wide product is cut into whole waves of 256 x 256 tiles."""
import torch

from lumen.ops import gemm


def test_wave_cols():
    cuts = 0
    for M in (1, 255, 256, 300, 1300, 1900, 2048, 3300, 4010, 4096, 4874, 5120, 6500, 7300, 8000, 8192, 8193,
              9500, 65536, 65537, 1 << 20):
        for N in (8, 1000, 2048, 4096, 11008, 11264, 12288, 22016, 22020, 25344, 32000, 95744):
            n1 = gemm.wave_cols(M, N, 4096)
            tm, tn = -(-M // 256), -(-N // 256)
            assert n1 % 256 == 0 and 0 <= n1 < N
            if n1 or gemm.split_cols(M, N):
                assert M * N >= gemm.MIN_CUT
            if not n1:
                continue
            cuts += 1
            assert N % 8 == 0 and tm * tn % 256 and M <= 8192          # the measured range
            # the main part: at least two whole waves of the columns of tiles that fit one
            per_wave = 256 // tm
            waves = n1 // 256 // per_wave
            assert n1 // 256 % per_wave == 0 and 2 <= waves <= tm * tn // 256
            # no wave more than in one piece, but up to 8 waves, where a rest of two was faster all the same
            rest = tm * (tn - n1 // 256)
            if waves > 8:
                assert waves + -(-rest // 256) <= -(-tm * tn // 256)
            assert gemm.wave_cols(M, N, 1024) == 0
    assert cuts > 60
    assert gemm.wave_cols(4010, 22016, 4096) == 20480
    assert gemm.wave_cols(4874, 22016, 4096) == 72 * 256        # 20 row tiles: 12 columns a wave
    assert gemm.wave_cols(5100, 32000, 4096) == 0               # 9 waves, 340 tiles left: one wave more
    assert gemm.wave_cols(7300, 25344, 2048) == gemm.wave_cols(6500, 32000, 4096) == 0
    assert gemm.wave_cols(4096, 4096, 4096) == 0                # whole waves already
    assert gemm.wave_cols(300, 152064, 4096) == 2 * 128 * 2 * 256 and gemm.wave_cols(200, 152064, 4096) == 0


def test_cpu_and_tracked_calls_keep_one_product():
    x, w = torch.randn(300, 64, requires_grad=True), torch.randn(32, 64)
    y = gemm.mm_nt(x, w)
    y.sum().backward()
    assert torch.allclose(y, x @ w.t()) and x.grad is not None
    assert gemm.split_slices(x, w) == 0 and gemm._split_plan(x, w) == 0


def on_gpu(monkeypatch, enabled=True, tuning=False, results=()):
    """CPU (meta) tensors taken for the GPU's, and a tuned table that says so."""
    import torch.cuda.tunable as tn

    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    monkeypatch.setattr(tn, "is_enabled", lambda: enabled)
    monkeypatch.setattr(tn, "tuning_is_enabled", lambda: tuning)
    monkeypatch.setattr(tn, "get_results", lambda: list(results))
    monkeypatch.setattr(gemm, "_plans", {})
    monkeypatch.setattr(gemm, "_tuned", dict(gemm._tuned, n=-1))


def operands(M, N, K, dt=torch.bfloat16):
    return (torch.empty(M, K, dtype=dt, device="meta"), torch.empty(N, K, dtype=dt, device="meta"))


def test_no_product_is_cut_while_solutions_are_timed(monkeypatch):
    """TunableOp's rotating copies of a column view read past the end of the buffer it is a view of."""
    x, w = operands(4010, 22016, 4096)
    on_gpu(monkeypatch)
    assert gemm._split_plan(x, w) == 20480
    on_gpu(monkeypatch, tuning=True)
    assert gemm._split_plan(x, w) == 0
    on_gpu(monkeypatch, enabled=False, tuning=True)
    assert gemm._split_plan(x, w) == 20480


def test_plans_are_of_one_type_and_one_table(monkeypatch):
    """A bf16 solution says nothing of the fp16 product, and a plan made before the table was there
    does not outlive its loading."""
    sig = "tn_22016_2048_4096_ld_4096_4096_22016"
    cut = gemm.wave_cols(2048, 22016, 4096)
    bf, half = operands(2048, 22016, 4096), operands(2048, 22016, 4096, torch.float16)
    assert cut
    on_gpu(monkeypatch, results=[("GemmTunableOp_BFloat16_TN", sig, "x", 1.0)])
    for _ in range(2):
        assert gemm._split_plan(*bf) == 0 and gemm._split_plan(*half) == cut
    on_gpu(monkeypatch)                                          # before a table is loaded
    assert gemm._split_plan(*bf) == cut
    import torch.cuda.tunable as tn
    monkeypatch.setattr(tn, "get_results", lambda: [("GemmTunableOp_BFloat16_TN", sig, "x", 1.0)])
    assert gemm._split_plan(*bf) == 0 and gemm._split_plan(*half) == cut
    # the whole-wave parts of 4096 rows: tuned in bf16 only
    parts = [("GemmTunableOp_BFloat16_TN", f"tn_{n}_4096_4096_ld_4096_4096_22016", "x", 1.0)
             for n in (20480, 1536)]
    bf, half = operands(4096, 22016, 4096), operands(4096, 22016, 4096, torch.float16)
    on_gpu(monkeypatch, results=parts + [("GemmTunableOp_Half_TN", "tn_22016_4096_4096_ld_4096_4096_22016",
                                          "x", 1.0)])
    assert gemm._split_plan(*bf) == 20480 and gemm._split_plan(*half) == 0
    monkeypatch.setattr(tn, "get_results", lambda: [])
    gemm.forget_plans()                                          # another table has been read
    assert gemm._split_plan(*half) == gemm.wave_cols(4096, 22016, 4096)


def test_table_is_whole_when_its_size_says_it_is_read(monkeypatch):
    """A second thread that plans a product while the first reads the table."""
    class Watched(dict):
        def __setitem__(self, k, v):
            super().__setitem__(k, v)
            if k == "n":
                seen.append(gemm._tuned_sigs(torch.bfloat16))

    seen, sig = [], "tn_22016_2048_4096_ld_4096_4096_22016"
    on_gpu(monkeypatch, results=[("GemmTunableOp_BFloat16_TN", sig, "x", 1.0)])
    monkeypatch.setattr(gemm, "_tuned", Watched(n=-1, sigs={}))
    assert gemm._tuned_sigs(torch.bfloat16) == {sig} and seen == [{sig}]
