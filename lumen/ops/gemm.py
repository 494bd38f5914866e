"""Projection GEMMs for decode: y = x @ W^T.

Up to 64 rows the projection is a stream of the weight matrix: the HIP kernels
``seqmix/thin_gemm.hip`` (1 - 64 rows) and ``kernels/skinny_gemm.hip`` (1 row) run it where they
measured faster than a library GEMM; from 17 rows on wide results, results of about one round of its tiles, and long
contractions, cut along K, run on ``kernels/tile_gemm.hip``.  The rest (and CPU tensors) goes to ``torch.matmul``
(hipBLASLt with the tuned table)."""
from __future__ import annotations

import os
import threading
from contextlib import contextmanager
from typing import Optional

import torch
import torch.nn.functional as F
from torch.autograd import forward_ad

from ._native import native, use_native

# One row: the rows-per-lane weight-streaming kernel reaches 4.3-6.5 TB/s and beats hipBLASLt at
# every Llama-2-7B projection (qkv 17.0 vs 22.9 us, o 7.8 vs 22.7, gate_up 27.8 vs 37.3, down 16.5 vs
# 27.5, lm_head 38.4 vs 60.6); 2 - 4 rows that the thin kernel does not take (K not a multiple of 64)
# go to it as well, where it wins or ties (2 rows everywhere, 3 - 4 rows up to N = 4096).
SKINNY_MAX_M = int(os.environ.get("LUMEN_SKINNY_MAX_M", "4"))
SKINNY_MAX_N = int(os.environ.get("LUMEN_SKINNY_MAX_N", str(1 << 30)))
SKINNY_WIDE_MAX_M = 2  # above this M only N <= 4096 projections take the GEMV


def skinny_ok(x: torch.Tensor, w: torch.Tensor) -> bool:
    return (0 < x.shape[0] <= min(SKINNY_MAX_M, 16) and w.shape[0] <= SKINNY_MAX_N
            and (x.shape[0] <= SKINNY_WIDE_MAX_M or w.shape[0] <= 4096)
            and use_native(x) and x.dim() == 2
            and w.dim() == 2 and x.dtype == w.dtype and x.dtype in (torch.bfloat16, torch.float16)
            and x.stride(1) == 1 and w.is_contiguous() and x.shape[1] == w.shape[1]
            and (w.shape[0] % 4 == 0 and w.shape[1] % 8 == 0 and x.stride(0) % 8 == 0
                 if x.shape[0] <= 4 else w.shape[0] % 16 == 0 and w.shape[1] % 128 == 0))


def _plain(*tensors: torch.Tensor) -> bool:
    """A call with nothing to differentiate (backward or forward), batch, trace or cast: the kernels that
    are launched from here compute on the values alone."""
    grad = torch.is_grad_enabled()
    for t in tensors:
        if (grad and t.requires_grad or type(t) not in (torch.Tensor, torch.nn.Parameter)
                or t.layout is not torch.strided or t.is_neg()):
            return False
    if (torch.compiler.is_compiling() or torch._C._functorch.peek_interpreter_stack() is not None
            or torch._C._get_tracing_state() is not None or torch._C._len_torch_dispatch_stack()):
        return False
    if forward_ad._current_level >= 0 and any(
            forward_ad.unpack_dual(t).tangent is not None for t in tensors):
        return False
    return not (torch.is_autocast_enabled("cuda")
                and torch.get_autocast_dtype("cuda") != tensors[0].dtype)


def _here(x: torch.Tensor) -> bool:
    """Is ``x`` on the current device?  The library follows its operands to another one; the kernels
    launched from here take their memory and stream where the program is."""
    i = x.device.index
    return i is None or i == torch._C._cuda_getDevice()


# Thin GEMM (seqmix/thin_gemm.hip, whose header holds the measurements).  One row where the GEMV could take it:
# matrices under 128 MB with K <= 3072 (2048 x 2048: 3.8 vs 4.4 us with the GEMV; 2048 x 5632: 7.3 vs 6.6,
# 22528 x 4096: 30.7 vs 28.5, and a batch-1 Llama step of 4 layers of width 4096: 432 vs 407 us -- those stay
# with it).  33 - 64 rows: up to 24 M weights (11264 x 2048: 15.3 vs 17.6 us in the library; 22528 x 4096: 52.0 vs
# 45.1).  Anything between, and one row with an fp32 result (32000 x 4096: 44.0 vs 55.3 in the library): up
# to 208 M weights (50256 x 4096, 32 rows: 90.0 vs 96.8; 32000 x 8192, fp32 result: 108 vs 97).
THIN_MAX_M = 64
THIN_ROW_MAX_K, THIN_ROW_MAX_W = 3072, 1 << 26
THIN_BATCH_MAX_W = 24 << 20
THIN_MAX_W = 208 << 20
THIN_MAX_K, THIN_MAX_LD = 1 << 24, 1 << 25    # 64 rows lie within 32-bit byte offsets


def thin_ok(x: torch.Tensor, w: torch.Tensor, gemv: bool = True) -> bool:
    """Can and should the thin GEMM run x [M, K] @ w [N, K]^T?  ``gemv``: one row could go to the GEMV."""
    xs, ws = x.shape, w.shape                      # (in order of host time: short prompts wait for it)
    if len(xs) != 2 or not 0 < xs[0] <= THIN_MAX_M or len(ws) != 2 or not x.is_cuda:
        return False
    (M, K), (N, Kw), dt = xs, ws, x.dtype
    if (K != Kw or K % 64 or not 0 < K < THIN_MAX_K or N % 4 or dt != w.dtype
            or dt not in (torch.bfloat16, torch.float16) or x.device != w.device):
        return False
    if M == 1 and gemv:
        if K > THIN_ROW_MAX_K or N * K >= THIN_ROW_MAX_W:
            return False
    elif N * K > (THIN_MAX_W if M <= 32 else THIN_BATCH_MAX_W):
        return False
    if not _plain(x, w) or not w.is_contiguous() or not _here(x):
        return False
    ld, one = x.stride()
    return one == 1 and ld % 8 == 0 and K <= ld < THIN_MAX_LD and (x.data_ptr() | w.data_ptr()) % 16 == 0


def row_bias_ok(bias: Optional[torch.Tensor], x: torch.Tensor, N: int) -> bool:
    """Is ``bias`` (or None) one the kernels add: N consecutive values of x's type, on its device?"""
    return bias is None or (bias.dtype == x.dtype and bias.dim() == 1 and bias.shape[0] == N
                            and bias.is_contiguous() and bias.device == x.device)


def weights_ok(wts: Optional[torch.Tensor], h: torch.Tensor, E: int) -> bool:
    """Are ``wts`` routing weights the kernels read for the rows of ``h``: [rows, E] fp32, its device?"""
    return (wts is not None and wts.dtype == torch.float32 and wts.is_contiguous()
            and wts.dim() == 2 and wts.shape[0] == h.shape[0] and wts.shape[1] == E
            and wts.device == h.device)


def thin_linear(x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor] = None,
                out_dtype: Optional[torch.dtype] = None, blocks: Optional[tuple] = None
                ) -> torch.Tensor:
    """x [M, K] @ w [N, K]^T (+ ``bias`` [N]) on the thin GEMM kernel, fp32 accumulation; the result
    in x's dtype or (``out_dtype``) fp32.  ``blocks`` = (wts [M, E], E, ff, ffs): K is E blocks of ff
    and one of ffs, and the blocks whose column of wts is all zero are taken as zero without being
    read.  The kernel is handed bare addresses: what does not fit them is an error here."""
    if x.dim() != 2 or x.stride(1) != 1 or w.dim() != 2 or not w.is_contiguous() \
            or x.shape[1] != w.shape[1] or x.dtype != w.dtype or x.device != w.device:
        raise ValueError("few-row GEMM: rows x [M, K] and contiguous w [N, K] of one type and device")
    K, N = x.shape[1], w.shape[0]
    if not row_bias_ok(bias, x, N):
        raise ValueError(f"few-row GEMM: the bias is not [{N}] contiguous values like x's")
    if blocks is not None:
        wts, E, ff, ffs = blocks
        if not weights_ok(wts, x, E) or E * ff + ffs != K:
            raise ValueError("few-row GEMM: routing weights [M, E] in fp32, K = E blocks of ff and one of ffs")
    return _thin(x, w, bias, out_dtype, blocks)


def _thin(x, w, bias=None, out_dtype=None, blocks=None) -> torch.Tensor:
    """``thin_linear`` of operands that ``thin_ok``, ``row_bias_ok`` and ``weights_ok`` have let pass."""
    from ._seqmix import DT, call, use_seqmix

    use_seqmix(x)
    (M, K), N, dt = x.shape, w.shape[0], x.dtype
    y = torch.empty((M, N), device=x.device, dtype=out_dtype or dt)
    call("sm_thin_gemm", DT[dt], x, x.stride(0), w, bias, y, N, M, N, K, int(out_dtype is torch.float32),
         *(blocks or (None, 0, 0, 0)))
    return y


MID_MAX_M = 64            # rows seqmix/mid_gemm.hip takes


def mid_ok(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Can the kernels of seqmix/mid_gemm.hip multiply x [M, K] with w [N, K]^T?"""
    xs, ws = x.shape, w.shape
    if len(xs) != 2 or not 1 < xs[0] <= MID_MAX_M or len(ws) != 2 or not x.is_cuda:
        return False
    K, (N, Kw), dt = xs[1], ws, x.dtype
    if (K != Kw or K % 128 or not 0 < K < THIN_MAX_K or N % 4 or N == 0 or dt != w.dtype
            or dt not in (torch.bfloat16, torch.float16) or x.device != w.device or not w.is_contiguous()):
        return False
    ld, one = x.stride()
    return (one == 1 and ld % 8 == 0 and K <= ld < THIN_MAX_LD and (x.data_ptr() | w.data_ptr()) % 16 == 0
            and _plain(x, w) and _here(x))


def mid_slabs(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """fp32 sums of x @ w^T over S slices of K, [S, M, N], for operands that ``mid_ok`` has let pass.  A workgroup per
    CU, at most eight slices (us with the norm that adds them, 64 rows: 2048 x 5632 in 4 / 8 / 16 slices 14.1 / 12.4 / 14.9,
    1024 x 2816 10.1 / 8.6 / 9.8, 4096 x 11264 in 2 / 4 / 8 36.2 / 26.7 / 29.0, 3072 x 8448 in 4 / 5 / 8 20.7 / 19.7 / 22.3)."""
    from ._seqmix import DT, call, use_seqmix

    use_seqmix(x)
    (M, K), N = x.shape, w.shape[0]
    S = max(1, min(8, 256 // -(-N // 64), K // 128))
    y = torch.empty(S, M, N, dtype=torch.float32, device=x.device)
    call("sm_mid_slabs", DT[x.dtype], x, x.stride(0), w, y, M, N, K, S)
    return y


ROW_MAX_K = 8192          # K a workgroup of seqmix/row_gemv.hip holds


def row_norm_ok(x: torch.Tensor, norm_w: torch.Tensor, res: Optional[torch.Tensor], w: torch.Tensor) -> bool:
    """Can ``row_norm_linear`` run: one row, everything contiguous, of one 16-bit type and on one device?"""
    xs = x.shape
    if len(xs) != 2 or xs[0] != 1 or not x.is_cuda or w.dim() != 2:
        return False
    K, (N, Kw), dt = xs[1], w.shape, x.dtype
    if (K != Kw or K % 8 or not 0 < K <= ROW_MAX_K or N % 4 or N == 0 or dt != w.dtype
            or dt not in (torch.bfloat16, torch.float16) or tuple(norm_w.shape) != (K,)):
        return False
    ts = (x, norm_w, w) if res is None else (x, norm_w, w, res)
    return (all(t.dtype == dt and t.device == x.device and t.is_contiguous() and t.data_ptr() % 16 == 0 for t in ts)
            and (res is None or res.shape == xs) and _plain(*ts) and _here(x) and use_native(x))


def row_norm_linear(x: torch.Tensor, norm_w: torch.Tensor, eps: float, res: Optional[torch.Tensor],
                    w: torch.Tensor, gated: bool = False) -> tuple:
    """(y, s) of one row: s = x + ``res`` (x itself without one), y = w rms_norm(s) -- ``gated``: silu(first half) *
    second half of it.  For operands that ``row_norm_ok`` has let pass."""
    from ._seqmix import DT, call, use_seqmix

    use_seqmix(x)
    K, N = x.shape[1], w.shape[0]
    F = N // 2 if gated else N
    y = torch.empty((1, F), device=x.device, dtype=x.dtype)
    s = torch.empty_like(x) if res is not None else x
    call("sm_row_gemv", DT[x.dtype], x, res, norm_w, s if res is not None else None, w, y, K, F, int(gated), eps)
    return y, s


def row_stream_ok(x: torch.Tensor, y: Optional[torch.Tensor], norm_w: torch.Tensor, w: torch.Tensor,
                  bias: Optional[torch.Tensor] = None) -> bool:
    """Can ``row_stream_linear`` run: one fp32 row ``x`` and its norm's weight, ``y``, ``w`` and ``bias`` of one 16-bit type?"""
    xs = x.shape
    if len(xs) != 2 or xs[0] != 1 or not x.is_cuda or w.dim() != 2 or w.dtype not in (torch.bfloat16, torch.float16):
        return False
    K, (N, Kw), dt = xs[1], w.shape, w.dtype
    if K != Kw or K % 8 or not 0 < K <= ROW_MAX_K or N == 0 or tuple(norm_w.shape) != (K,) \
            or x.dtype != torch.float32 or norm_w.dtype != torch.float32:
        return False
    ts = (x, norm_w, w) if y is None else (x, norm_w, w, y)
    return (all(t.device == x.device and t.is_contiguous() and t.data_ptr() % 16 == 0 for t in ts)
            and (y is None or y.shape == xs and y.dtype == dt)
            and (bias is None or row_bias_ok(bias, w, N) and _plain(bias)) and _plain(*ts) and _here(x) and use_native(x))


def row_stream_linear(x: torch.Tensor, y: Optional[torch.Tensor], norm_w: torch.Tensor, eps: float, w: torch.Tensor,
                      bias: Optional[torch.Tensor] = None, act: Optional[str] = None, out32: bool = False) -> tuple:
    """(z, s) of one row of an fp32 stream that a sublayer's output ``y`` joins: s = x + y (x itself without one), z = act(w
    rms_norm(s) + bias), in w's type or (``out32``) fp32.  For operands that ``row_stream_ok`` has let pass.  (HIP
    ``csrc/seqmix/row_gemv.hip``.)"""
    from ._seqmix import DT, call, use_seqmix
    from .moe import GATE_ACTS

    use_seqmix(x)
    K, N = x.shape[1], w.shape[0]
    z = torch.empty((1, N), device=x.device, dtype=torch.float32 if out32 else w.dtype)
    s = torch.empty_like(x) if y is not None else x
    call("sm_row_stream", DT[w.dtype], x, y, norm_w, s if y is not None else None, w, bias, z, K, N,
         -1 if act is None else GATE_ACTS[act], int(out32), eps)
    return z, s


# Split-K GEMM (kernels/tile_gemm.hip): contractions whose output has too few tiles to fill the chip.  Tiles of 128 columns
# and 64 rows, from 65 rows on 128, from some 200 on 256.  us, library or thin kernel -> split:
#  * 241 rows and more, K from 8192 on: K = 11008, N = 4096, rows 256 / 512 / 1000: 51 -> 35, 72 -> 50, 113 -> 87; K = 22016 at 512:
#    139 (tuned) -> 91; K = 32000 at 512: 290 -> 123; K = 11264, N = 2048 at 320 / 1000: 48 -> 32, 72 -> 51.  Below, the slabs cost
#    what the split gains (K = 4096 at 512 rows: 28.2 and 28.4).
#  * 33 - 64 rows (256-row tiles were no gain): 64 x 2048 x 11264 32.7 -> 19.5, x 8192 23.9 -> 16.4, 64 x 4096 x 11008 33.3 -> 25.4, 48 x
#    3072 x 5632 17.7 -> 15.6 (33 x 4096 x 5632 16.2 -> 17.8); 17 - 32 rows from K = 11008 on: 24 x 2048 x 11264 21.5 -> 18.4 (3072 x 8448 17.5 -> 18.3).  Shorter K where
#    neither the thin kernel nor few_tiles takes the width: 64 x 5120 x 4096 24.5 -> 16.5, 6144 x 3072 21.1 -> 15.7; but 64 x 4096 x
#    4096 14.4 -> 14.9, 2048 x 5632 13.6 -> 13.2, 8192 x 4096 18.9 -> 20.1.
#  * 65 - 128 rows (256-row tiles -> 128): 128 x 4096 x 11008 39.2 -> 29.1, 72 x 2048 x 8192 23.0 -> 18.5; library -> here 128 x 4096 x 5632
#    33.6 -> 21.7, 72 x 4096 x 4096 22.1 -> 17.9, 100 x 8192 x 4096 25.1 -> 23.9; but 2048 x 5632 13.9 -> 16.4, 3072 x 4096 14.5 -> 16.4.
#  * 129 - 240 rows: 180 x 4096 x 11008 44.4 -> 34.6, 180 x 3072 x 5632 26.8 -> 21.3, 224 x 6144 x 4096 38.7 -> 27.9; 180 x 6144 x 4096 even.
# Over 128 tiles a slice would be less than half of K on more workgroups than CUs; under 128 workgroups most CUs idle.
# Walks apart (as in few_tiles) for up to 256 rows of 4096 columns and more.  Slices already start at different k, and which K
# still meet in the same channels was not to be told from the rows' distance (us, in step / apart: 64 x 8192 x 8192 40.1 / 33.2, 64 x 6144 x 11008
# 39.4 / 32.3, but x 11264 32.7 / 33.3, 256 x 6144 x 14336 57.0 / 60.1, x 4096 x 8192 31.1 / 33.1): over 280 sizes of K 3072 - 14336 apart is
# 0.94 - 1.22 times as fast, 1.016 in the mean, and under 4096 columns even but for K = 11008 (80 sizes, 1.018).
# Between the sizes above: 255 drawn ones of 17 - 256 rows, K 3072 - 14400 1.34 times as fast as the better of the thin kernel and the library
# in the mean, three of them below 0.97 (worst 66 x 4512 x 4096 16.6 -> 19.6).
SPLIT_MIN_K, SPLIT_FEW_K, SPLIT_MAX_S, SPLIT_FEW_M = 8192, 3072, 8, 240


def split_plan(M: int, N: int, K: int) -> int:
    """The split-K GEMM's form for x [M, K] @ w [N, K]^T: S slices + 16 mj + 256 for walks apart (mj 8, in step: S alone), or 0."""
    if M < FEW_MIN_M or K < (SPLIT_FEW_K if M <= SPLIT_FEW_M else SPLIT_MIN_K):
        return 0
    if M <= 32:
        if K < 11008 or not 4096 <= N <= 8192:
            return 0
    elif K >= SPLIT_MIN_K:
        if N > 8192 if M <= 64 else N < 2048 and M <= SPLIT_FEW_M:
            return 0
    else:
        wide = 4096 < N < FEW_MIN_N
        if M <= 64:
            pays = wide or K >= 5632 and 3072 <= N <= 4096 and M > 40
        elif M <= 128:
            pays = wide or (K >= 5632 and N >= 3072 or K >= 4096 and N >= 4096) and N <= 8192
        else:
            pays = K >= 4096 and (wide or N == 4096) or K >= 5632 and 3072 <= N < FEW_MIN_N
        if not pays:
            return 0
    mj = (8 if M > SPLIT_FEW_M else 2 if M <= 64 else
          4 if M <= 128 or N <= (5376 if M <= 192 else 2048 if K >= SPLIT_MIN_K else 4096) else 8)
    tiles = -(-M // (32 * mj)) * -(-N // 128)
    if not 0 < tiles <= 128:
        return 0
    S = min(SPLIT_MAX_S if M > SPLIT_FEW_M else 12, TILE_CUS // tiles)
    if tiles * S < 128:
        return 0
    apart = 256 if M <= 256 and N >= 4096 else 0
    return S + apart + 16 * mj if apart or mj < 8 else S


def split_slices(x: torch.Tensor, w: torch.Tensor) -> int:
    """``split_plan`` of x [M, K] @ w [N, K]^T of 65 rows and more, 0 where the kernel cannot run it (leave it to the others)."""
    return _slices(x, w) if x.shape[0] > THIN_MAX_M else 0


def _slices(x: torch.Tensor, w: torch.Tensor) -> int:
    xs = x.shape
    if len(xs) != 2 or xs[1] < SPLIT_FEW_K or w.dim() != 2 or not x.is_cuda:
        return 0                                   # (nearly every call: as little host time as can be)
    (M, K), (N, Kw), dt = xs, w.shape, x.dtype
    S = split_plan(M, N, K)
    if not S and not (_step.decoded and M <= REPLAY_MAX_M):
        S = short_slices(M, N, K)
    if (not S or K != Kw or K % 64 or N % 4 or K >= 1 << 22 or dt != w.dtype
            or dt not in (torch.bfloat16, torch.float16) or x.device != w.device
            or not _plain(x, w) or not _here(x) or not use_native(x)):
        return 0
    return S if _aligned(x, w, K) else 0


def split_linear(x: torch.Tensor, w: torch.Tensor, S: int) -> torch.Tensor:
    """x [M, K] @ w [N, K]^T in slices of K, their fp32 sums added in order and rounded once.  Callers
    take S from ``split_slices``."""
    return native().split_gemm(x, w, S & 15, S >> 4 & 15 or 8, S > 255)


# One round of 256 x 32 ni tiles (kernels/tile_gemm.hip) where some ni makes the result about one wave of the chip.  At
# 0.85 of the tiles' area filled it is as fast as the library or faster over 350 shapes of 300 - 8000 rows, K 512 - 22016,
# both types, tuned solutions included (us, library -> tiles: 4010 x 2048 x 2048 32.4 -> 31.3, x 5632 75 -> 72, x 11264 161
# -> 143, 4010 x 2560 x 2048 44 -> 37, 2048 x 4096 x 11008 160 -> 143, 1000 x 8192 x 2048 34.7 -> 32.3, 512 x 22528 x
# 4096 89 -> 84; worst 1280 x 8192 x 5632, filled 0.83, 96 -> 105).  Where N is no multiple of 1024 the library's own tiles fill
# badly too: from 0.75 on (4010 x 2112 x 2048 42 -> 34, 3000 x 2112 x 2048 36 -> 29, 700 x 11264 x 2048 45 -> 36;
# worst 3000 x 1536 x 2048, 0.73, 23.2 -> 24.4).
TILE_MIN_M, TILE_MIN_K, TILE_CUS = 256, 512, 256
TILE_FILL, TILE_FILL_ODD = 0.85, 0.75


def tile_columns(M: int, N: int, K: int) -> int:
    """``ni`` of the 256 x 32 ni tiles on which x [M, K] @ w [N, K]^T should run (0: leave it to the library)."""
    if M < TILE_MIN_M or K < TILE_MIN_K:
        return 0
    tm = -(-M // 256)
    for ni in (3, 4, 5, 6):
        if tm * -(-N // (32 * ni)) <= TILE_CUS:
            fill = M * N / (TILE_CUS * 8192 * ni)
            return ni if fill >= TILE_FILL or N % 1024 and fill >= TILE_FILL_ODD else 0
    return 0


# Up to 256 rows of wide matrices, and 96- and 160-column tiles above (us, library or thin kernel -> here, bf16, weights
# from HBM; K where nothing is said 4096).  A tile takes 64 rows, from 65 on 128, for the widest from 177 on 256, and the
# narrowest number of columns that makes the result one round of workgroups.
#  * Tiles of one column start their walk of k apart where rows of w lie a multiple of 4 KiB apart: in step, all tiles would
#    read a stage of their rows from the same memory channels (in step / apart: 40 x 24576 45.9 / 38.8, x 2048 26.0 / 21.4, x
#    6144 71.6 / 57.0; x 3072 30.5 / 31.0; columns of a wider matrix go by its rows: 24576 x 2816 of rows of 4096 33.6 / 28.7, x 4096 of rows
#    of 4224 38.3 / 38.8).  The library and the thin kernel walk in step, so this is where most is gained.
#    From 257 rows on x costs more than w and is better read in step.
#  * 17 - 64 rows, from three quarters of a round on (32 columns: nine tenths): 40 x 8192 18.4 -> 16.7, 24576 47.5 -> 38.8, 32000 61 -> 48, 64000 124 -> 98, 32000
#    x 2048 33.6 -> 27.7, 24576 x 1024 19.4 -> 13.2.  Not less than that (40 x 4096 12.6 -> 15.2).  Long K in step only with 32
#    or 96 columns (40 x 8192 x 2816 19.9 -> 13.3, 24576 x 5120 51.2 -> 48.8; 64 x 14336 x 5120 33.3 -> 36.1, 7680 x 5632 25.2
#    -> 26.6, 32000 x 5120 63.6 -> 67.4).  Up to 32 rows the thin kernel keeps 32-column tiles of long K (20 x 8192 14.7 -> 15.9) and what takes
#    128 - 192 columns (20 x 32000 x 2048 26.5 -> 27.4).
#  * 65 - 128 rows, from nine tenths of a round on, up to K = 2048 three quarters: 100 x 22016 49.1 -> 41.3, 32000 64 -> 51, 64000
#    132 -> 104, 12288 x 1024 12.1 -> 10.3; not long K in step (32000 x 2816 39.3 -> 39.5, 128 x 22016 x 2816 32.8 -> 35.2).
#  * 177 - 256 rows as 2 x 64- or 96-column tiles: 256 x 8192 42.5 -> 31.9, x 12288 x 2048 28.5 -> 22.3, 180 x 12288 40.6 -> 33.8, 8192
#    27.5 -> 27.1; as 256 x 96: 200 x 22016 60.8 -> 56.1, x 1024 22.4 -> 19.5, x 5120 even.  At
#    130 - 160 rows the second row tile is mostly padding (161 x 24576 x 1024 19.8 -> 21.8).
#  * above: 1000 x 3072 32.3 -> 29.0, 500 x 5120 38.1 -> 34.6, 1000 x 5120 50.3 -> 46.3, x 1024 19.2 -> 15.8; long K even (512 x 5120 x
#    5632 49.1 -> 49.5), other widths are the library's (512 x 8192 41.7 -> 42.8, 768 x 6144 x 2816 33.9 -> 34.2).
# Between the sizes above: 245 drawn ones of 17 - 256 rows, 7168 - 66000 columns and K 1024 - 8128 1.14 times as fast as the better of the thin
# kernel and the library in the mean, one of them below 0.97 (250 x 12048 x 7936 71.9 -> 75.8).
FEW_MIN_M, FEW_MIN_N, FEW_MIN_MN = 17, 7168, 1 << 21
FEW_NI = {2: (1, 2, 3, 4, 5, 6, 8), 4: (2, 3, 4, 5, 6, 8), 8: (3, 4, 5, 6)}


def _round(M: int, N: int, mj: int) -> tuple:
    """(ni, filled share of its rounds) of the narrowest 32 mj x 32 ni tiles that are one round, else the widest."""
    tm = -(-M // (32 * mj))
    for ni in FEW_NI[mj]:
        tiles = tm * -(-N // (32 * ni))
        if tiles <= TILE_CUS:
            break
    return ni, tiles / (-(-tiles // TILE_CUS) * TILE_CUS)


def few_tiles(M: int, N: int, K: int, ld: Optional[int] = None) -> int:
    """The tiles on which x [M, K] @ w [N, K]^T should run beside ``tile_columns``: ni + 16 mj + 256 for walks apart, or 0.  ``ld``:
    elements from one row of w to the next (K)."""
    if M < FEW_MIN_M or K < 1024 or K >= SPLIT_MIN_K:
        return 0
    if M > 256:
        if K > 4096 or M * N > TILE_CUS * 4096 * 5:    # (first: short prompts and training steps wait for the host)
            return 0
        tm, lead = -(-M // 128), 0.8 * TILE_CUS * 4096
        if tm * -(-N // 96) <= TILE_CUS < tm * -(-N // 64):
            return 3 + 64 if M * N >= 3 * lead else 0
        if tm * -(-N // 160) <= TILE_CUS < tm * -(-N // 128):
            return 5 + 64 if M * N >= 5 * (lead if K <= 2048 else 0.95 * TILE_CUS * 4096) else 0
        return 0
    apart = 256 if (ld or K) % 2048 == 0 else 0
    free = apart or K <= 2048                          # not held up by what the others read
    if M <= 64:
        ni, fill = _round(M, N, 2)
        pays = fill >= (0.88 if ni == 1 else 0.72) and (free or ni in (1, 3)) and (
            K <= (3072 if M <= 32 else 4096) if ni == 1 else M > 32 or ni <= 3 or ni == 8)
        return ni + 32 + apart if pays else 0
    if M <= 128:
        ni, fill = _round(M, N, 4)
        return ni + 64 + apart if free and N <= 65536 and fill >= (0.72 if K <= 2048 else 0.88) else 0
    if M <= 176:
        return 0
    ni, fill = _round(M, N, 4)
    if ni <= 3:
        return ni + 64 + apart if fill >= 0.88 else 0
    ni, fill = _round(M, N, 8)
    return ni + 128 + apart if ni == 3 and fill >= 0.88 and (apart or K <= 4608) else 0


# Short products of prompts: the library takes the host 18 us a call (19 - 21 with a tuned table, which is asked), its kernel 5 - 17, so a
# step of 65 - 1000 rows of width 1024 - 2048 waits for the host whatever the card does; a tile launch takes the host 8 us and the card
# no more than 18, one round of 128-row tiles whose walk of k is short (from K = 2049 on for the down projections of narrow models).  (Above, the kernel's own time counts: 4010 x 576 x
# 2048 13.2 us in the library, 17 here.  So it does in a step of decoded rows, which a graph replays without the host:
# 128 x 2048 x 2048 9.3 us in the library, 11.2 - 13 here: see ``decoded_rows``.)
# Steps of 4 layers, us: Llama, 200 tokens of width 1024 663 -> 445, 100 of width 2048 668 -> 528; dalavik 1159 -> 787, 1148 -> 859; silonex 831 ->
# 608, 824 -> 694; where the card is nearly the longer one (tazulix, 240 of width 2048) 780 -> 774.
SHORT_MK, SHORT_NIK, SHORT_MAX_K, SHORT_NK = 1 << 20, 6144, 3072, 1 << 22
REPLAY_MAX_M = 256        # the most decoded rows a graph replays


class _Step(threading.local):
    decoded = False


_step = _Step()


@contextmanager
def decoded_rows():
    """Products of this thread belong to a step of decoded rows.  The caller says so for the eager step, the warm-up of a
    capture and the capture alike, so all of them run the same kernels (and round alike), and the library has seen each
    of its products before one is captured."""
    before, _step.decoded = _step.decoded, True
    try:
        yield
    finally:
        _step.decoded = before


def short_tiles(M: int, N: int, K: int) -> int:
    """The tiles (as ``few_tiles``) of a product that is over before the host has called the library for the next, or 0."""
    if M <= THIN_MAX_M or M * K > SHORT_MK or K > 2048 and (K > SHORT_MAX_K or N * K > SHORT_NK) or K < 128 or N < 64:
        return 0
    tm = -(-M // 128)
    for ni in (2, 3, 4, 5):
        if tm * -(-N // (32 * ni)) <= TILE_CUS:
            return ni + 64 if ni * K <= SHORT_NIK else 0
    return 0


def short_slices(M: int, N: int, K: int) -> int:
    """As ``short_tiles`` for longer walks of k: the split-K GEMM's form (``split_plan``) on 128-row tiles, or 0.  Two launches of 11 us
    for the host; 180 x 2048 x 5632 18.1 us on the card, 17.8 in the library, 100 rows 15.5 and 13.1."""
    if M <= THIN_MAX_M or not SHORT_MAX_K < K < SPLIT_MIN_K or M * K > 2 * SHORT_MK or N * K > 3 * SHORT_NK or N < 1024:
        return 0
    tiles = -(-M // 128) * -(-N // 128)
    S = min(12, TILE_CUS // tiles, K // 256)
    return S + 64 if S > 1 else 0


def _aligned(x: torch.Tensor, w: torch.Tensor, K: int) -> bool:
    (lx, ex), (lw, ew) = x.stride(), w.stride()
    return (ex == 1 and ew == 1 and lx % 8 == 0 and lw % 8 == 0 and K <= lx <= 1 << 22 and K <= lw <= 1 << 22
            and (x.data_ptr() | w.data_ptr()) % 16 == 0)


def tile_ok(x: torch.Tensor, w: torch.Tensor) -> int:
    """``tile_columns``, ``few_tiles`` or ``short_tiles`` of x @ w^T, 0 where the kernel cannot run it."""
    xs, ws = x.shape, w.shape
    if len(xs) != 2 or len(ws) != 2 or not x.is_cuda:
        return 0
    (M, K), (N, Kw), dt = xs, ws, x.dtype
    ni = tile_columns(M, N, K) or (few_tiles(M, N, K, w.stride(0)) if M > 256 or N >= FEW_MIN_N else 0)
    if not ni and not (_step.decoded and M <= REPLAY_MAX_M):
        ni = short_tiles(M, N, K)
    if (not ni or K != Kw or K % 64 or N % 4 or K >= 1 << 22 or dt != w.dtype
            or dt not in (torch.bfloat16, torch.float16) or x.device != w.device
            or not _plain(x, w) or not _here(x) or not use_native(x) or not _aligned(x, w, K)):
        return 0
    return ni


def tile_linear(x: torch.Tensor, w: torch.Tensor, ni: int, bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """x [M, K] @ w [N, K]^T (+ ``bias`` [N]) on 256 x 32 ni tiles or ``few_tiles``', rounded once.  Callers take ``ni`` from
    ``tile_ok``."""
    return native().tile_gemm(x, w, ni & 15, bias, None, ni >> 4 & 15 or 8, ni > 255)


def matmul_nt(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x @ w[N, K]^T: the split-K GEMM or one round of tiles where they are the faster ones, else ``torch.matmul``."""
    xs = x.shape
    if len(xs) == 2:                               # (short prompts wait for the host)
        S = split_slices(x, w) if xs[1] >= SPLIT_FEW_K else 0
        if S:
            return split_linear(x, w, S)
        ni = (tile_ok(x, w) if xs[0] * w.shape[0] >= FEW_MIN_MN or w.shape[0] >= FEW_MIN_N
              or xs[1] <= SHORT_MAX_K and THIN_MAX_M < xs[0] and xs[0] * xs[1] <= SHORT_MK else 0)
        if ni:
            return tile_linear(x, w, ni)
    return torch.matmul(x, w.t())


def _mm_into(x: torch.Tensor, w: torch.Tensor, y: torch.Tensor) -> None:
    """y = x @ w^T into a column view of operands that ``_split_plan`` has let pass."""
    ni = tile_ok(x, w)
    if ni and y.stride(0) % 4 == 0 and y.data_ptr() % 8 == 0:
        native().tile_gemm(x, w, ni & 15, None, y, ni >> 4 & 15 or 8, ni > 255)
    else:
        torch.mm(x, w.t(), out=y)


def _bias_ok(bias: torch.Tensor, x: torch.Tensor, w: torch.Tensor) -> bool:
    return row_bias_ok(bias, x, w.shape[0]) and _plain(bias) and bias.data_ptr() % 8 == 0


def project(x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``F.linear`` of a served stack: few rows on the weight-streaming kernels (thin GEMM; GEMV for
    one row of a large matrix), the library otherwise."""
    xs = x.shape
    if len(xs) == 2 and xs[0] > THIN_MAX_M:            # (first: short prompts are bound by the host)
        (M, K), N = xs, w.shape[0]
        many = M * N >= FEW_MIN_MN or N >= FEW_MIN_N or K <= SHORT_MAX_K and M * K <= SHORT_MK
        if bias is None and (many or K >= SPLIT_MIN_K or K >= SPLIT_FEW_K and M * K <= 2 * SHORT_MK) and x.is_cuda:
            return mm_nt(x, w)
        ni = tile_ok(x, w) if many and bias is not None and _bias_ok(bias, x, w) else 0
        return tile_linear(x, w, ni, bias) if ni else F.linear(x, w, bias)
    if len(xs) == 2 and xs[0] >= FEW_MIN_M:            # (as in ``linear_nt``)
        S = _slices(x, w) if bias is None and xs[1] >= SPLIT_FEW_K else 0
        if S:
            return split_linear(x, w, S)
        ni = tile_ok(x, w) if w.shape[0] >= FEW_MIN_N and (bias is None or _bias_ok(bias, x, w)) else 0
        if ni:
            return tile_linear(x, w, ni, bias)
    if thin_ok(x, w) and (bias is None or row_bias_ok(bias, x, w.shape[0]) and _plain(bias)):
        return _thin(x, w, bias)
    if bias is None and len(xs) == 2 and xs[0] == 1 and _plain(x, w) and _here(x) and skinny_ok(x, w):
        y = torch.empty(1, w.shape[0], device=x.device, dtype=x.dtype)
        native().skinny_gemm(x, w, y)
        return y
    return F.linear(x, w, bias)


def _thin_tail(x, w, tanh_from: int = 1 << 30, cache=None, cache_from: int = 0, slots=None) -> torch.Tensor:
    from ._seqmix import DT, call, use_seqmix

    use_seqmix(x)
    (M, K), N = x.shape, w.shape[0]
    y = torch.empty((M, N), device=x.device, dtype=x.dtype)
    call("sm_thin_tail", DT[x.dtype], x, x.stride(0), w, y, M, N, K, tanh_from, cache,
         N - cache_from if cache is not None else 0, cache_from, slots)
    return y


def project_tanh(x: torch.Tensor, w: torch.Tensor, start: int = 0) -> tuple:
    """x @ w^T and the tanh of its columns from ``start`` on: (the columns before, which are left as they are and are
    only valid there; the tanh's) as views or tensors of their own.  Few rows form it in the epilogue, from the fp32 sums."""
    if 0 <= start < w.shape[0] and thin_ok(x, w):
        y = _thin_tail(x, w, tanh_from=start)
        return y[:, :start], y[:, start:]
    y = project(x, w)
    return y[:, :start], torch.tanh(y[:, start:])


def project_write_keys(x: torch.Tensor, w: torch.Tensor, cache: torch.Tensor, slots: torch.Tensor,
                       start: int) -> torch.Tensor:
    """x @ w^T, whose columns from ``start`` on also go to the rows ``slots`` (-1: none) of the paged key cache
    [blocks, block, heads, dim] (``write_key_cache``); few rows do so in the epilogue."""
    from .attention import write_key_cache

    GD = cache.shape[2] * cache.shape[3]
    if (thin_ok(x, w) and start % 4 == 0 and 0 <= start and w.shape[0] - start == GD and GD % 4 == 0
            and cache.is_contiguous() and cache.dtype == x.dtype and cache.device == x.device
            and slots.dtype == torch.int64 and slots.is_contiguous() and slots.numel() == x.shape[0]
            and slots.device == x.device and cache.data_ptr() % 8 == 0 and _plain(cache)):
        return _thin_tail(x, w, cache=cache, cache_from=start, slots=slots)
    y = project(x, w)
    write_key_cache(y[:, start:], cache, slots)
    return y


# Decode batches 5..256 that neither the few-row nor the tiled kernels take: the decode-batch MFMA GEMM
# (kernels/decode_gemm.hip) where the measured plan table (configs/kernels/decode_gemm_plans.json or LUMEN_DGEMM_PLANS, written
# by lumen/bench/decode_gemm_probe.py) has a (BM, BN, split-K) that beats the library's kernel, hipBLASLt with the tuned table
# otherwise (256 x 5120 x 5120: 51.2 -> 37.5 us; at the other shapes of Llama-2-7B and -13B the tiled kernels are 1.05 - 1.3 times as
# fast as its best form, or the library is).  (Two earlier hand-written attempts lost, scripts/probes/: 32-row M tiles, and all-M-rows tiles over
# all of K whose every workgroup pulled the whole x through its CU's load path.)
DG_BMS = (64, 128, 192, 256)
DG_BNS = {256: (64, 96, 128, 160), 192: (64, 96, 128), 128: (64, 96, 128, 192, 256),
          64: (64, 128, 192, 256)}
DG_BNS8 = {256: (64, 128), 128: (128, 256)}   # 8-wave variants
DGEMM = os.environ.get("LUMEN_DGEMM", "1") != "0"
_dg_ws: dict = {}
_dg_old: list = []
_dg_plans: Optional[dict] = None


def dg_bucket(M: int) -> int:
    return next(b for b in DG_BMS if M <= b)


def decode_gemm(x: torch.Tensor, w: torch.Tensor, bm: int, bn: int, s: int, nw: int = 4,
                out: Optional[torch.Tensor] = None, flags: int = 0,
                m: Optional[int] = None) -> torch.Tensor:
    """y = x @ w^T on the decode-batch MFMA kernel with block tile (bm, bn), split-K s and nw
    (4 or 8) waves per block.  ``flags``: bit 0 rotates each tile's k loop start; bit 1 takes
    x in the k-tiled layout [K / 64, bm, 64] (``x_ktiled``) with ``m`` valid rows."""
    rows = x.shape[0] if not flags & 2 else int(m)
    y = out if out is not None else torch.empty(rows, w.shape[0], device=x.device, dtype=x.dtype)
    ws = cnt = None
    if s > 1:
        # one slab workspace + ticket counters per (device, stream): split-K slabs and tickets
        # of GEMMs on different streams never interleave (a side-stream GEMM gets its own)
        key = _dg_key(x.device)
        got = _dg_ws.get(key)
        need = -(-w.shape[0] // bn) * s * bm * bn
        if got is None or got[0].numel() < need or got[1].numel() < -(-w.shape[0] // bn):
            # generous size; a superseded pair stays alive (_dg_old): a captured decode graph
            # keeps pointing at the buffers it was captured with
            n = max(need, 1 << 24)
            if got is not None:
                _dg_old.append(got)
            got = (torch.empty(n, dtype=torch.float32, device=x.device),
                   torch.zeros(max(4096, -(-w.shape[0] // bn)), dtype=torch.int32,
                               device=x.device))
            _dg_ws[key] = got
        ws, cnt = got
    native().decode_gemm(x, w, y, ws, cnt, bm, bn, s, nw, flags)
    return y


def x_ktiled(x: torch.Tensor, bm: int = 256) -> torch.Tensor:
    """[M, K] -> [K / 64, bm, 64] (rows past M zero): the decode GEMM's k-tiled x layout."""
    M, K = x.shape
    t = torch.zeros(K // 64, bm, 64, device=x.device, dtype=x.dtype)
    t[:, :M].copy_(x.reshape(M, K // 64, 64).transpose(0, 1))
    return t


def _dg_key(device) -> tuple:
    return (str(device), torch.cuda.current_stream(device).cuda_stream)


def dg_workspace(device) -> Optional[tuple]:
    """(slab workspace, ticket counters) of the current stream on ``device`` (None before the
    first split-K call there)."""
    return _dg_ws.get(_dg_key(device))


def dg_plans() -> dict:
    """{(N, K, BM): (BN, S, waves)} from configs/kernels/decode_gemm_plans.json (measured wins only)."""
    global _dg_plans
    if _dg_plans is None:
        import json

        path = os.environ.get("LUMEN_DGEMM_PLANS", os.path.join(
            os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__)))),
            "configs", "kernels", "decode_gemm_plans.json"))
        _dg_plans = {}
        if os.path.exists(path):
            with open(path) as f:
                for e in json.load(f).get("plans", []):
                    _dg_plans[(e["N"], e["K"], e["BM"])] = (e["BN"], e["S"], e.get("NW", 4))
    return _dg_plans


def dg_plan(x: torch.Tensor, w: torch.Tensor) -> Optional[tuple]:
    if not DGEMM or x.dim() != 2 or w.dim() != 2 or not 4 < x.shape[0] <= DG_BMS[-1] or not x.is_cuda:
        return None
    bm = dg_bucket(x.shape[0])
    p = dg_plans().get((w.shape[0], w.shape[1], bm))   # (most shapes have none: asked first)
    if p is None:
        return None
    if not (use_native(x) and x.dtype == w.dtype and x.dtype in (torch.bfloat16, torch.float16)
            and x.stride(1) == 1 and x.stride(0) % 8 == 0 and w.is_contiguous()
            and x.shape[1] == w.shape[1] and w.shape[1] % 64 == 0 and w.shape[0] % 4 == 0):
        return None
    return (bm,) + tuple(p)


# Training-shape GEMMs run 256 x 256 macro tiles, one per CU at a time, so a GEMM with 5.375 or
# 2.69 waves of tiles on the 256-CU chip takes 6 or 3 waves (Llama-2-7B at T = 4096: gate|up
# forward 16 x 86 tiles, down input-grad 16 x 43).  ``mm_nt`` splits the output columns at the
# last whole wave and runs the remainder as its own (separately tuned) GEMM, both writing column
# views of one buffer (ldc = full width, no copies).  scripts/probes/split_gemm_probe.py measures it.
GEMM_SPLIT = os.environ.get("LUMEN_GEMM_SPLIT", "1") != "0"
SPLIT_TILE, SPLIT_CUS = 256, 256
SPLIT_MAX_TAIL = float(os.environ.get("LUMEN_GEMM_SPLIT_MAX_TAIL", "0.75"))


def split_cols(M: int, N: int) -> int:
    """Column count of the whole-wave part of an [M, N] output (0: no split).  Splits only when
    the last wave is at most ``SPLIT_MAX_TAIL`` full and the wave boundary is a column-tile
    boundary."""
    if M % SPLIT_TILE or N % 8:
        return 0
    tm, tn = M // SPLIT_TILE, -(-N // SPLIT_TILE)
    total = tm * tn
    waves, tail = divmod(total, SPLIT_CUS)
    if waves == 0 or tail == 0 or tail > SPLIT_MAX_TAIL * SPLIT_CUS or SPLIT_CUS % tm:
        return 0
    n1 = waves * (SPLIT_CUS // tm) * SPLIT_TILE
    return n1 if 0 < n1 < N else 0


# A shape that the tuned table does not hold takes the library's own choice, a 256 x 256 stream-K kernel that
# pays for an unfilled last wave with more than the wave (0.9 - 1.25 PFLOP/s against 1.45 on whole waves).  Cut
# after ``waves`` times as many columns of tiles as fit one wave, from two waves on, us: 4010 x 22016 x 4096
# 637 -> 490, x 11008 407 -> 266, 4010 x 11264 x 2048 162 -> 141, 1300 x 22016 x 4096 299 -> 207, 300 x 95744 x
# 4096 325 -> 238, 8000 x 11008 x 4096 627 -> 477.  Taking the columns that fill the waves nearest instead
# (39 of 43 at 3100 rows x 11008: 507 of 512 tiles) sends the main part back to stream-K: 354 -> 369, with 38
# columns 218.  With one whole wave it is even (2305 x 12288 173 -> 172): left whole here.
# Where the row tiles do not divide 256, every wave of the main part leaves 256 mod tm tiles to the rest.  Up to 8
# waves that costs less than stream-K does even when the rest passes one wave (4874 x 22016: 734 -> 647, 5100 x
# 22016 x 2048 in fp16 369 -> 379); from 9 on it does not (5100 x 32000 897 -> 1032, 7300 x 25344 580 -> 644):
# left whole.  So is everything over 32 row tiles, where both forms win by turns (16000 x 25344 1252 -> 1173,
# 9500 x 12288 667 -> 732, 11000 x 12288 819 -> 1039).  Over 250 timings of cuts by this rule (300 - 8000 rows, K
# 2048 - 4096, both types) the mean is 0.90 of the whole product's time; 19 are more than 2.5 % above it,
# most of them at 1300 - 1536 rows and 2.3 - 2.9 waves (1500 x 28672 x 2048 139 -> 153, worst 116 -> 129).
WAVE_MIN, WAVE_MIN_K = 2, 2048
WAVE_MIN_M, WAVE_MAX_TM, WAVE_SPILL_MAX = 300, 32, 8
MIN_CUT = 1 << 24         # fewer elements than any cut product has


def wave_cols(M: int, N: int, K: int) -> int:
    """Column count of the whole waves of 256 x 256 tiles of an [M, N] output with any M (0: no cut)."""
    tm, tn = -(-M // SPLIT_TILE), -(-N // SPLIT_TILE)
    if M < WAVE_MIN_M or tm > WAVE_MAX_TM or N % 8 or K < WAVE_MIN_K:
        return 0
    waves, tail = divmod(tm * tn, SPLIT_CUS)
    n1 = waves * (SPLIT_CUS // tm) * SPLIT_TILE
    if waves < WAVE_MIN or not tail or not 0 < n1 < N:
        return 0
    rest = tail + waves * (SPLIT_CUS % tm)
    return n1 if waves <= WAVE_SPILL_MAX or rest <= SPLIT_CUS else 0


def round_cols(M: int, N: int, K: int) -> int:
    """Column count of the one whole wave of 256 x 256 tiles in an [M, N] output whose rest is one round of narrow tiles of
    kernels/tile_gemm.hip (0: no cut).  us, whole -> cut: 2048 x 11264 x 2048 88 -> 82, 4010 x 5632 x 4096 158 -> 142, 4096 x 6144 x
    5632 215 -> 205; 43 such shapes 0.99 - 1.15 times as fast, mean 1.05.  Rests of wider tiles (ni 5 - 6): 0.94 - 1.03."""
    tm, tn = -(-M // SPLIT_TILE), -(-N // SPLIT_TILE)
    if M < WAVE_MIN_M or tm > WAVE_MAX_TM or N % 8 or K < WAVE_MIN_K or tm * tn // SPLIT_CUS != 1:
        return 0
    n1 = SPLIT_CUS // tm * SPLIT_TILE
    return n1 if n1 < N and tile_columns(M, N - n1, K) in (3, 4) else 0


_tuned: dict = {"n": -1, "sigs": {}}
_OP = {torch.bfloat16: "GemmTunableOp_BFloat16_TN", torch.float16: "GemmTunableOp_Half_TN"}


def _tuned_sigs(dtype: torch.dtype) -> frozenset:
    """Problem signatures that the loaded TunableOp table holds for x @ w^T in ``dtype`` (read again when
    the table's size changes)."""
    try:
        import torch.cuda.tunable as tn

        if not tn.is_enabled():
            return frozenset()
        res = tn.get_results()
    except Exception:  # noqa: BLE001
        return frozenset()
    if len(res) != _tuned["n"]:
        _tuned["sigs"] = {dt: frozenset(r[1] for r in res if r[0] == op) for dt, op in _OP.items()}
        _tuned["n"] = len(res)                     # (last: another thread may ask in between)
    return _tuned["sigs"][dtype]


def _tuning() -> bool:
    """Is TunableOp timing solutions?  Its rotating copies of C start at the column view's address and
    would read past the buffer's end (utils/gemm_tuning.py): then no untuned product is cut."""
    import torch.cuda.tunable as tn

    return tn.is_enabled() and tn.tuning_is_enabled()


def _split_plan(x: torch.Tensor, w: torch.Tensor) -> int:
    xs, ws = x.shape, w.shape
    if len(xs) != 2 or len(ws) != 2 or xs[0] * ws[0] < MIN_CUT:
        return 0                                   # (nearly every call: as little host time as can be)
    if not (GEMM_SPLIT and x.is_cuda and x.dtype in _OP and x.dtype == w.dtype and x.stride(1) == 1
            and w.stride(1) == 1):
        return 0
    (M, K), N = xs, ws[0]
    n1, n2 = split_cols(M, N), wave_cols(M, N, K) or round_cols(M, N, K)
    if not (n1 or n2):
        return 0
    # the first where both parts have tuned solutions, the second where neither the whole nor the parts
    # have; decided once per problem, type and table (utils/gemm_tuning.py forgets the plans when it loads one)
    key = (M, N, K, w.stride(0), x.stride(0), x.dtype)
    hit = _plans.get(key)
    if hit is None:
        sigs = _tuned_sigs(x.dtype)
        lds = f"ld_{w.stride(0)}_{x.stride(0)}_{N}"
        if n1 and f"tn_{n1}_{M}_{K}_{lds}" in sigs and f"tn_{N - n1}_{M}_{K}_{lds}" in sigs:
            hit = (n1, True)
        else:
            hit = (0 if f"tn_{N}_{M}_{K}_{lds}" in sigs else n2, False)
        if sigs:                                   # (no table: it may still be loaded)
            if len(_plans) >= MAX_PLANS:
                _plans.clear()
            _plans[key] = hit
    cols, tuned = hit
    return cols if cols and _plain(x, w) and (tuned or not _tuning()) else 0


_plans: dict = {}
MAX_PLANS = 4096          # (M, N, K, strides, type) -> columns; ragged prompts bring a new M each


def forget_plans() -> None:
    """The tuned table has changed: products are planned again."""
    _plans.clear()
    _tuned["n"] = -1


def mm_nt(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x [M, K] @ w[N, K]^T -> [M, N] (w row-contiguous), split at the last whole wave of tiles
    on the GPU (see ``split_cols`` and ``wave_cols``)."""
    n1 = _split_plan(x, w)
    if not n1:
        return matmul_nt(x, w)
    y = torch.empty(x.shape[0], w.shape[0], device=x.device, dtype=x.dtype)
    torch.mm(x, w[:n1].t(), out=y[:, :n1])
    _mm_into(x, w[n1:], y[:, n1:])
    return y


def linear_nt(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x [M, K] @ w[N, K]^T -> [M, N]; operands of other dimensions as ``torch.matmul`` takes them."""
    M = x.shape[0]
    if x.dim() == 2 and FEW_MIN_M <= M <= SPLIT_FEW_M:     # (before the planned shapes: 128 x 4096 x 11008 38 -> 28 us)
        S = _slices(x, w) if x.shape[1] >= SPLIT_FEW_K else 0
        if S:
            return split_linear(x, w, S)
        ni = tile_ok(x, w) if w.shape[0] >= FEW_MIN_N else 0
        if ni:
            return tile_linear(x, w, ni)
    if M <= THIN_MAX_M:
        if thin_ok(x, w) and use_native(x):
            return _thin(x, w)
        if skinny_ok(x, w):
            y = torch.empty(x.shape[0], w.shape[0], device=x.device, dtype=x.dtype)
            native().skinny_gemm(x, w, y)
            return y
    p = dg_plan(x, w) if M <= DG_BMS[-1] else None
    if p is not None:
        return decode_gemm(x, w, *p)
    # prefill / mixed steps (M = 2048-4096 tokens): the whole-wave column split where both
    # parts are tuned, as in training (profiles/r5_serve_split)
    return mm_nt(x, w)


# batch <= 4 decode, opt-in (LUMEN_SWIGLU_GEMV=1): SwiGLU formed inside the rows-per-lane weight
# stream, one launch fewer per layer.  Measured slower both ways: the row-group GEMV form 21.4 vs
# 18.5 us per call, the rows-per-lane form 3.085 vs 2.99-3.01 ms per batch-1 decode step
# -- every workgroup re-reads and re-activates the whole 2 x 11008 gate|up row
SWIGLU_GEMV = os.environ.get("LUMEN_SWIGLU_GEMV", "0") == "1"


def swiglu_linear_nt(gu: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """(silu(gu[:, :F]) * gu[:, F:]) @ w[N, F]^T, the MLP down projection."""
    from .activation import swiglu

    M, F = gu.shape[0], gu.shape[1] // 2
    if (SWIGLU_GEMV and 0 < M <= 4 and gu.dim() == 2 and gu.shape[1] == 2 * F
            and gu.stride(1) == 1 and gu.stride(0) % 8 == 0 and use_native(gu)
            and w.dim() == 2 and w.shape[1] == F and w.is_contiguous() and gu.dtype == w.dtype
            and gu.dtype in (torch.bfloat16, torch.float16) and w.shape[0] % 4 == 0
            and F % 8 == 0 and skinny_ok(gu[:, :F], w)):
        y = torch.empty(M, w.shape[0], device=gu.device, dtype=gu.dtype)
        native().skinny_swiglu_gemm(gu, w, y)
        return y
    return linear_nt(swiglu(gu), w)
