"""Mixture-of-experts routing and gated activations (HIP: ``csrc/seqmix/moe.hip``).

Two ways to run a layer's experts, both on library GEMMs over weights stacked once at load (the
gate|up rows of every expert and of the shared expert in one [E * 2ff + 2ffs, W] weight, the down
projections side by side in one [W, E * ff + ffs] weight):

* ``moe_dense``: TWO GEMMs over all tokens and all experts.  Between them ``gated_act``
  multiplies each expert's activation by the token's routing weight (zero for experts the token
  did not choose), so the second GEMM's reduction over [experts x ff] IS the weighted sum of the
  chosen experts -- no gather / scatter, no host-visible token counts, graph-capturable.  Decode
  steps use it: at a few rows per step the cost is reading the expert weights, which a batch
  touches almost all of anyway.
* ``moe_grouped``: tokens sorted by expert, one pair of GEMMs per expert on its rows (slices of
  the same stacked weights), weighted rows added back in fp32.  It does top / E of the dense
  form's expert FLOPs but needs the per-expert row counts on the host (one synchronisation), so
  it serves prefill-sized steps outside graph capture.
* ``moe_grouped_mm``: the same arithmetic on the library's grouped GEMM (16-bit dtypes): the
  sorted (row, expert) pairs have a static count, the group offsets stay on the device, nothing
  synchronises and a layer's experts are three launches.
* ``moe_chosen``: the (row, expert) pairs sorted by expert on the device, both products on HIP kernels
  (``csrc/seqmix/expert_gemm.hip``) that gather the rows themselves.  16-bit steps of more than a few rows take it
  (``chosen_pays``), decode graphs included; the other forms serve fp32, sizes without kernels and the few-row steps.
"""
from __future__ import annotations

from dataclasses import dataclass
from typing import Optional, Union

import torch
import torch.nn.functional as F

from .gemm import (MID_MAX_M, THIN_BATCH_MAX_W, THIN_MAX_K, THIN_MAX_M, _here, _plain, _thin, few_tiles, mid_ok, project, row_bias_ok,
                   thin_ok, weights_ok)


def route_topk_ref(z: torch.Tensor, top: int) -> torch.Tensor:
    val, idx = torch.sort(z.float(), dim=-1, descending=True, stable=True)  # ties: lowest index
    val, idx = val[:, :top], idx[:, :top]
    return torch.zeros_like(z, dtype=torch.float32).scatter_(1, idx, torch.softmax(val, -1))


def route_topk(z: torch.Tensor, top: int) -> torch.Tensor:
    """Router logits z [T, E] (fp32) -> dense routing weights [T, E] (fp32): the softmax over
    each row's ``top`` largest logits at their places, zero elsewhere (ties: lowest index)."""
    from ._seqmix import call, use_seqmix

    if not use_seqmix(z):
        return route_topk_ref(z, top)
    assert z.dtype == torch.float32 and z.is_contiguous()
    T, E = z.shape
    if E > 1024:
        raise ValueError(f"route_topk supports at most 1024 experts, got {E}")
    out = torch.empty_like(z)
    call("sm_route_topk", z, out, T, E, top)
    return out


def router_logits(h: torch.Tensor, w: torch.Tensor,
                  bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """fp32 router logits h [T, W] @ w [E, W]^T (+ ``bias`` [E]) for operands in the model dtype.
    16-bit values multiply exactly in fp32, so on the GPU the product runs on the matrix cores with
    fp32 accumulation and an fp32 result -- the arithmetic of an fp32 GEMM on the widened operands
    without the pass that widens them."""
    if thin_ok(h, w, gemv=False) and (bias is None or row_bias_ok(bias, h, w.shape[0])
                                      and _plain(bias)):
        return _thin(h, w, bias, torch.float32)
    if h.is_cuda and h.dtype == w.dtype and h.dtype in (torch.bfloat16, torch.float16):
        z = torch.mm(h, w.t(), out_dtype=torch.float32)
    else:
        z = h.float() @ w.float().t()
    return z if bias is None else z.add_(bias)


def route_groups_ref(z, correction, top, n_groups, keep, scale, sum_eps=1e-20, rank_top=2,
                     score="sigmoid", normalize=True):
    T, E = z.shape
    s = torch.softmax(z.float(), -1) if score == "softmax" else torch.sigmoid(z.float())
    c = s + correction.float() if correction is not None else s
    if n_groups > 1 and keep < n_groups:
        per = E // n_groups
        cg = c.view(T, n_groups, per)
        rank = torch.sort(cg, dim=-1, descending=True).values[..., :min(rank_top, per)].sum(-1)
        best = torch.sort(rank, dim=-1, descending=True, stable=True).indices[:, :keep]
        allow = torch.zeros(T, n_groups, dtype=torch.bool, device=z.device).scatter_(1, best, True)
        c = cg.masked_fill(~allow.view(T, n_groups, 1), float("-inf")).reshape(T, E)
    idx = torch.sort(c, dim=-1, descending=True, stable=True).indices[:, :top]
    chosen = torch.gather(s, 1, idx)
    wt = (chosen / (chosen.sum(-1, keepdim=True) + sum_eps) if normalize else chosen) * scale
    return torch.zeros_like(s).scatter_(1, idx, wt)


def route_groups(z: torch.Tensor, correction: Optional[torch.Tensor], top: int, n_groups: int,
                 keep: int, scale: float = 1.0, sum_eps: float = 1e-20, rank_top: int = 2,
                 score: str = "sigmoid", normalize: bool = True) -> torch.Tensor:
    """Router logits z [T, E] (fp32) -> dense routing weights [T, E] (fp32) of a router with a
    choice correction and a limit to the best groups: the scores are s = sigmoid(z), or with
    ``score`` = "softmax" the softmax of z over all experts; the
    choice ranks c = s + ``correction`` [E] (None: c = s); the experts form ``n_groups`` equal groups of
    neighbours, a group ranks by the sum of its ``rank_top`` largest c, and only experts of the
    ``keep`` best groups can be chosen (``keep`` = ``n_groups``: no limit); the ``top`` eligible
    experts with the largest c get s_e / (sum of the chosen s + ``sum_eps``) * ``scale`` at their
    places (``normalize`` False: s_e * ``scale``, the scores as they are), all others zero.  Ties
    go to the lowest index.  ``rank_top`` = 1 ranks a group by its best member."""
    from ._seqmix import call, use_seqmix

    T, E = z.shape
    if n_groups < 1 or E % n_groups or not 1 <= keep <= n_groups:
        raise ValueError(f"{E} experts do not form {n_groups} equal groups of which {keep} are kept")
    if not 1 <= top <= keep * (E // n_groups):
        raise ValueError(f"top {top} exceeds the {keep * (E // n_groups)} eligible experts")
    if score not in ("sigmoid", "softmax"):
        raise ValueError(f"unknown router score {score!r}")
    if not use_seqmix(z):
        return route_groups_ref(z, correction, top, n_groups, keep, scale, sum_eps, rank_top,
                                score, normalize)
    assert z.dtype == torch.float32 and z.is_contiguous()
    assert correction is None or (correction.dtype == torch.float32 and correction.is_contiguous())
    if E > 1024:
        raise ValueError(f"route_groups supports at most 1024 experts, got {E}")
    out = torch.empty_like(z)
    call("sm_route_groups", z, correction, out, T, E, top, n_groups, keep, rank_top, scale, sum_eps,
         int(score == "softmax"), int(bool(normalize)))
    return out


# Few rows: the norm before the experts, the router's product and the routing in one launch (seqmix/route_rows.hip, a
# workgroup per row, which reads the router for itself; more rows or experts are better off with the product on
# matrix cores).
ROUTE_MAX_M, ROUTE_MAX_E, ROUTE_MAX_W = 64, 64, 8192


def _route_rows_pay(rows: int, W: int, E: int, normed: bool) -> bool:
    """A workgroup reads the whole router, and few rows have few workgroups: a large one is better read by the thin GEMM
    (us, separate launches and one, 1 / 16 / 32 / 64 rows.  Given rows, experts x width: 64 x 2048 7.6 and 7.8, 8.1 and 8.0, -, 10.5
    and 8.1; 64 x 3072 8.4 and 10.4, 8.8 and 10.8, 9.9 and 10.7, 12.2 and 10.8; 64 x 8192 10.3 and 16.3, 12.7 and 17.1, -, 21.1 and 17.1; 48 x
    4096 9.2 and 9.5, 9.5 and 9.9, 11.0 and 9.8, 13.9 and 9.9; 32 x 6144 9.2 and 10.4, 11.2 and 10.8, 13.4 and 10.8, 17.5 and 10.8.
    With the norm: 64 x 4096 13.1 and 12.0 for one; 64 x 8192 15.3 and 17.8, -, 21.5 and 18.8)."""
    if normed:
        return E * W <= 1 << 18 or rows >= E // 2
    return E * W < 3 << 16 or rows >= E - 16


def _route_rows_ok(h: torch.Tensor, router: torch.Tensor, bias, correction, top: int, groups: int, keep: int,
                   rank_top: int, normed: bool = False) -> bool:
    """``h``: the normed rows, or (``normed``: the launch norms) the sublayer's output that the stream takes first."""
    if h.dim() != 2 or not 0 < h.shape[0] <= ROUTE_MAX_M or not h.is_cuda or router.dim() != 2:
        return False
    (E, W), dt = router.shape, h.dtype
    if (W != h.shape[1] or W % 8 or not 0 < W <= ROUTE_MAX_W or not 0 < E <= ROUTE_MAX_E or dt != router.dtype
            or dt not in (torch.bfloat16, torch.float16) or router.device != h.device or not router.is_contiguous()
            or not _route_rows_pay(h.shape[0], W, E, normed)
            or not row_bias_ok(bias, h, E) or not _plain(h, router) or not _here(h)):
        return False
    if bias is not None and not _plain(bias) or correction is not None and not (
            correction.dtype == torch.float32 and correction.is_contiguous() and correction.numel() == E
            and correction.device == h.device and _plain(correction)):
        return False
    if groups and (E % groups or not 1 <= keep <= groups or top > keep * (E // groups) or not 1 <= rank_top <= 4):
        return False
    return (1 <= top <= E and h.stride(1) == 1 and h.stride(0) % 8 == 0 and h.stride(0) >= W
            and (h.data_ptr() | router.data_ptr()) % 16 == 0)


def _stream_ok(x: torch.Tensor, y: torch.Tensor, rows: tuple, ones: tuple = ()) -> bool:
    """Can the fused form take ``y`` into the fp32 stream ``x``, with norms' ``rows`` of [W] and single values?"""
    if not (x.dtype == torch.float32 and x.shape == y.shape and x.is_contiguous() and y.is_contiguous()
            and x.device == y.device and x.data_ptr() % 16 == 0 and _plain(x)):
        return False
    return (all(t.dtype == torch.float32 and t.device == x.device and _plain(t) for t in rows + ones)
            and all(t.is_contiguous() and t.numel() == x.shape[1] and t.data_ptr() % 16 == 0 for t in rows)
            and all(t.numel() == 1 for t in ones))


def _route_rows(kind, x, y, h, norm, post, eps, router, bias, top, groups=0, keep=0, rank_top=1, softmax=False,
                normalize=True, scale=1.0, sum_eps=0.0, correction=None) -> torch.Tensor:
    from ._seqmix import DT, call, use_seqmix

    use_seqmix(h)
    T, W = h.shape
    E = router.shape[0]
    out = torch.empty(T, E, dtype=torch.float32, device=h.device)
    call("sm_route_rows", DT[h.dtype], kind, x, y, h, h.stride(0), *norm, *post, router, bias, out, T, W, E, eps, top,
         groups, keep, rank_top, int(softmax), int(bool(normalize)), scale, sum_eps, correction)
    return out


_NONE3 = (None, None, None)


def routed_groups(h: torch.Tensor, router: torch.Tensor, correction: Optional[torch.Tensor], top: int, n_groups: int,
                  keep: int, scale: float = 1.0, sum_eps: float = 1e-20, rank_top: int = 2,
                  score: str = "sigmoid", normalize: bool = True) -> torch.Tensor:
    """``route_groups`` of ``router_logits``."""
    if score in ("sigmoid", "softmax") and _route_rows_ok(h, router, None, correction, top, n_groups, keep, rank_top):
        return _route_rows(0, None, None, h, _NONE3, _NONE3, 0.0, router, None, top, n_groups, keep, rank_top,
                           score == "softmax", normalize, scale, sum_eps, correction)
    return route_groups(router_logits(h, router), correction, top, n_groups, keep, scale, sum_eps, rank_top, score,
                        normalize)


def residual_rms_routed(x: torch.Tensor, y: torch.Tensor, w: torch.Tensor, eps: float, router: torch.Tensor, top: int,
                        normalize: bool = True) -> tuple:
    """``residual_rms`` into the experts' input h, and its routing by sigmoid scores (``route_groups`` of one
    group): (h, weights)."""
    from .norm import residual_rms

    if _route_rows_ok(y, router, None, None, top, 1, 1, 1, True) and _stream_ok(x, y, (w,)):
        h = torch.empty_like(y)
        return h, _route_rows(1, x, y, h, (w, None, None), _NONE3, eps, router, None, top, 1, 1, 1, False, normalize,
                              1.0, 1e-20)
    h = residual_rms(x, y, w, eps)
    return h, route_groups(router_logits(h, router), None, top, 1, 1, normalize=normalize)


def dyt_residual_routed(x: torch.Tensor, y: torch.Tensor, post, pre, router: torch.Tensor,
                        bias: Optional[torch.Tensor], top: int, dtype: torch.dtype) -> tuple:
    """``dyt_residual`` into the experts' input h, and its routing over the ``top`` logits: (x, h, weights)."""
    from .norm import dyt_residual

    if y.dtype == dtype and _route_rows_ok(y, router, bias, None, top, 0, 0, 1, True) \
            and _stream_ok(x, y, (*post[:2], *pre[:2]), (post[2], pre[2])):
        h = torch.empty_like(y)
        return x, h, _route_rows(2, x, y, h, pre, post, 0.0, router, bias, top)
    x, h = dyt_residual(x, y, post, pre, dtype)
    return x, h, route_topk(router_logits(h, router, bias), top)


GATE_ACTS = {"silu": 0, "relu": 1, "gelu_tanh": 2, "relu2": 3}
_ACT_FN = {"silu": F.silu, "relu": F.relu, "gelu_tanh": lambda z: F.gelu(z, approximate="tanh"),
           "relu2": lambda z: F.relu(z) ** 2}


@dataclass(frozen=True)
class ClampedGate:
    """The gated activation g * sigmoid(slope * g) * (u + shift) with g = min(gate, limit) and
    u = clamp(up, -limit, limit); the unweighted block (the shared expert) has ``limit_shared``."""
    limit: float
    limit_shared: float
    slope: float = 1.0
    shift: float = 0.0


def gated_act_ref(gu, wts, E, ff, ffs, act="silu", weigh="output"):
    T = gu.shape[0]

    def pair(g, u, limit):
        if isinstance(act, str):
            return _ACT_FN[act](g) * u
        g, u = torch.clamp(g, max=limit), torch.clamp(u, min=-limit, max=limit)
        return g * torch.sigmoid(act.slope * g) * (u + act.shift)

    lim, lim_s = (0.0, 0.0) if isinstance(act, str) else (act.limit, act.limit_shared)
    parts = []
    if E:
        g = gu[:, :E * 2 * ff].float().view(T, E, 2, ff)
        wt = wts.float()[:, :, None]
        y = (pair(g[:, :, 0] * wt, g[:, :, 1] * wt, lim) if weigh == "input"
             else pair(g[:, :, 0], g[:, :, 1], lim) * wt)
        parts.append(y.reshape(T, E * ff))
    if ffs:
        s = gu[:, E * 2 * ff:].float().view(T, 2, ffs)
        parts.append(pair(s[:, 0], s[:, 1], lim_s))
    return torch.cat(parts, 1).to(gu.dtype)


def gated_act(gu: torch.Tensor, wts: Optional[torch.Tensor], E: int, ff: int,
              ffs: int, act: Union[str, ClampedGate] = "silu",
              weigh: str = "output") -> torch.Tensor:
    """act(gate) * up over stacked [gate | up] blocks (``act``: silu, i.e. SwiGLU, relu or
    gelu_tanh, or a ``ClampedGate``): ``gu`` [T, E * 2 * ff + 2 * ffs] holds E expert blocks (gate
    rows then up rows, ff each) and one unweighted block of ffs (a dense feed-forward, or the
    shared expert); expert e's activation is scaled by ``wts[:, e]``, or with ``weigh`` = "input"
    its gate and up values are (they are linear in the expert's input, so this is the expert of the
    weighted input).  Returns [T, E * ff + ffs]."""
    from ._seqmix import DT, call, use_seqmix

    if weigh not in ("output", "input"):
        raise ValueError(f"unknown place of the routing weight {weigh!r}")
    if not use_seqmix(gu):
        return gated_act_ref(gu, wts, E, ff, ffs, act, weigh)
    assert gu.is_contiguous() and gu.shape[1] == E * 2 * ff + 2 * ffs
    out = torch.empty(gu.shape[0], E * ff + ffs, dtype=gu.dtype, device=gu.device)
    code, c = (GATE_ACTS[act], (0.0,) * 4) if isinstance(act, str) else (
        4, (act.limit, act.limit_shared, act.slope, act.shift))
    call("sm_gated_act", DT[gu.dtype], gu, wts, out, gu.shape[0], E, ff, ffs, code,
         int(weigh == "input"), *c)
    return out


def scaled_act_ref(u, wts, E, ff, ffs, act="relu2"):
    T = u.shape[0]
    fn = _ACT_FN[act]
    parts = []
    if E:
        parts.append((fn(u[:, :E * ff].float()).view(T, E, ff) * wts.float()[:, :, None])
                     .reshape(T, E * ff))
    if ffs:
        parts.append(fn(u[:, E * ff:].float()))
    return torch.cat(parts, 1).to(u.dtype)


def scaled_act(u: torch.Tensor, wts: Optional[torch.Tensor], E: int, ff: int, ffs: int,
               act: str = "relu2") -> torch.Tensor:
    """act(u) over the stacked up projections of experts WITHOUT a gate (``act``: as for
    ``gated_act``, plus relu2 = relu(.)^2): ``u`` [T, E * ff + ffs] holds E expert blocks of ff and
    one unweighted block of ffs; expert e's activation is scaled by ``wts[:, e]``.  Same shape
    out."""
    from ._seqmix import DT, call, use_seqmix

    if not use_seqmix(u):
        return scaled_act_ref(u, wts, E, ff, ffs, act)
    assert u.is_contiguous() and u.shape[1] == E * ff + ffs
    out = torch.empty_like(u)
    call("sm_scaled_act", DT[u.dtype], u, wts, out, u.shape[0], E, ff, ffs, GATE_ACTS[act])
    return out


def _act(z, wts, E, ff, ffs, act, gated, weigh):
    if gated:
        return gated_act(z, wts, E, ff, ffs, act, weigh)
    if weigh != "output":
        raise ValueError("experts without a gate take their weight on the output")
    return scaled_act(z, wts, E, ff, ffs, act)


# Few-row steps: the first projection forms the activation in its epilogue (seqmix/thin_gemm.hip), one
# launch and the [T, 2 ff] intermediate less.  ``top`` known and T * top <= SPARSE_ROWS * E: a row's experts
# are few enough that reading the chosen ones only pays (uniform choices leave exp(-T top / E) of them out:
# 5 % at 3, about the cost of reading the routing weights first).
THIN_ACT_MAX_M, THIN_ACT_MAX_WTS, THIN_ACT_MAX_E = 32, 2048, 64
SPARSE_ROWS = 3


def thin_act_ok(h, wts, gu_w, E: int, ff: int, ffs: int, act="silu", gated: bool = True,
                weigh: str = "output", sparse: bool = False) -> bool:
    """Can and should ``thin_act`` run the first projection and the activation in one kernel?  ``sparse``:
    it would read the chosen experts only."""
    if not (h.dim() == 2 and 0 < h.shape[0] <= THIN_ACT_MAX_M and h.is_cuda and ff % 16 == 0
            and ffs % 16 == 0 and 0 < E * ff + ffs < THIN_MAX_K and E <= THIN_ACT_MAX_E
            and h.shape[0] * E <= THIN_ACT_MAX_WTS and (gated or isinstance(act, str))
            and (E == 0 or weights_ok(wts, h, E) and _plain(wts))):
        return False
    k = 2 if gated else 1
    if gu_w.shape[0] != k * (E * ff + ffs) or (weigh == "input" and not gated):
        return False
    # thin_ok also says whether the thin kernel beats the library on a huge matrix, which a stack of experts
    # is not a case of (16 rows of it stand for the strides), and for one row the GEMV on a long K.  The GEMV
    # reads every expert: skipping wins at any width (one row, both projections, us: width 4096, 16 experts
    # of 2816, top 3, and a shared one 174 -> 57, of 1408 94 -> 36; 4 of 1024, top 2 28 -> 20; ungated 120 -> 49).
    return thin_ok(h, gu_w[:16] if E else gu_w, gemv=not sparse)


def thin_act(h, gu_w, wts, E: int, ff: int, ffs: int, act="silu", gated: bool = True,
             weigh: str = "output", sparse: bool = False) -> torch.Tensor:
    """``gated_act`` (or ``scaled_act``) of h @ gu_w^T, [T, E * ff + ffs], from the fp32 sums.
    ``sparse``: the blocks of experts that no row chose are left unwritten."""
    if weigh not in ("output", "input"):
        raise ValueError(f"unknown place of the routing weight {weigh!r}")
    if h.dim() != 2 or h.stride(1) != 1 or not gu_w.is_contiguous() or gu_w.dtype != h.dtype \
            or gu_w.device != h.device or (E and not weights_ok(wts, h, E)) \
            or tuple(gu_w.shape) != ((2 if gated else 1) * (E * ff + ffs), h.shape[1]):
        raise ValueError("few-row experts: rows h, stacked weights and routing weights do not fit")
    return _thin_act(h, gu_w, wts, E, ff, ffs, act, gated, weigh, sparse)


def _thin_act(h, gu_w, wts, E, ff, ffs, act="silu", gated=True, weigh="output", sparse=False):
    """``thin_act`` of operands that ``thin_act_ok`` has let pass."""
    from ._seqmix import DT, call, use_seqmix

    use_seqmix(h)
    M, K = h.shape
    out = torch.empty((M, E * ff + ffs), dtype=h.dtype, device=h.device)
    code, c = (GATE_ACTS[act], (0.0,) * 4) if isinstance(act, str) else (
        4, (act.limit, act.limit_shared, act.slope, act.shift))
    call("sm_thin_act", DT[h.dtype], h, h.stride(0), gu_w, wts, out, M, K, E, ff, ffs, int(gated),
         int(sparse), code, int(weigh == "input"), *c)
    return out


def mid_act_ok(h: torch.Tensor, gu_w: torch.Tensor, ff: int, act="silu", gated: bool = True) -> bool:
    """Should ``mid_act`` run a dense first projection and its activation?  In the measured range, widths of 1024 on: from 33 rows on, where a round of tiles of
    32 (ungated 64) columns is enough (us with the activation, 64 rows, before -> now: 5632 x 2048 20.3 -> 15.7, 2816 x
    1024 13.0 -> 8.8, 4224 x 1536 17.3 -> 12.1; 264 tiles, 8448 x 3072, 34.9 -> 38.1); from 17 on if the tiles also fill half
    the chip (17 rows: 132 tiles 11.6 -> 10.2, 176 14.5 -> 13.5, 88 6.2 -> 7.8)."""
    M = h.shape[0]
    tiles = -(-ff // (32 if gated else 64))
    return (16 < M <= MID_MAX_M and 0 < tiles <= 256 and (M > THIN_ACT_MAX_M or tiles >= 128) and ff % 4 == 0
            and h.shape[-1] >= 1024 and (gated or isinstance(act, str)) and gu_w.shape[0] == (2 if gated else 1) * ff
            and (ff + 64) * h.shape[-1] < 1 << 31 and mid_ok(h, gu_w))


def mid_act(h, gu_w, ff: int, act="silu", gated: bool = True) -> torch.Tensor:
    """act(gate) * up (or act) of h @ gu_w^T, [M, ff], from the fp32 sums, for operands that ``mid_act_ok`` has let pass."""
    from ._seqmix import DT, call, use_seqmix

    use_seqmix(h)
    M, K = h.shape
    out = torch.empty((M, ff), dtype=h.dtype, device=h.device)
    code, c = (GATE_ACTS[act], (0.0,) * 4) if isinstance(act, str) else (
        4, (act.limit, act.limit_shared, act.slope, act.shift))
    call("sm_mid_act", DT[h.dtype], h, h.stride(0), gu_w, out, M, ff, K, int(gated), code, *c)
    return out


def act_rounds(M: int, ff: int) -> tuple:
    """Column ranges (c0, c1, ni) of the launches of ``tile_act``: whole rounds of 256 workgroups on tiles of 256 rows by 128
    columns, the rest on one round of the narrowest tiles that make it one."""
    tm = -(-M // 256)
    per = 256 // tm * 128                          # columns of a round
    if per == 0:
        return ()
    c = ff // per * per
    out = [(0, c, 8)] if c else []
    if c < ff:
        out.append((c, ff, next(ni for ni in (4, 6, 8) if tm * -(-(ff - c) // (16 * ni)) <= 256)))
    return tuple(out)


# Which products with a gated activation ``tile_act`` runs (us, product and pass -> here, bf16): width 2048, ff 5632: 300 rows
# 34.8 -> 26.4, 1000 51.3 -> 42.0, 4010 165 -> 148, 8000 314 -> 291; 1024, 2816: 512 18.4 -> 16.2, 4010 61 -> 48; 4096, 11008: 256 64 ->
# 62, 1000 164 -> 151, 4010 553 -> 526.  It needs the more of the tiles' area filled the longer a product is, as the library cuts
# long products of few tiles along K: over 98 sizes of 130 - 8000 rows and widths 512 - 4096 it is 0.90 - 1.76 times as fast under
# this rule, 1.19 in the mean (worst: 224 rows, ff 4224, width 1536 18.4 -> 20.5, 1290 x 5632 x 2048 72.7 -> 78.0; left out: 300 rows,
# width 4096, filled 0.54, 78 -> 80; 1290 rows, 0.68, 235 -> 248; 220, ff 3000, width 2048, 0.16, 20 -> 25).
# Up to 256 rows the product has tiles of 128 rows, and up to 224 walks of k apart, which are worth more than the pass (192 x 5632 x
# 2048 28.8 here, 23.7 with the pass, 224 x 11008 x 4096 62.9 and 61.0; 256 x 11264 x 4096 60.3 and 63.0).
ACT_TILE_FILL, ACT_TILE_FILL_MANY = 8192, 6000             # K over the filled share, up to 256 rows and above


def _act_tiles_pay(M: int, ff: int, K: int) -> bool:
    tm = -(-M // 256)
    cells = sum(256 * 256 * 16 * ni * -(-(tm * -(-(c1 - c0) // (16 * ni))) // 256) for c0, c1, ni in act_rounds(M, ff))
    few = few_tiles(M, 2 * ff, K) if M <= 256 else 0
    if few and (M <= 224 or few >> 4 & 15 == 4):
        return False
    return M * ff * (ACT_TILE_FILL if M <= 256 else ACT_TILE_FILL_MANY) >= K * cells > 0


def tile_act_ok(h: torch.Tensor, gu_w: torch.Tensor, ff: int, act="silu", gated: bool = True,
                rows: Optional[int] = None) -> bool:
    """Can and should ``tile_act`` run a dense first projection and its activation?  ``rows``: those of the batch that h is a
    part of, which decide, so that the parts round as the whole does."""
    xs, ws = h.shape, gu_w.shape
    if len(xs) != 2 or not h.is_cuda or not gated or not MID_MAX_M < (rows or xs[0]) <= 65536 or len(ws) != 2:
        return False
    M, K, dt = rows or xs[0], xs[1], h.dtype
    if M * ff < 512 * K:                           # less than the rule asks of one round (first: short prompts wait for the host)
        return False
    if (ws[0] != 2 * ff or ws[1] != K or K % 64 or K == 0 or ff % 8 or ff == 0 or 4 * ff * K >= 1 << 32 or dt != gu_w.dtype
            or dt not in (torch.bfloat16, torch.float16) or gu_w.device != h.device or not gu_w.is_contiguous()
            or not _act_tiles_pay(M, ff, K)):
        return False
    ld, one = h.stride()
    return (one == 1 and ld % 8 == 0 and K <= ld <= 1 << 22 and (h.data_ptr() | gu_w.data_ptr()) % 16 == 0
            and _plain(h, gu_w) and _here(h))


def tile_act(h, gu_w, ff: int, act="silu") -> torch.Tensor:
    """act(gate) * up of h @ gu_w^T, [M, ff], from the fp32 sums, for operands that ``tile_act_ok`` has let pass.  (HIP
    ``csrc/seqmix/tile_act.hip``.)"""
    from ._seqmix import DT, call, use_seqmix

    use_seqmix(h)
    M, K = h.shape
    out = torch.empty((M, ff), dtype=h.dtype, device=h.device)
    code, c = (GATE_ACTS[act], (0.0,) * 3) if isinstance(act, str) else (4, (act.limit_shared, act.slope, act.shift))
    for c0, c1, ni in act_rounds(M, ff):
        call("sm_tile_act", DT[h.dtype], h, h.stride(0), gu_w, out, M, K, ff, c0, c1, ni, code, *c)
    return out


def moe_dense(h, wts, gu_w, down_w, E: int, ff: int, ffs: int, act="silu", gated: bool = True,
              weigh: str = "output", top: Optional[int] = None) -> torch.Tensor:
    """``top`` (optional): every row has at most that many non-zero weights."""
    M = h.shape[0]
    sparse = (M <= THIN_ACT_MAX_M and top is not None and 0 < E and M * top <= SPARSE_ROWS * E
              and ff % 64 == 0 and ffs % 64 == 0 and down_w.is_contiguous()
              and down_w.dim() == 2 and down_w.shape[1] == E * ff + ffs
              and down_w.dtype == h.dtype and down_w.device == h.device
              and down_w.shape[0] % 4 == 0 and down_w.data_ptr() % 16 == 0 and _plain(down_w))
    if M <= THIN_ACT_MAX_M and thin_act_ok(h, wts, gu_w, E, ff, ffs, act, gated, weigh, sparse):
        a = _thin_act(h, gu_w, wts, E, ff, ffs, act, gated, weigh, sparse)
        if sparse:
            return _thin(a, down_w, blocks=(wts, E, ff, ffs))
        return project(a, down_w)
    return project(_act(project(h, gu_w), wts, E, ff, ffs, act, gated, weigh), down_w)


def feed_forward(h, gu_w, down_w, ff: int, act="silu", gated: bool = True) -> torch.Tensor:
    """Dense feed-forward W_down (act(W_gate h) * W_up h) ([gate | up] rows stacked in ``gu_w``), or
    without a gate W_down act(W_up h)."""
    return project(ff_act(h, gu_w, ff, act, gated), down_w)


def ff_act(h, gu_w, ff: int, act="silu", gated: bool = True) -> torch.Tensor:
    """The first half of ``feed_forward``: act(W_gate h) * W_up h, or act(W_up h)."""
    if h.dim() == 2 and h.shape[0] <= MID_MAX_M:
        if mid_act_ok(h, gu_w, ff, act, gated):
            return mid_act(h, gu_w, ff, act, gated)
        if h.shape[0] <= THIN_ACT_MAX_M and thin_act_ok(h, None, gu_w, 0, 0, ff, act, gated):
            return _thin_act(h, gu_w, None, 0, 0, ff, act, gated)
    elif tile_act_ok(h, gu_w, ff, act, gated):
        return tile_act(h, gu_w, ff, act)
    return _act(project(h, gu_w), None, 0, 0, ff, act, gated, "output")


def moe_grouped(h, wts, gu_w, down_w, E: int, ff: int, ffs: int, act="silu", gated: bool = True,
                weigh: str = "output") -> torch.Tensor:
    """Same result as ``moe_dense`` (to rounding) running each expert on its own rows only."""
    T = h.shape[0]
    k = 2 if gated else 1                                 # rows of the first weight per ff
    tok, exp = (wts > 0).nonzero(as_tuple=True)           # (host sync) pairs in token order
    order = torch.argsort(exp, stable=True)
    tok, exp = tok[order], exp[order]
    counts = torch.bincount(exp, minlength=E).tolist()
    x = h.index_select(0, tok)
    wsel = wts[tok, exp].unsqueeze(1)
    out = torch.zeros(T, h.shape[1], dtype=torch.float32, device=h.device)
    ys = torch.empty(x.shape[0], h.shape[1], dtype=h.dtype, device=h.device)
    a = 0
    for e, n in enumerate(counts):
        if n:
            gu = F.linear(x[a:a + n], gu_w[e * k * ff:(e + 1) * k * ff])
            torch.matmul(_act(gu, wsel[a:a + n], 1, ff, 0, act, gated, weigh),
                         down_w[:, e * ff:(e + 1) * ff].t(), out=ys[a:a + n])
            a += n
    out.index_add_(0, tok, ys.float())
    if ffs:
        gu = F.linear(h, gu_w[E * k * ff:])
        out += F.linear(_act(gu, None, 0, 0, ffs, act, gated, weigh), down_w[:, E * ff:]).float()
    return out.to(h.dtype)


def grouped_mm_ok(h: torch.Tensor, ff: int) -> bool:
    """Can ``moe_grouped_mm`` run: the library's grouped GEMM (one launch for all experts, group
    offsets read on the device) exists, a 16-bit dtype on the GPU, 16-byte aligned rows."""
    return (h.is_cuda and h.dtype in (torch.bfloat16, torch.float16)
            and hasattr(torch, "_grouped_mm") and ff % 8 == 0 and h.shape[1] % 8 == 0)


def moe_grouped_mm(h, wts, gu_w, down_w, E: int, top: int, ff: int, ffs: int, act="silu",
                   gated: bool = True, weigh: str = "output") -> torch.Tensor:
    """``moe_grouped`` without the host in the loop: every row has exactly ``top`` chosen
    experts, so the (row, expert) pairs are a [T * top] list of static size; sorted by expert they
    feed ONE grouped GEMM per projection whose group offsets stay on the device.  No
    synchronisation, three launches per layer instead of three per expert."""
    T, W = h.shape
    k = 2 if gated else 1
    val, idx = torch.topk(wts, top, dim=1)                         # [T, top]: weights, experts
    exp = idx.reshape(-1)
    order = torch.argsort(exp, stable=True)
    tok = torch.div(order, top, rounding_mode="floor")
    offs = torch.cumsum(torch.bincount(exp, minlength=E), 0).to(torch.int32)
    x = h.index_select(0, tok)
    u = torch._grouped_mm(x, gu_w[:E * k * ff].view(E, k * ff, W).transpose(1, 2), offs=offs)
    a = _act(u, val.reshape(-1)[order].reshape(-1, 1).contiguous(), 1, ff, 0, act, gated,
             weigh)
    y = torch._grouped_mm(a, down_w[:, :E * ff].view(W, E, ff).permute(1, 2, 0), offs=offs)
    out = torch.zeros(T, W, dtype=torch.float32, device=h.device)
    out.index_add_(0, tok, y.float())
    if ffs:
        gu = F.linear(h, gu_w[E * k * ff:])
        out += F.linear(_act(gu, None, 0, 0, ffs, act, gated, weigh), down_w[:, E * ff:]).float()
    return out.to(h.dtype)


def chosen_ok(h, wts, gu_w, down_w, E: int, top: int, ff: int, ffs: int, act="silu", gated: bool = True,
              weigh: str = "output") -> bool:
    """Can ``moe_chosen`` run these operands?"""
    from ._seqmix import DT, expert_ok, use_seqmix

    if not (h.is_cuda and h.dim() == 2 and h.dtype in (torch.bfloat16, torch.float16) and use_seqmix(h)):
        return False
    (T, W), k, N = h.shape, 2 if gated else 1, E * ff + ffs
    return (T > 0 and h.stride(1) == 1 and h.stride(0) % 8 == 0 and h.stride(0) >= W and T * h.stride(0) < 1 << 31
            and tuple(gu_w.shape) == (k * N, W) and tuple(down_w.shape) == (W, N)
            and gu_w.dtype == down_w.dtype == h.dtype and gu_w.is_contiguous() and down_w.is_contiguous()
            and gu_w.device == down_w.device == h.device and weights_ok(wts, h, E)
            and (h.data_ptr() | gu_w.data_ptr() | down_w.data_ptr()) % 16 == 0
            and 2 * max(ff, ffs) * W < 1 << 31 and 256 * N < 1 << 31 and 128 * max(ff, ffs) < 1 << 31
            and (gated or isinstance(act, str) and weigh == "output")
            and expert_ok(DT[h.dtype], T, W, E, top, ff, ffs) and _plain(h, gu_w, down_w, wts) and _here(h))


def moe_chosen(h, wts, gu_w, down_w, E: int, top: int, ff: int, ffs: int, act="silu", gated: bool = True,
               weigh: str = "output", checked: bool = False) -> torch.Tensor:
    """The weighted sum of each row's chosen experts (+ the shared one) on the rows that chose them: HIP kernels that
    read the rows where they lie and the counts on the device (seqmix/expert_gemm.hip).  A row has at most ``top``
    non-zero weights.  Results of an expert stay fp32 until their sum is rounded.  ``checked``: ``chosen_ok`` has let
    these operands pass."""
    from ._seqmix import DT, call

    if weigh not in ("output", "input"):
        raise ValueError(f"unknown place of the routing weight {weigh!r}")
    if not (checked or chosen_ok(h, wts, gu_w, down_w, E, top, ff, ffs, act, gated, weigh)):
        raise ValueError("chosen experts: rows, stacked weights and routing weights do not fit the kernels")
    T, W = h.shape
    dev, dt = h.device, DT[h.dtype]
    n = T * top
    # one buffer for what lies between the launches, its parts by address (short prompts wait for the host)
    sizes = (n * ff * 2, T * ffs * 2, n * W * 4, T * W * 4 if ffs else 0, 4 * n, 4 * n, 4 * n, 4 * (E + 1))
    at = [0]
    for b in sizes:
        at.append(at[-1] + (b + 255 & ~255))
    ws = torch.empty(at[-1], dtype=torch.uint8, device=dev)
    p0 = ws.data_ptr()
    a, a_s, y, y_s, idx, place, wt, off = (p0 + o for o in at[:-1])
    if not ffs:
        a_s = y_s = None
    call("sm_expert_sort", wts, off, idx, wt, place, T, E, top)
    code, c = (GATE_ACTS[act], (0.0,) * 4) if isinstance(act, str) else (
        4, (act.limit, act.limit_shared, act.slope, act.shift))
    call("sm_expert_act", dt, h, h.stride(0), gu_w, off, idx, wt, a, a_s, T, W, E, top, ff, ffs, int(gated), code,
         int(weigh == "input"), *c)
    out = torch.empty(T, W, dtype=h.dtype, device=dev)
    call("sm_expert_down", dt, a, a_s, down_w, off, place, y, y_s, out, T, W, E, top, ff, ffs)
    return out


# When the grouped form pays.  Measured on MI355X (bf16, 16 experts, widths 1024 - 4096, 512 - 16384
# rows): the two stacked GEMMs of the dense form run at ~850 TFLOP/s, the grouped GEMMs at ~300, and
# sorting the (row, expert) pairs costs ~0.4 - 0.8 ms per layer whatever the size.  The grouped form does
# top / E of the dense form's FLOPs at about a third of its rate, so it needs E > 3 top to save
# anything, and enough products saved in the experts' first GEMM to cover the sorting: the two forms
# take the same time between 90 and 170 G multiply-adds at every size (inside a model the dense form's
# two launches also hide better), so the grouped one is taken above that.
GROUPED_RATE_RATIO = 3
GROUPED_MIN_SAVING = 180e9          # rows x (E - GROUPED_RATE_RATIO * top) x an expert's [k ff, W]


def grouped_pays(rows: int, E: int, top: int, expert_weights: int) -> bool:
    """Do ``rows`` rows save enough by visiting only their chosen experts (``expert_weights``:
    elements of one expert's first projection)?"""
    return rows * (E - GROUPED_RATE_RATIO * top) * expert_weights >= GROUPED_MIN_SAVING


# Up to 32 rows the activation forms in the thin GEMM's epilogue and experts no row chose are not read; up to 64 the
# thin GEMM still has the smaller stacks (width 1024, 8 experts of 704, top 2, 48 rows: 32 us against 39).  Beyond, a layer's
# time from weights in HBM, dense -> chosen in us (bf16, experts of 2.75 / 4 of the width):
#   16 experts  width 1024: 72 rows 53 -> 46, 256 63 -> 50;  1536: 118 -> 64, 158 -> 69;  2048, top 3 and a shared one: 33 rows
#               156 -> 90, 72 100 -> 91, 512 167 -> 99;  4096: 8192 rows 2721 (the library's grouped product) -> 1685
#   8 experts   width 4096: 33 rows 243 -> 153, 72 169 -> 154;  3072: 152 -> 103, 110 -> 103
#               but 1024: 72 rows 39 -> 43, 160 43 -> 44, 320 55 -> 46;  1536: 72 55 -> 61, 160 60 -> 61, 192 77 -> 63;  2048: 33
#               62 -> 68, 72 61 -> 69, 160 69 -> 70, 192 71 -> 72, 256 76 -> 74, 512 96 -> 79
#   4 experts   width 2048, top 1: 72 rows 38 -> 58, 512 64 -> 68, 768 81 -> 68;  4096: 72 86 -> 104, 256 112 -> 115, 320 126 -> 118
# A tile of rows per expert costs the same at any width, and few experts leave the dense product little to spare: they
# take their own rows from where that pays.  (Widths below 1024, which no served layer has: not measured, by row count alone.)
CHOSEN_MANY_EXPERTS, CHOSEN_WIDE = 16, 3072


def chosen_pays(rows: int, gu_w: torch.Tensor, E: int) -> bool:
    """Do ``rows`` rows run faster on their chosen experts' own rows than on all ``E`` experts?"""
    W = gu_w.shape[1]
    if E < CHOSEN_MANY_EXPERTS and W >= 1024:
        least = (0 if E >= 8 else 256) if W >= CHOSEN_WIDE else (160 if E >= 8 else 512)
        if rows <= least:
            return False
    return rows > THIN_MAX_M or rows > THIN_ACT_MAX_M and gu_w.numel() > THIN_BATCH_MAX_W


def moe(h, wts, gu_w, down_w, E: int, top: int, ff: int, ffs: int, act="silu",
        gated: bool = True, weigh: str = "output") -> torch.Tensor:
    """Weighted sum of each row's chosen experts (+ the shared expert): [T, W] in h's dtype.
    ``gated``: an expert is W_down (act(W_gate h) * W_up h) with [gate | up] rows stacked per
    expert in ``gu_w`` (``act`` also a ``ClampedGate``); else W_down act(W_up h) with the up rows
    alone.  ``weigh`` = "input": an expert sees its weight times h instead of weighing in with its
    output (gated experts)."""
    if chosen_pays(h.shape[0], gu_w, E) and chosen_ok(h, wts, gu_w, down_w, E, top, ff, ffs, act, gated, weigh):
        return moe_chosen(h, wts, gu_w, down_w, E, top, ff, ffs, act, gated, weigh, True)
    grouped = (grouped_pays(h.shape[0], E, top, (2 if gated else 1) * ff * h.shape[1])
               and not (h.is_cuda and torch.cuda.is_current_stream_capturing()))
    if grouped and grouped_mm_ok(h, ff):
        return moe_grouped_mm(h, wts, gu_w, down_w, E, top, ff, ffs, act, gated, weigh)
    if grouped:
        return moe_grouped(h, wts, gu_w, down_w, E, ff, ffs, act, gated, weigh)
    return moe_dense(h, wts, gu_w, down_w, E, ff, ffs, act, gated, weigh, top)
