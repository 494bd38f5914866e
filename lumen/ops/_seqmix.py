"""Loader for the sequence-mixing kernel library ``lumen/_C_seqmix.so`` (``lumen/csrc/seqmix``).

The library is plain ``extern "C"`` launchers (raw pointers, sizes, a HIP stream) bound through
ctypes, so it builds in seconds without the torch headers and a model that needs only these
kernels does not wait for the full extension.  Policy as for ``lumen._C``: on a GPU tensor the
HIP kernel is THE implementation; when the library is missing it is built once (hipcc, gfx950),
and if that is impossible every op raises.  CPU tensors take the torch reference path.
"""
from __future__ import annotations

import ctypes
import os

import torch

_lib = None
_err = None

_T = {"p": ctypes.c_void_p, "i": ctypes.c_int, "l": ctypes.c_longlong, "f": ctypes.c_float}

# launcher name -> argument kinds (p pointer, i int32, l int64, f float); a hipStream_t follows
SIGNATURES = {
    "sm_dyt": "iipppppii",
    "sm_dyt_residual": "iipppppppppii",
    "sm_dyt_canon": "ipppppppppppiii",
    "sm_canon_tail": "ppppppppiii",
    "sm_token_shift": "ippppppppiii",
    "sm_shift_tail": "ippppii",
    "sm_wkv": "iplplplplpiplppppplpppiiif",
    "sm_gdelta": "iplplplplpiplplppppplpppiiifff",
    "sm_write_k": "iplppii",
    "sm_chunk_attn": "iplpppippiiiiiffii",
    "sm_chunk_attn_tiles": "iplpppipippiiiiffiii",
    "sm_route_topk": "ppiii",
    "sm_gated_act": "ipppiiiii" "iffff",
    "sm_group_rms": "iiplpppliiif",
    "sm_gate_rows": "iplplpiipi",
    "sm_rotate_heads": "iplliiippi",
    "sm_latent_write": "iplpppppppiiiiif",
    "sm_head_norm_write": "iplpppppiiiiif",
    "sm_latent_attn": "i" "plli" "plli" "pl" "pi" "pll" "pi" "pp" "iii" "fffi" "ppp" "pl" "iiipp",
    "sm_row_attn": "i" "plli" "plli" "pl" "pli" "pll" "pi" "pp" "iiiii" "fffi" "pppp" "piipl"
                   "pi" "iipp",
    "sm_win_attn_tiles": "iplppppl" "pi" "pi" "pp" "iiii" "ff" "p" "iii" "ipi",
    "sm_fresh_tiles": "i" "plplplpl" "p" "piii" "pp" "iiii" "f",
    "sm_talk_tiles": "i" "pll" "pp" "pll" "pi" "pii" "pp" "iiiii" "fffi" "pppp",
    "sm_expert_sort": "pppppiii",
    "sm_expert_act": "iplp" "ppppp" "iiiiii" "iii" "ffff",
    "sm_expert_down": "ippp" "pp" "ppp" "iiiiii",
    "sm_row_gemv": "ipppppp" "iii" "f",
    "sm_row_stream": "ippppppp" "iiii" "f",
    "sm_row_norm_write": "iplpppppiiif",
    "sm_layer_norm": "iippfpppiif",
    "sm_embed_pos": "ipppppiiii",
    "sm_route_groups": "pppiiiiiiffii",
    "sm_latent_in": "iplpp" "pppp" "pp" "iiiiii" "f",
    "sm_latent_query": "iplipp" "iiiiii" "pp",
    "sm_latent_out": "ippi" "pll" "pl" "p" "pll" "iiii",
    "sm_mid_slabs": "iplpp" "iiii",
    "sm_mid_act": "iplpp" "iiiii" "ffff",
    "sm_tile_act": "iplpp" "iiiiii" "i" "fff",
    "sm_slab_rms": "ipippp" "iii" "f",
    "sm_thin_tail": "iplpp" "iiii" "plip",
    "sm_thin_gate": "iplpp" "iii" "plp",
    "sm_route_rows": "ii" "pp" "pl" "ppp" "ppp" "ppp" "iii" "f" "iiiiii" "ff" "p",
    "sm_rotary_write": "iplppppiiiiipii",
    "sm_min_gru": "iplpppppppiifppii",
    "sm_diff_combine": "ipplpiiiifff",
    "sm_depth_mix": "iipipppppppppppiif",
    "sm_embed_scaled": "ipppiiif",
    "sm_soft_cap": "ipplf",
    "sm_scaled_act": "ipppiiiii",
    "sm_gated_rms": "ipplppiiiiiif",
    "sm_hyper_mix": "i" "pppi" "ppppf" "ppp" "ppf" "pp" "iiii",
    "sm_head_norm_rotary": "ipl" "ppppppp" "iiiiiiif",
    "sm_row_norm_rotary": "ipl" "ppppppp" "iiiiii" "ff",
    "sm_stream_rms": "ipi" "ppifp" "p" "pppf" "ppi" "iif",
    "sm_head_scan_chunk": "ii" "plplplplpl" "pppp" "pp" "ppp" "iiiiiiff",
    "sm_head_scan_ahead": "ii" "plplplplpl" "pppp" "pp" "ppp" "iiiiiiff" "pi",
    "sm_head_scan_step": "ii" "plplplplpl" "pppp" "pp" "ppp" "iiiiiiff",
    "sm_short_conv": "iplpppp" "pppp" "iii",
    "sm_conv_tail": "iiplpppp" "ppp" "iii",
    "sm_fill_step": "ppippippi" "pp" "ppl" "ppii" "ii",
    "sm_dyt_canon_rows": "ippppp" "pppppp" "ppi" "ppp" "iiii",
    "sm_latent_tiles": "i" "plli" "plli" "pl" "pi" "pll" "pi" "pii" "pp" "ii" "fffi" "ppp" "pl",
    "sm_scan_chunk": "ii" "plplplplpl" "pppp" "ppp" "iii" "ff",
    "sm_thin_gemm": "iplpppliiii" "piii",
    "sm_thin_act": "iplppp" "iiiiiiiii" "ffff",
}


def _load():
    global _lib, _err
    if _lib is not None or _err is not None:
        return _lib
    try:
        from ..csrc.build import build_seqmix, seqmix_path, seqmix_stale

        path = seqmix_path()
        if not os.path.exists(path) or seqmix_stale():
            build_seqmix(verbose=False)
        lib = ctypes.CDLL(path)
        for name, sig in SIGNATURES.items():
            fn = getattr(lib, name)
            fn.argtypes = [_T[c] for c in sig] + [ctypes.c_void_p]
            fn.restype = ctypes.c_int
        lib.sm_chunk_attn_tiles_ok.argtypes = [ctypes.c_int, ctypes.c_int]
        lib.sm_chunk_attn_tiles_ok.restype = ctypes.c_int
        lib.sm_win_attn_tiles_ok.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int]
        lib.sm_win_attn_tiles_ok.restype = ctypes.c_int
        lib.sm_fresh_tiles_ok.argtypes = [ctypes.c_int] * 4
        lib.sm_fresh_tiles_ok.restype = ctypes.c_int
        lib.sm_talk_tiles_ok.argtypes = [ctypes.c_int] * 5
        lib.sm_talk_tiles_ok.restype = ctypes.c_int
        lib.sm_expert_ok.argtypes = [ctypes.c_int] * 7
        lib.sm_expert_ok.restype = ctypes.c_int
        lib.sm_row_attn_lds.argtypes = [ctypes.c_int, ctypes.c_int]
        lib.sm_row_attn_lds.restype = ctypes.c_int
        lib.sm_latent_attn_ok.argtypes = [ctypes.c_int] * 5
        lib.sm_latent_attn_ok.restype = ctypes.c_int
        lib.sm_latent_tiles_ok.argtypes = [ctypes.c_int] * 6
        lib.sm_latent_tiles_ok.restype = ctypes.c_int
        lib.sm_latent_plan.argtypes = [ctypes.c_int] * 6 + [ctypes.POINTER(ctypes.c_int)]
        lib.sm_latent_plan.restype = ctypes.c_int
        lib.sm_step_attn_ok.argtypes = [_T[k] for k in "ipllii" "plpli" "pll" "iiiiii"]
        lib.sm_step_attn_ok.restype = ctypes.c_int
        lib.sm_head_scan_ahead_bytes.argtypes = [ctypes.c_int] * 5
        lib.sm_head_scan_ahead_bytes.restype = ctypes.c_longlong
        lib.sm_min_gru_sub.argtypes = []
        lib.sm_min_gru_sub.restype = ctypes.c_int
        _lib = lib
    except Exception as e:  # pragma: no cover - depends on build state
        _err = e
    return _lib


def seqmix_error():
    _load()
    return _err


def use_seqmix(t: torch.Tensor) -> bool:
    """True when ``t`` lives on the GPU (the HIP path must run, or this raises)."""
    if not t.is_cuda:
        return False
    if _load() is None:
        raise RuntimeError(f"lumen sequence-mixing kernels are not available ({_err!r}); build "
                           "them with `python -m lumen.csrc.build --seqmix`")
    return True


DT = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}


def tiles_ok(dt: int, D: int) -> bool:
    """Does the matrix-core prefill attention have a kernel for this dtype code / head size?"""
    return bool(_load().sm_chunk_attn_tiles_ok(dt, D))


def win_tiles_ok(dt: int, D: int, Dv: int = 0) -> bool:
    """Does the matrix-core prefill attention over paged key and value caches have a kernel for
    this dtype code / key size / value size (0: the key size)?"""
    return bool(_load().sm_win_attn_tiles_ok(dt, D, Dv or D))


def fresh_tiles_ok(dt: int, D1: int, Dr: int, Dv: int) -> bool:
    """Does the prompt attention over a step's own rows have a kernel for this dtype code / key size / shared key
    size / value size?"""
    return bool(_load().sm_fresh_tiles_ok(dt, D1, Dr, Dv))


def talk_tiles_ok(dt: int, H: int, G: int, D: int, Dv: int) -> bool:
    """Does the prompt attention with mixed heads have a kernel for this dtype code / heads / sizes?"""
    return bool(_load().sm_talk_tiles_ok(dt, H, G, D, Dv))


def expert_ok(dt: int, T: int, W: int, E: int, top: int, ff: int, ffs: int) -> bool:
    """Do the products over chosen experts have kernels for this dtype code and these sizes?"""
    return bool(_load().sm_expert_ok(dt, T, W, E, top, ff, ffs))


def row_attn_lds(HB: int, Dk: int) -> int:
    """LDS bytes the row-attention kernel needs for a block of HB heads with key size Dk."""
    return int(_load().sm_row_attn_lds(HB, Dk))


def latent_attn_ok(dt: int, Dv: int, Dk: int, D1: int, bs: int) -> bool:
    """Does the matrix-core latent attention have a kernel for these sizes?"""
    return bool(_load().sm_latent_attn_ok(dt, Dv, Dk, D1, bs))


def latent_plan(Dv: int, Dk: int, T: int, H: int, keys: int, joined: bool) -> tuple:
    """(keys that a workgroup of the latent attention takes, splits of the keys) for T rows with H heads behind tables of
    ``keys`` keys.  ``joined``: the expansion adds the splits, else a launch of its own does."""
    n = ctypes.c_int()
    return int(_load().sm_latent_plan(Dv, Dk, T, H, keys, int(joined), ctypes.byref(n))), n.value


def latent_tiles_ok(dt: int, Dv: int, Dk: int, D1: int, bs: int, max_blocks: int) -> bool:
    """Does the latent attention have a kernel that shares key tiles among rows for these sizes?"""
    return bool(_load().sm_latent_tiles_ok(dt, Dv, Dk, D1, bs, max_blocks))


def step_attn_ok(dt: int, q1, D1: int, D2: int, kc, krow: int, vc, vrow: int, Dv: int, out, H: int, G: int, bs: int, mixed: bool,
                 sigmoid: bool, vdiv: int) -> bool:
    """Does the row attention take the kernels of decode steps (csrc/seqmix/step_attention.hip) for these operands?"""
    return bool(_load().sm_step_attn_ok(dt, q1.data_ptr(), q1.stride(0), q1.stride(1), D1, D2, kc.data_ptr(), krow, vc.data_ptr(), vrow,
                                        Dv, out.data_ptr(), out.stride(0), out.stride(1), H, G, bs, int(mixed), int(sigmoid), vdiv))


def head_scan_ahead_bytes(delta: bool, Dk: int, H: int, rep: int, chunks: int) -> int:
    """Workspace of the scan whose chunks are built ahead for a step of ``chunks`` chunks; 0: no such kernel."""
    return int(_load().sm_head_scan_ahead_bytes(int(delta), Dk, H, rep, chunks))


def min_gru_sub() -> int:
    """Sub-chunks the minGRU scan cuts a tile of prompt rows into (sizes its scratch)."""
    return int(_load().sm_min_gru_sub())


def call(name: str, *args) -> None:
    """Launch ``name`` on the current stream; tensors are passed by their data pointers."""
    lib = _load()
    sig = SIGNATURES[name]
    if len(args) != len(sig):
        raise TypeError(f"{name}: {len(args)} arguments for signature {sig!r}")
    dev, vals = None, []
    for kind, v in zip(sig, args):                 # (host time: short prompts are bound by it)
        if kind == "p":
            if isinstance(v, torch.Tensor):
                if dev is None:
                    dev = v.device.index
                v = v.data_ptr()
        elif kind == "f":
            v = float(v)
        elif type(v) is not int:
            v = int(v)
        vals.append(v)
    rc = getattr(lib, name)(*vals, torch._C._cuda_getCurrentRawStream(dev))
    if rc != 0:
        raise RuntimeError(f"{name}: HIP error {rc}")
