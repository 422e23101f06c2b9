"""ctypes binding of the C ABI declared in ``include/tttj_amd.h`` (library ``libtttj_amd.so``).

There is no fallback: if the library is missing or fails to load, every optimized entry point
raises.  Loading needs no GPU (the bookkeeping exports work on a CPU-only host); the compute
exports need a gfx950 device.
"""

from __future__ import annotations

import ctypes
import pathlib
import threading

LIB_PATH = pathlib.Path(__file__).resolve().parent / "libtttj_amd.so"

TT_OK, TT_ERR_INVALID, TT_ERR_HIP = 0, 1, 2
PLAN_AUTO, PLAN_LAYERWISE, PLAN_MEGAKERNEL, PLAN_FUSED_LN = 0, 1, 2, 3
EPILOGUES = {"bias": 0, "gelu": 1, "resid_masked": 2, "masked_resid": 3, "qkv": 4}

_P = ctypes.c_void_p
_I = ctypes.c_int
_I64 = ctypes.c_int64
_F = ctypes.c_float

# name -> (restype, argtypes); must match include/tttj_amd.h exactly.
SIGNATURES = {
    "tt_version": (ctypes.c_char_p, []),
    "tt_last_error_string": (ctypes.c_char_p, []),
    "tt_device_count": (_I, []),
    "tt_weight_layout": (_I, [_I, _I, _I, ctypes.POINTER(_I64), ctypes.POINTER(_I64),
                              ctypes.POINTER(_I64), ctypes.POINTER(_I64)]),
    "tt_workspace_bytes": (_I, [_I, _I, _I, _I, _I, _I, _I, ctypes.POINTER(_I64)]),
    "tt_resolve_plan": (_I, [_I, _I, _I, _I, _I, _I]),
    "tt_forward_packs_rows": (_I, [_I, _I, _I, _I, _I, _I]),
    "tt_forward_packing_override": (_I, [_I]),
    "tt_stage_offsets": (_I, [_I, _I, _I, _I, _I, _I, _I, ctypes.POINTER(_I64),
                              ctypes.POINTER(_I64), ctypes.POINTER(_I64)]),
    "tt_megakernel_status": (_I, [_P, _I, _I, _I, _I, _I, ctypes.POINTER(_I), _P]),
    "tt_megakernel_tasks": (_I, [_I, _I, _I, _I, _I, _I]),
    "tt_megakernel_error_offset": (_I, [_I, _I, _I, _I, _I, _I, ctypes.POINTER(_I64)]),
    "tt_megakernel_set_spin_limit": (_I, [_I64]),
    "tt_megakernel_attach_status": (_I, [_P, _I64, _I, _I, _I, _I, _I, _I, _P, _P]),
    "tt_megakernel_trace_fwd": (_I, [_P, _P, _P, _P, _P, _I64, _I, _I, _I, _I, _I, _I, _I, _P,
                                     _I64, _P]),
    "tt_layernorm_fwd": (_I, [_P, _P, _P, _P, _P, _I, _I, _F, _P]),
    "tt_linear_fwd": (_I, [_P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _I, _I, _P]),
    "tt_gemm_tile_override": (_I, [_I]),
    "tt_pack_derived": (_I, [_P, _I, _I, _I, _P]),
    "tt_mask_info": (_I, [_P, _P, _I, _I, _P]),
    "tt_attention_fwd": (_I, [_P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _P]),
    "tt_attention_masked_fwd": (_I, [_P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _I, _P]),
    "tt_attention_fwd_prescaled": (_I, [_P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _P]),
    "tt_transformer_fwd": (_I, [_P, _P, _P, _P, _P, _I64, _I, _I, _I, _I, _I, _I, _I, _I, _P]),
    "tt_noalloc_scratch_bytes": (_I, [ctypes.POINTER(_I64)]),
    "tt_transformer_fwd_noalloc": (_I, [_P, _P, _P, _P, _I, _I, _I, _I, _I, _I, _I, _I, _P]),
    "tt_noalloc_status": (_I, [ctypes.POINTER(_I), _P]),
}

_lock = threading.Lock()
_lib = None


class LibraryError(RuntimeError):
    pass


def load() -> ctypes.CDLL:
    """Load (once) and return the library with typed signatures."""
    global _lib
    with _lock:
        if _lib is None:
            if not LIB_PATH.exists():
                raise LibraryError(
                    f"{LIB_PATH} is not built; run `python -m tttj_2026_amd.build` "
                    "(or __graft_entry__.build()) first")
            lib = ctypes.CDLL(str(LIB_PATH))
            for name, (res, args) in SIGNATURES.items():
                fn = getattr(lib, name)
                fn.restype = res
                fn.argtypes = args
            _lib = lib
        return _lib


def last_error() -> str:
    return load().tt_last_error_string().decode(errors="replace")


def check(rc: int, what: str) -> None:
    """Raise for a non-zero status: ValueError for argument errors, RuntimeError for HIP errors."""
    if rc == TT_OK:
        return
    msg = f"{what}: {last_error()}"
    if rc == TT_ERR_INVALID:
        raise ValueError(msg)
    raise RuntimeError(msg)


LAYER_SEGMENTS = 18


def weight_layout(d_model: int, ffn_dim: int, num_layers: int):
    """Return (LAYER_SEGMENTS per-layer offsets, layer stride, final-norm offset, total
    elements)."""
    lib = load()
    offs = (_I64 * LAYER_SEGMENTS)()
    stride, final, total = _I64(), _I64(), _I64()
    check(lib.tt_weight_layout(d_model, ffn_dim, num_layers, offs, ctypes.byref(stride),
                               ctypes.byref(final), ctypes.byref(total)), "tt_weight_layout")
    return list(offs), stride.value, final.value, total.value


def workspace_bytes(batch: int, seq: int, d_model: int, heads: int, ffn_dim: int,
                    num_layers: int = 1, plan: int = PLAN_LAYERWISE) -> int:
    out = _I64()
    check(load().tt_workspace_bytes(batch, seq, d_model, heads, ffn_dim, num_layers, plan,
                                    ctypes.byref(out)), "tt_workspace_bytes")
    return out.value


def stage_offsets(batch: int, seq: int, d_model: int, heads: int, ffn_dim: int, num_layers: int,
                  plan: int):
    """(qkv, ctx, hidden) byte offsets of the last layer's intermediates in a forward's workspace
    (``tt_stage_offsets``; ctx is -1 where the plan overwrites it)."""
    q, c, h = _I64(), _I64(), _I64()
    check(load().tt_stage_offsets(batch, seq, d_model, heads, ffn_dim, num_layers, plan,
                                  ctypes.byref(q), ctypes.byref(c), ctypes.byref(h)),
          "tt_stage_offsets")
    return q.value, c.value, h.value


def megakernel_error_offset(batch: int, seq: int, d_model: int, heads: int, ffn_dim: int,
                            num_layers: int) -> int:
    out = _I64()
    check(load().tt_megakernel_error_offset(batch, seq, d_model, heads, ffn_dim, num_layers,
                                            ctypes.byref(out)), "tt_megakernel_error_offset")
    return out.value


def forward_packs_rows(batch: int, seq: int, d_model: int, num_heads: int, ffn_dim: int,
                       plan: int = PLAN_AUTO) -> bool:
    """Whether a masked forward of this shape runs on packed variable-length rows."""
    rc = load().tt_forward_packs_rows(batch, seq, d_model, num_heads, ffn_dim, plan)
    if rc < 0:
        check(TT_ERR_INVALID, "tt_forward_packs_rows")
    return bool(rc)


def packed_row_tokens(mask, seq: int):
    """Token index (b * S + s) of every packed row of a masked forward that packs rows, -1 for the
    rows that pad a right-padded sequence to a multiple of 8 (the layout of
    ``tt_forward_packs_rows``; computed on the host from a CPU bool mask [B, S])."""
    rows = []
    for b in range(mask.shape[0]):
        valid = mask[b].nonzero().flatten().tolist()
        kv_end = valid[-1] + 1 if valid else 0
        if len(valid) == kv_end:  # right-padded prefix (or empty)
            n = min((kv_end + 7) // 8 * 8, seq)
            rows += [b * seq + s if s < kv_end else -1 for s in range(n)]
        else:
            rows += [b * seq + s for s in valid]
    return rows


def resolve_plan(batch: int, seq: int, d_model: int, num_heads: int, ffn_dim: int,
                 plan: int) -> int:
    rc = load().tt_resolve_plan(batch, seq, d_model, num_heads, ffn_dim, plan)
    if rc < 0:
        check(TT_ERR_INVALID, "tt_resolve_plan")
    return rc
