"""ctypes binding of libnvl_seq.so (C ABI in include/nvl_seq.h): the kernels of layers that carry per-sequence state,
of windowed paged attention with any head size and of norms on a 32-bit residual stream.

As in ops.py, PyTorch owns memory and the stream and every function hands raw device pointers to a hand-written gfx950
kernel; there is no fallback. Activation / weight tensors are bfloat16 or float32 (`_code`), state and the residual
stream are float32. The library is built on first use when it is missing (a fresh checkout), by hipcc, in-tree.
"""
from __future__ import annotations

import ctypes
import os
from ctypes import c_char_p, c_float, c_int, c_int64, c_void_p

import torch

from . import build as _build
from .attn_meta import get_context, plain_calls as _launch

ABI_VERSION = 7
_P, _I, _L, _F = c_void_p, c_int, c_int64, c_float

SIGNATURES = {
    "nvs_abi_version": (c_int, []),
    "nvs_last_error": (c_char_p, []),
    "nvs_embed_sinusoid": (c_int, [_P, _I, _P, _P, _L, _I, _F, _F, _P, _P, _P]),
    "nvs_norm_residual": (c_int, [_P, _P, _P, _P, _P, _I, _L, _I, _F, _P, _P, _P]),
    "nvs_scalar_norm_rows": (c_int, [_P, _P, _L, _I, _P, _I, _F, _P, _P]),
    "nvs_xielu": (c_int, [_P, _P, _F, _I, _L, _P, _P]),
    "nvs_causal_conv": (c_int, [_P, _L, _I, _P, _P, _I, _I, _I, _P, _P, _P, _P, _I, _L, _P, _P, _I, _P]),
    "nvs_sandwich_norm": (c_int, [_P, _P, _F, _P, _F, _P, _P, _L, _P, _F, _I, _I, _F, _P, _P, _P]),
    "nvs_gated_memory_scan_workspace": (c_int64, [_I, _I, _I, _I, _L]),
    "nvs_gated_memory_scan": (c_int, [_P, _L, _L, _L, _L, _L, _L, _I, _P, _P, _F, _F, _I, _I, _I, _P, _P, _P, _I, _L, _L, _P, _P, _P, _P, _P,
                                      _L, _P]),
    "nvs_moe_table_route": (c_int, [_P, _P, _L, _I, _F, _P, _P, _P]),
    "nvs_rglru_scan_workspace": (c_int64, [_I, _I, _L]),
    "nvs_rglru_gates": (c_int, [_P, _P, _P, _P, _I, _F, _I, _I, _L, _P, _P]),
    "nvs_rglru_scan": (c_int, [_P, _P, _P, _L, _I, _P, _F, _I, _I, _P, _P, _P, _I, _L, _L, _P, _P, _P, _L, _P]),
    "nvs_rglru_scan_pairs": (c_int, [_P, _P, _L, _I, _I, _P, _P, _P, _I, _L, _L, _P, _P, _P, _L, _P]),
    "nvs_ssd_scan_workspace": (c_int64, [_I, _I, _I, _I, _L]),
    "nvs_ssd_scan": (c_int, [_P, _P, _L, _L, _I, _P, _P, _P, _I, _I, _I, _I, _P, _P, _P, _I, _L, _L, _P, _P, _P, _L, _P]),
    "nvs_decay_scan": (c_int, [_P, _L, _L, _L, _L, _I, _P, _I, _I, _I, _P, _P, _P, _I, _L, _L, _P, _P, _P, _L, _P]),
    "nvs_gated_group_norm": (c_int, [_P, _P, _L, _I, _P, _I, _I, _I, _F, _I, _L, _P, _P, _P]),
    "nvs_delta_scan": (c_int, [_P, _L, _P, _L, _L, _L, _P, _L, _I, _P, _P, _F, _I, _I, _I, _I, _I, _P, _P, _P, _I, _L, _L, _P, _P, _P]),
    "nvs_delta_force": (None, [_I]),
    "nvs_embed_norm": (c_int, [_P, _I, _P, _L, _I, _P, _F, _P, _P]),
    "nvs_shift_norm": (c_int, [_P, _P, _P, _P, _P, _I, _P, _P, _P, _P, _I, _L, _I, _F, _P, _P, _P, _P]),
    "nvs_gated_lookup": (c_int, [_P, _L, _P, _L, _L, _I, _P, _I, _L, _P, _P]),
    "nvs_qk_rows": (c_int, [_P, _L, _I, _P, _P, _L, _I, _P, _F, _I, _I, _I, _I, _P, _P, _P, _I, _L, _P, _P, _P, _I, _I, _P, _L, _P, _P, _P, _P]),
    "nvs_chosen_norm": (c_int, [_P, _P, _L, _P, _P, _I, _P, _L, _P, _P, _L, _F, _P, _L, _P, _F, _I, _I, _F, _I, _P, _P]),
    "nvs_branch_norm": (c_int, [_P, _P, _P, _L, _P, _P, _I, _I, _L, _P, _P, _I, _F, _P, _P]),
    "nvs_qkv_store": (c_int, [_P, _P, _P, _L, _I, _I, _I, _I, _I, _P, _P, _I, _I, _F, _I, _F, _F, _P, _L, _P, _I, _P, _L, _P, _P, _P]),
    "nvs_pool_rows": (c_int64, [_I, _I]),
    "nvs_pool_blocks": (c_int, [_P, _P, _I, _I, _I, _I, _I, _I, _P, _P, _P, _L, _P, _L, _P, _P, _P]),
    "nvs_knorm_kvstore": (c_int, [_P, _P, _L, _I, _P, _F, _I, _I, _I, _I, _P, _P, _P, _I, _L, _P, _P, _P]),
    "nvs_window_attn_force_scalar": (None, [_I]),
    "nvs_window_attn": (c_int, [_P, _L, _P, _F, _P, _P, _L, _I, _I, _P, _P, _P, _L, _I, _P, _P, _P, _I, _L, _I, _I, _I, _I, _F, _F, _I,
                                _I, _I, _P, _P, _P, _I, _P, _F, _I, _P, _P]),
    "nvs_add_group_norm": (c_int, [_P, _P, _F, _P, _P, _L, _P, _I, _I, _I, _F, _I, _P, _P]),
    "nvs_scale_softcap": (c_int, [_P, _I, _F, _F, _L, _P, _P]),
    "nvs_latent_prep": (c_int, [_P, _L, _I, _I, _I, _P, _P, _I, _I, _I, _P, _P, _P, _I, _I, _F, _F, _I, _P, _P, _P, _L, _P]),
    "nvs_latent_prep_turn": (c_int, [_P, _L, _I, _I, _I, _P, _P, _I, _I, _I, _P, _P, _P, _I, _I, _F, _F, _I, _P, _P, _P, _P, _L, _P]),
    "nvs_latent_prompt_fits": (c_int, [_L, _I, _I, _I]),
    "nvs_latent_prompt": (c_int, [_P, _L, _P, _P, _P, _I, _I, _P, _L, _P, _P, _P, _L, _I, _P, _P, _I, _L, _I, _F, _I, _P, _P]),
    "nvs_latent_heads": (c_int, [_P, _L, _I, _P, _I, _I, _I, _P, _L, _I, _I, _I, _I, _I, _P, _L, _P]),
    "nvs_rotate_heads": (c_int, [_P, _L, _I, _P, _L, _I, _I, _I, _I, _P, _P, _I, _I, _F, _L, _P]),
    "nvs_glu_act": (c_int, [_P, _L, _I, _I, _I, _F, _F, _L, _P, _P]),
    "nvs_linear_rows": (c_int, [_P, _L, _P, _P, _I, _L, _I, _I, _I, _F, _F, _P, _L, _P]),
    "nvs_moe_route": (c_int, [_P, _L, _P, _L, _I, _I, _I, _I, _F, _I, _I, _P, _P, _P]),
    "nvs_moe_router": (c_int, [_P, _L, _I, _P, _P, _I, _I, _P, _L, _I, _I, _I, _I, _F, _I, _I, _P, _P, _P, _P, _L, _P]),
    "nvs_moe_router_workspace": (c_int64, [_L, _I, _I, _I]),
    "nvs_moe_rows": (c_int64, [_L, _I, _I]),
    "nvs_moe_plan": (c_int, [_P, _L, _I, _I, _I, _P, _P, _P, _P]),
    "nvs_moe_plan_scratch": (c_int64, [_L, _I]),
    "nvs_moe_plan_wide": (c_int, [_P, _L, _I, _I, _I, _P, _P, _P, _P, _L, _P]),
    "nvs_silu_linear": (c_int, [_P, _L, _P, _I, _I, _L, _I, _P, _L, _P]),
    "nvs_linear_tiles": (c_int, [_P, _L, _P, _P, _I, _I, _L, _P, _L, _P]),
    "nvs_moe_gemm": (c_int, [_P, _L, _P, _I, _I, _I, _I, _P, _P, _L, _I, _P, _L, _P]),
    "nvs_moe_force_plain": (None, [_I]),
    "nvs_moe_combine": (c_int, [_P, _L, _P, _P, _I, _P, _L, _P, _P, _L, _I, _L, _I, _P, _P, _P]),
}

_lib = None


class NvsError(RuntimeError):
    pass


def load_library() -> ctypes.CDLL:
    """Load libnvl_seq.so, building it first when the checkout has none (or an older one than its sources)."""
    global _lib
    if _lib is not None:
        return _lib
    path = _build.build_seq()
    lib = ctypes.CDLL(path)
    for name, (restype, argtypes) in SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype, fn.argtypes = restype, argtypes
    if lib.nvs_abi_version() != ABI_VERSION:
        raise NvsError(f"libnvl_seq.so ABI version {lib.nvs_abi_version()} != binding version {ABI_VERSION}; rebuild")
    if os.environ.get("NVL_ATTN_SCALAR") == "1":      # A/B switch: bf16 windowed attention on the scalar kernel too
        lib.nvs_window_attn_force_scalar(1)
    elif os.environ.get("NVL_ATTN_NO_LDS") == "1":    # ... or on the matrix cores without the LDS-shared K / V tiles
        lib.nvs_window_attn_force_scalar(2)
    elif os.environ.get("NVL_ATTN_UNPACKED") == "1":  # ... or never with heads in the query tiles of single-token steps
        lib.nvs_window_attn_force_scalar(3)
    _lib = lib
    return lib


def load_if_built() -> bool:
    """For a model that can do without this library (qwen3): is it loaded now? It is if it is there as its sources have it; nothing is built."""
    if _lib is None and _build.seq_is_fresh():
        load_library()
    return _lib is not None


def loaded() -> bool:
    return _lib is not None


def _check(rc: int) -> None:
    if rc != 0:
        raise NvsError(f"nvs error {rc}: {_lib.nvs_last_error().decode()}")


def _stream() -> int:
    # (the handle alone: building a Stream object around it took 6 of a launch's 25 us on the host)
    return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device())


def _code(t: torch.Tensor) -> int:
    if t.dtype == torch.bfloat16:
        return 0
    if t.dtype == torch.float32:
        return 1
    raise NvsError(f"unsupported activation dtype {t.dtype} (bfloat16 or float32)")


def _ptr(t: torch.Tensor | None) -> int | None:
    if t is None:
        return None
    if not t.is_cuda:
        raise NvsError("device (HIP) tensors only; the hot path has no CPU fallback")
    return t.data_ptr()


def _same(code_of: torch.Tensor, *others: torch.Tensor | None) -> int:
    for o in others:
        if o is not None and o.dtype != code_of.dtype:
            raise NvsError(f"dtype mismatch: {o.dtype} beside {code_of.dtype}")
    return _code(code_of)


class Portions:
    """Device-side description of a step's packed portions (see include/nvl_seq.h): cu_q [nseq + 1], ctx0 [nseq],
    slot [nseq], tseq [n], all int32."""
    __slots__ = ("cu_q", "ctx0", "slot", "tseq", "nseq", "n", "max_q")

    def __init__(self, cu_q, ctx0, slot, tseq, nseq: int, n: int, max_q: int = 0):
        self.cu_q, self.ctx0, self.slot, self.tseq, self.nseq, self.n = cu_q, ctx0, slot, tseq, nseq, n
        self.max_q = max_q or n                        # the longest portion (a host-side bound; n when unknown)
        for t in (cu_q, ctx0, slot, tseq):
            assert t.dtype == torch.int32 and t.is_cuda and t.is_contiguous()
        assert cu_q.numel() >= nseq + 1 and ctx0.numel() >= nseq and slot.numel() >= nseq and tseq.numel() >= n


@_launch
def embed_sinusoid(table, ids, pos, scale: float, base: float, x: torch.Tensor, xh: torch.Tensor | None):
    lib = load_library()
    n, width = ids.numel(), table.shape[1]
    assert x.dtype == torch.float32 and x.shape == (n, width) and x.is_contiguous() and table.is_contiguous()
    assert ids.dtype == torch.int64 and pos.dtype == torch.int64 and pos.numel() == n
    assert xh is None or (xh.shape == x.shape and xh.is_contiguous())
    _check(lib.nvs_embed_sinusoid(_ptr(table), _same(table, xh), _ptr(ids), _ptr(pos), n, width, scale, base, _ptr(x),
                                  _ptr(xh), _stream()))


@_launch
def norm_residual(x: torch.Tensor, m: torch.Tensor, g: torch.Tensor, eps: float, xh: torch.Tensor | None,
                  m2: torch.Tensor | None = None, w1: torch.Tensor | None = None, w2: torch.Tensor | None = None):
    """x += g * rms(m), or with a second branch x += g * rms((rms(m) w1 + rms(m2) w2) / 2)."""
    lib = load_library()
    n, width = x.shape
    assert x.dtype == torch.float32 and x.is_contiguous() and m.shape == x.shape and m.is_contiguous()
    assert m2 is None or (m2.shape == x.shape and m2.is_contiguous() and w1.numel() == width and w2.numel() == width)
    assert xh is None or (xh.shape == x.shape and xh.is_contiguous())
    _check(lib.nvs_norm_residual(_ptr(m), _ptr(m2), _ptr(w1), _ptr(w2), _ptr(g), _same(m, m2, w1, w2, g, xh), n, width, eps,
                                 _ptr(x), _ptr(xh), _stream()))


@_launch
def scalar_norm_rows(x: torch.Tensor, rows: torch.Tensor | None, nrows: int, g: torch.Tensor, eps: float, out: torch.Tensor):
    lib = load_library()
    assert x.dtype == torch.float32 and x.is_contiguous() and out.is_contiguous() and out.shape == (nrows, x.shape[1])
    assert rows is None or (rows.dtype == torch.int32 and rows.numel() >= nrows)
    assert rows is not None or nrows <= x.shape[0]
    _check(lib.nvs_scalar_norm_rows(_ptr(x), _ptr(rows), nrows, x.shape[1], _ptr(g), _same(out, g), eps, _ptr(out), _stream()))


@_launch
def xielu(z: torch.Tensor, pq: torch.Tensor, beta: float = 0.5) -> torch.Tensor:
    """In place."""
    lib = load_library()
    assert z.is_contiguous() and pq.numel() == 2
    _check(lib.nvs_xielu(_ptr(z), _ptr(pq), beta, _same(z, pq), z.numel(), _ptr(z), _stream()))
    return z


@_launch
def causal_conv(inp: torch.Tensor, w: torch.Tensor, b: torch.Tensor | None, act: int, por: Portions, state: torch.Tensor,
                out: torch.Tensor):
    """inp: [n, channels] view (unit column stride) of a projection output; state [nslots, taps - 1, channels] fp32; out 32-bit or
    of inp's type."""
    lib = load_library()
    channels, taps = w.shape
    assert inp.shape == (por.n, channels) and inp.stride(1) == 1 and w.is_contiguous()
    assert state.dtype == torch.float32 and state.is_contiguous() and tuple(state.shape[1:]) == (taps - 1, channels)
    assert out.dtype in (torch.float32, inp.dtype) and out.is_contiguous() and out.shape == (por.n, channels)
    _check(lib.nvs_causal_conv(_ptr(inp), inp.stride(0), _same(inp, w, b), _ptr(w), _ptr(b), channels, taps, act, _ptr(por.cu_q),
                               _ptr(por.ctx0), _ptr(por.slot), _ptr(por.tseq), por.nseq, por.n, _ptr(state), _ptr(out), _code(out), _stream()))


@_launch
def rglru_gates(u: torch.Tensor, w: torch.Tensor, bias: torch.Tensor, lam: torch.Tensor, c: float, blocks: int) -> torch.Tensor:
    """u [n, channels], w [blocks, 128, 256], bias [blocks, 1, 256], all 32-bit -> pairs [n, channels, 2] for rglru_scan: log a and the added term."""
    lib = load_library()
    n, channels = u.shape
    assert u.dtype == w.dtype == bias.dtype == torch.float32 and u.is_contiguous() and w.is_contiguous() and bias.is_contiguous()
    assert w.shape == (blocks, 128, 256) and bias.numel() == blocks * 256 and channels == blocks * 128 and lam.numel() == channels and lam.is_contiguous()
    pairs = torch.empty(n, channels, 2, dtype=torch.float32, device=u.device)
    _check(lib.nvs_rglru_gates(_ptr(u), _ptr(w), _ptr(bias), _ptr(lam), _code(lam), c, channels, blocks, n, _ptr(pairs), _stream()))
    return pairs


@_launch
def rglru_scan(gates: torch.Tensor, u: torch.Tensor | None, ypre: torch.Tensor, lam: torch.Tensor, c: float, blocks: int, por: Portions,
               S: torch.Tensor, out: torch.Tensor):
    """gates [blocks, n, 2 bw] are the pre-activations, u [n, channels] the input; u None: gates are rglru_gates' pairs."""
    lib = load_library()
    n, channels = out.shape
    bw = channels // blocks
    assert n == por.n and gates.dtype == torch.float32 and gates.is_contiguous() and gates.shape == ((n, channels, 2) if u is None else (blocks, n, 2 * bw))
    assert u is None or u.dtype == torch.float32 and u.is_contiguous() and u.shape == (n, channels)
    assert ypre.shape == (n, channels) and ypre.stride(1) == 1
    assert S.dtype == torch.float32 and S.is_contiguous() and S.shape[1] == channels and lam.numel() == channels
    assert out.shape == (n, channels) and out.is_contiguous()
    need = 0 if torch.cuda.is_current_stream_capturing() else lib.nvs_rglru_scan_workspace(channels, por.nseq, por.max_q)
    ws = torch.empty(need, dtype=torch.float32, device=out.device) if need else None
    if u is None:
        _check(lib.nvs_rglru_scan_pairs(_ptr(gates), _ptr(ypre), ypre.stride(0), _same(ypre, lam, out), channels, _ptr(por.cu_q), _ptr(por.ctx0), _ptr(por.slot),
                                        por.nseq, n, por.max_q, _ptr(S), _ptr(out), _ptr(ws), need, _stream()))
        return
    _check(lib.nvs_rglru_scan(_ptr(gates), _ptr(u), _ptr(ypre), ypre.stride(0), _same(ypre, lam, out), _ptr(lam), c, channels,
                              blocks, _ptr(por.cu_q), _ptr(por.ctx0), _ptr(por.slot), por.nseq, n, por.max_q, _ptr(S), _ptr(out), _ptr(ws), need,
                              _stream()))


@_launch
def ssd_scan(xbc: torch.Tensor, proj: torch.Tensor, dt_col: int, dt_bias, A_log, D, heads: int, P: int, N: int, G: int,
             por: Portions, S: torch.Tensor, y: torch.Tensor):
    lib = load_library()
    n = por.n
    inner = heads * P
    assert xbc.dtype == torch.float32 and xbc.is_contiguous() and xbc.shape == (n, inner + 2 * G * N)
    assert proj.shape[0] == n and proj.stride(1) == 1 and dt_col + heads <= proj.shape[1]
    assert S.dtype == torch.float32 and S.is_contiguous() and tuple(S.shape[1:]) == (heads, P, N)
    assert y.dtype == torch.float32 and y.is_contiguous() and y.shape == (n, inner)
    assert dt_bias.numel() == heads and A_log.numel() == heads and D.numel() == heads
    need = 0 if torch.cuda.is_current_stream_capturing() else lib.nvs_ssd_scan_workspace(heads, P, N, por.nseq, por.max_q)
    ws = torch.empty(need, dtype=torch.float32, device=xbc.device) if need else None
    _check(lib.nvs_ssd_scan(_ptr(xbc), _ptr(proj), proj.stride(0), dt_col, _same(proj, dt_bias, A_log, D), _ptr(dt_bias),
                            _ptr(A_log), _ptr(D), heads, P, N, G, _ptr(por.cu_q), _ptr(por.ctx0), _ptr(por.slot), por.nseq, n,
                            por.max_q, _ptr(S), _ptr(y), _ptr(ws), need, _stream()))


@_launch
def gated_group_norm(y: torch.Tensor, z: torch.Tensor, w: torch.Tensor, groups: int, eps: float, out: torch.Tensor,
                     norm_first: bool = False, den: torch.Tensor | None = None, silu: bool = False):
    """out = group_rms(y * silu(z)) * w, or with norm_first group_rms(y) * w * sigmoid(z) (silu: * silu(z)); den [n, groups] (32-bit,
    norm_first only): group g of row t is divided by den[t, g] before anything else. w has an entry per column, or, shared by the
    groups, per column of a group."""
    lib = load_library()
    n, inner = y.shape
    assert y.dtype == torch.float32 and y.is_contiguous() and z.shape == (n, inner) and z.stride(1) == 1
    assert w.numel() in (inner, inner // groups) and out.shape == (n, inner) and out.is_contiguous() and (norm_first or not silu)
    assert den is None or (norm_first and den.dtype == torch.float32 and den.shape == (n, groups) and den.is_contiguous())
    _check(lib.nvs_gated_group_norm(_ptr(y), _ptr(z), z.stride(0), _same(z, w, out), _ptr(w), w.numel(), inner, groups, eps,
                                    2 if silu else int(norm_first), n,
                                    _ptr(den), _ptr(out), _stream()))


def _rotation(rot_freq: torch.Tensor | None) -> int:
    if rot_freq is None:
        return 0
    assert rot_freq.dtype == torch.float32 and rot_freq.is_contiguous() and rot_freq.is_cuda
    return 2 * rot_freq.numel()


@_launch
def knorm_kvstore(k: torch.Tensor, v: torch.Tensor, knorm: torch.Tensor | None, eps: float, G: int, d: int, dv: int,
                  block_size: int, slots: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor,
                  pos: torch.Tensor | None = None, rot_freq: torch.Tensor | None = None):
    """k [n, G*d], v [n, G*dv]: column ranges of ONE projection output (same row stride). v_cache has the shape
    [pages * block_size, G, dv] but is laid out [page][G][dv][block_size] (see include/nvl_seq.h)."""
    assert k_cache.shape[0] % block_size == 0
    lib = load_library()
    n = k.shape[0]
    assert k.shape == (n, G * d) and v.shape == (n, G * dv) and k.stride(1) == 1 and v.stride(1) == 1 and k.stride(0) == v.stride(0)
    assert slots.dtype == torch.int32 and slots.numel() >= n
    assert k_cache.is_contiguous() and v_cache.is_contiguous()
    assert tuple(k_cache.shape[1:]) == (G, d) and tuple(v_cache.shape[1:]) == (G, dv)
    assert rot_freq is None or (pos is not None and pos.dtype == torch.int64 and pos.numel() >= n and pos.is_contiguous())
    _check(lib.nvs_knorm_kvstore(_ptr(k), _ptr(v), k.stride(0), _same(k, v, knorm, k_cache, v_cache), _ptr(knorm), eps, G, d, dv,
                                 block_size, _ptr(slots), _ptr(pos) if rot_freq is not None else None, _ptr(rot_freq),
                                 _rotation(rot_freq), n, _ptr(k_cache), _ptr(v_cache), _stream()))


@_launch
def qkv_store(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, H: int, G: int, d: int, dv: int, block_size: int, slots: torch.Tensor, k_cache,
              v_cache, pos: torch.Tensor | None, rot: "Rotation | None", unit: bool, eps: float, q_scale: float,
              first: torch.Tensor | None = None, mix: torch.Tensor | None = None):
    """q [n, H*d], k [n, G*d], v [n, G*dv]: column ranges of ONE projection output. Queries and keys are rotated, then (unit) divided by their
    root mean square per head; queries, times q_scale, are rewritten in place, keys and values stored. first [n, G*dv] and mix (one 32-bit
    number): the values stored are (1 - mix) v + mix first."""
    lib = load_library()
    n = q.shape[0]
    assert q.shape == (n, H * d) and k.shape == (n, G * d) and v.shape == (n, G * dv) and q.stride(1) == k.stride(1) == v.stride(1) == 1
    assert q.stride(0) == k.stride(0) == v.stride(0) and slots.dtype == torch.int32 and slots.numel() >= n
    assert k_cache.is_contiguous() and v_cache.is_contiguous() and k_cache.shape[0] % block_size == 0
    assert tuple(k_cache.shape[1:]) == (G, d) and tuple(v_cache.shape[1:]) == (G, dv)
    assert rot is None or (pos is not None and pos.dtype == torch.int64 and pos.numel() >= n and pos.is_contiguous() and rot.dims <= d)
    assert first is None or (first.shape == v.shape and first.stride(1) == 1 and mix.dtype == torch.float32 and mix.numel() == 1)
    _check(lib.nvs_qkv_store(_ptr(q), _ptr(k), _ptr(v), q.stride(0), _same(q, k, v, first, k_cache, v_cache), H, G, d, dv,
                             _ptr(pos) if rot else None, _ptr(rot.freq) if rot else None, rot.dims if rot else 0, int(rot.halves) if rot else 0,
                             rot.mag if rot else 1.0, int(unit), eps, q_scale, _ptr(first), first.stride(0) if first is not None else 0,
                             _ptr(mix) if first is not None else None, block_size, _ptr(slots), n, _ptr(k_cache), _ptr(v_cache), _stream()))


@_launch
def window_attn(q: torch.Tensor, qnorm: torch.Tensor | None, eps: float, gate: torch.Tensor | None, k_cache, v_cache,
                block_tables: torch.Tensor, block_size: int, por: Portions, H: int, G: int, d: int, dv: int, scale: float,
                window: int, out: torch.Tensor, chunk: int = 0, rot_freq: torch.Tensor | None = None, gate_per_head: bool = False,
                sink: torch.Tensor | None = None, q_temp: tuple[float, int] | None = None, q_row: torch.Tensor | None = None,
                softcap: float = 0.0, pool: int = 0, pool_k: torch.Tensor | None = None, pool_v: torch.Tensor | None = None):
    """window > 0: the last `window` positions; chunk > 0: the query's own block of `chunk` positions; neither: causal.
    rot_freq [r / 2] (32-bit): the first r entries of every query head turn in interleaved pairs by position * rot_freq.
    gate [n, H * dv], or [n, H] with gate_per_head: out *= sigmoid(gate). sink [H] (32-bit): head h's softmax denominator also holds
    exp(sink[h]). q_temp (coef, every): the query at position p is multiplied by 1 + coef * ln(floor((p + 1) / every) + 1).
    q_row [n] (32-bit, from qk_rows): qnorm [H * d] belongs to the whole projection and row t's factor is q_row[t]. softcap > 0:
    scores become softcap * tanh(score / softcap). pool > 0: a query also sees the mean key and value (pool_blocks) of every
    block of `pool` positions that lies wholly before its window."""
    lib = load_library()
    assert q_row is None or (q_row.dtype == torch.float32 and q_row.numel() == por.n and qnorm is not None and qnorm.numel() == H * d)
    assert not pool or (pool_k.is_contiguous() and pool_v.is_contiguous() and window > 0)
    n = por.n
    assert q.shape == (n, H * d) and q.stride(1) == 1 and out.shape == (n, H * dv) and out.is_contiguous()
    assert gate is None or (gate.shape == (n, H if gate_per_head else H * dv) and gate.stride(1) == 1)
    assert block_tables.dtype == torch.int32 and block_tables.stride(1) == 1 and block_tables.shape[0] >= por.nseq
    assert tuple(k_cache.shape[1:]) == (G, d) and tuple(v_cache.shape[1:]) == (G, dv)
    assert sink is None or (sink.dtype == torch.float32 and sink.numel() == H and sink.is_contiguous() and sink.is_cuda)
    qt_coef, qt_every = (float(q_temp[0]), int(q_temp[1])) if q_temp else (0.0, 0)
    _check(lib.nvs_window_attn(_ptr(q), q.stride(0), _ptr(qnorm), eps, _ptr(q_row), _ptr(gate), gate.stride(0) if gate is not None else 0,
                               int(gate_per_head), _same(q, qnorm, gate, k_cache, v_cache, out), _ptr(k_cache), _ptr(v_cache), _ptr(block_tables),
                               block_tables.stride(0), block_size, _ptr(por.cu_q), _ptr(por.ctx0), _ptr(por.tseq), por.nseq, n, H,
                               G, d, dv, scale, softcap, window, chunk, pool, _ptr(pool_k), _ptr(pool_v), _ptr(rot_freq), _rotation(rot_freq),
                               _ptr(sink), qt_coef, qt_every, _ptr(out), _stream()))


@_launch
def qk_rows(q: torch.Tensor, k: torch.Tensor | None, v: torch.Tensor | None, knorm: torch.Tensor | None, eps: float, G: int, d: int, dv: int,
            block_size: int, slots: torch.Tensor, k_cache, v_cache, pos: torch.Tensor, rot_freq: torch.Tensor | None, por: Portions,
            block_tables: torch.Tensor, pool: int = 0, pool_k: torch.Tensor | None = None, pool_v: torch.Tensor | None = None) -> torch.Tensor:
    """Norm over whole projections: returns the factors [n] of the query rows; with k / v (column ranges of one projection) the key
    rows are normed, rotated and stored with the values, and with `pool` the blocks that end in this step are averaged."""
    lib = load_library()
    n = q.shape[0]
    q_row = torch.empty(n, dtype=torch.float32, device=q.device)
    assert q.stride(1) == 1 and pos.dtype == torch.int64 and pos.numel() >= n and pos.is_contiguous() and slots.dtype == torch.int32
    single = por.n == por.nseq                        # one token per portion: the store's workgroups finish the blocks themselves
    if k is not None:
        assert k.shape == (n, G * d) and v.shape == (n, G * dv) and k.stride(1) == 1 and v.stride(1) == 1 and k.stride(0) == v.stride(0)
        assert knorm.numel() == G * d and k_cache.is_contiguous() and v_cache.is_contiguous() and k_cache.shape[0] % block_size == 0
        assert tuple(k_cache.shape[1:]) == (G, d) and tuple(v_cache.shape[1:]) == (G, dv)
    _check(lib.nvs_qk_rows(_ptr(q), q.stride(0), q.shape[1], _ptr(k), _ptr(v), k.stride(0) if k is not None else 0, _same(q, k, v, knorm),
                           _ptr(knorm), eps, G, d, dv, block_size, _ptr(slots), _ptr(pos), _ptr(rot_freq), _rotation(rot_freq), n, _ptr(q_row),
                           _ptr(k_cache), _ptr(v_cache), pool, int(single), _ptr(block_tables), block_tables.stride(0), _ptr(por.tseq),
                           _ptr(pool_k), _ptr(pool_v), _stream()))
    if k is not None and pool and not single:
        pool_blocks(k_cache, v_cache, G, d, dv, block_size, pool, slots, pos, block_tables, por, pool_k, pool_v)
    return q_row


def pool_rows(block_size: int, pool: int) -> int:
    """Blocks of `pool` tokens that a page of block_size tokens has room for (whole units of 8)."""
    return -(-block_size // (8 * pool)) * 8


@_launch
def pool_blocks(k_cache, v_cache, G: int, d: int, dv: int, block_size: int, pool: int, slots: torch.Tensor, pos: torch.Tensor,
                block_tables: torch.Tensor, por: Portions, pool_k: torch.Tensor, pool_v: torch.Tensor):
    """Means of the cached keys / values over the blocks of `pool` positions that end in this step."""
    lib = load_library()
    rows = pool_rows(block_size, pool) * (k_cache.shape[0] // block_size)
    assert pool_k.is_contiguous() and pool_k.numel() == rows * G * d and pool_v.is_contiguous() and pool_v.numel() == rows * G * dv
    assert pos.dtype == torch.int64 and slots.dtype == torch.int32 and block_tables.dtype == torch.int32
    _check(lib.nvs_pool_blocks(_ptr(k_cache), _ptr(v_cache), _same(k_cache, v_cache, pool_k, pool_v), G, d, dv, block_size, pool, _ptr(slots),
                               _ptr(pos), _ptr(block_tables), block_tables.stride(0), _ptr(por.tseq), por.n, _ptr(pool_k), _ptr(pool_v),
                               _stream()))


@_launch
def embed_norm(table: torch.Tensor, ids: torch.Tensor, w: torch.Tensor, eps: float, x: torch.Tensor):
    """x (32-bit) = rms(table[ids]) * w."""
    lib = load_library()
    n, width = ids.numel(), table.shape[1]
    assert x.dtype == torch.float32 and x.shape == (n, width) and x.is_contiguous() and table.is_contiguous() and ids.dtype == torch.int64
    _check(lib.nvs_embed_norm(_ptr(table), _same(table, w), _ptr(ids), n, width, _ptr(w), eps, _ptr(x), _stream()))


@_launch
def shift_norm(x: torch.Tensor, a: torch.Tensor | None, wa: torch.Tensor | None, w: torch.Tensor, mu: torch.Tensor, eps: float, por: Portions,
               state: torch.Tensor, out: torch.Tensor) -> torch.Tensor:
    """y = x + a (wa None) or x + rms(a) * wa; h = rms(y) * w; out = h + (h of the previous token - h) * mu, with the last h of every
    sequence kept in state [nslots, width]. Returns y (x itself when there is nothing to add)."""
    lib = load_library()
    n, width = x.shape
    assert n == por.n and x.dtype == torch.float32 and x.is_contiguous() and out.shape == x.shape and out.is_contiguous()
    assert a is None or (a.shape == x.shape and a.is_contiguous())
    assert w.numel() == width and mu.numel() == width and (wa is None or wa.numel() == width)
    assert state.dtype == torch.float32 and state.is_contiguous() and tuple(state.shape[1:]) == (width,)
    y = torch.empty_like(x) if a is not None else x
    _check(lib.nvs_shift_norm(_ptr(x), _ptr(a), _ptr(wa), _ptr(w), _ptr(mu), _same(out, a, wa, w, mu), _ptr(por.cu_q), _ptr(por.ctx0),
                              _ptr(por.slot), _ptr(por.tseq), por.nseq, n, width, eps, _ptr(state), _ptr(y), _ptr(out), _stream()))
    return y


@_launch
def gated_lookup(z: torch.Tensor, table: torch.Tensor, col0: int, ids: torch.Tensor) -> torch.Tensor:
    """gelu_tanh(z) * table[ids, col0 : col0 + dim], z [n, dim]."""
    lib = load_library()
    n, dim = z.shape
    assert z.stride(1) == 1 and table.is_contiguous() and ids.dtype == torch.int64 and ids.numel() == n
    out = torch.empty(n, dim, dtype=z.dtype, device=z.device)
    _check(lib.nvs_gated_lookup(_ptr(z), z.stride(0), _ptr(table), table.shape[1], col0, _same(z, table), _ptr(ids), dim, n, _ptr(out), _stream()))
    return out


@_launch
def delta_scan(qkv: torch.Tensor, gates: torch.Tensor, b_col: int, a_col: int, decays: torch.Tensor | None, A_log: torch.Tensor,
               dt_bias: torch.Tensor, q_scale: float, heads: int, G: int, dk: int, dv: int, por: Portions, S: torch.Tensor, y: torch.Tensor):
    """The gated delta rule (see include/nvl_seq.h) on qkv [n, 2 G dk + heads dv]; beta from columns b_col of `gates`; one decay per head
    from columns a_col of `gates` (decays None), or per head and key channel from columns a_col of `decays`. S [nslots, heads, dv, dk]."""
    lib = load_library()
    n = por.n
    assert qkv.shape == (n, 2 * G * dk + heads * dv) and qkv.stride(1) == 1 and gates.shape[0] == n and gates.stride(1) == 1
    assert decays is None or (decays.shape[0] == n and decays.stride(1) == 1)
    assert A_log.dtype == torch.float32 and A_log.numel() == heads and dt_bias.dtype == torch.float32
    assert dt_bias.numel() == (heads if decays is None else heads * dk) and dt_bias.is_contiguous()
    assert S.dtype == torch.float32 and S.is_contiguous() and tuple(S.shape[1:]) == (heads, dv, dk)
    assert y.dtype == torch.float32 and y.is_contiguous() and y.shape == (n, heads * dv)
    _check(lib.nvs_delta_scan(_ptr(qkv), qkv.stride(0), _ptr(gates), gates.stride(0), b_col, a_col, _ptr(decays),
                              decays.stride(0) if decays is not None else 0, _same(qkv, gates, decays), _ptr(A_log), _ptr(dt_bias), q_scale,
                              int(decays is not None), heads, G, dk, dv, _ptr(por.cu_q), _ptr(por.ctx0), _ptr(por.slot), por.nseq, n, por.max_q,
                              _ptr(S), _ptr(y), _stream()))


class ChosenRows:
    """A routed layer's output before it is summed (RoutedExperts.parts, and the layer's input for pass-through choices). add_group_norm and sandwich_norm take it in a's
    place and sum it on the way where they can. MI355X, us, sum and norm as launches of their own / in one, 16-bit rows: 64 rows of 1,024, three choices 4.9 / 3.5;
    four choices, 2,000 rows of 1,024 10.3 / 7.3, 14,200 of 1,024 52 / 41, of 2,048 131 / 104; three, 13,550 of 4,096 225 / 176."""
    __slots__ = ("h", "rows", "plan", "wts", "shared", "gate")

    def __init__(self, h: torch.Tensor, rows: torch.Tensor, plan: "MoePlan", wts: torch.Tensor, shared: torch.Tensor | None, gate: torch.Tensor | None):
        self.h, self.rows, self.plan, self.wts, self.shared, self.gate = h, rows, plan, wts, shared, gate

    def sum(self) -> torch.Tensor:
        out = torch.empty(self.h.shape, dtype=self.h.dtype, device=self.h.device)
        moe_combine(self.rows, self.plan, self.wts, self.h, self.shared, self.gate, out)
        return out

    def fits(self, x: torch.Tensor, *others: torch.Tensor | None) -> bool:
        """Whether nvs_chosen_norm takes the rows: whole accesses of four columns, aligned. Few wide rows stay two launches, the sum's spreads a row over several workgroups (a step
        of 70 rows of 4,096, one routed layer: 848 us, 852 in one)."""
        n, width = x.shape
        if n <= 512 and width > 2048 or width % 4 or width > 8192 or self.rows.stride(0) % 4 or self.h.stride(0) % 4:
            return False
        al = 0
        for t in (x, self.rows, self.h, self.shared, *others):
            if t is not None:
                al |= t.data_ptr()
        return al % 16 == 0


def _chosen_norm(x: torch.Tensor, c: ChosenRows, mult: float, wa: torch.Tensor | None, w: torch.Tensor | None, w_off: float, eps: float, center: bool,
                 out: torch.Tensor | None):
    n, width = x.shape
    h, rows, plan, wts, shared, gate = c.h, c.rows, c.plan, c.wts, c.shared, c.gate
    assert x.dtype == torch.float32 and x.is_contiguous() and h.shape == x.shape and h.stride(1) == 1
    assert rows.stride(1) == 1 and rows.shape[1] == width and wts.dtype == torch.float32 and wts.is_contiguous() and wts.shape[0] == n
    assert plan.pair_row.shape == wts.shape and (shared is None or (shared.shape == x.shape and shared.is_contiguous()))
    assert gate is None or (shared is not None and gate.dtype == torch.float32 and gate.shape[0] == n)
    assert out is None or (out.shape == x.shape and out.is_contiguous() and w.numel() == width)
    assert wa is None or wa.numel() == width
    _check(load_library().nvs_chosen_norm(_ptr(x), _ptr(rows), rows.stride(0), _ptr(plan.pair_row), _ptr(wts), wts.shape[1], _ptr(h), h.stride(0), _ptr(shared),
                                          _ptr(gate), gate.stride(0) if gate is not None else 0, mult, _ptr(wa), n, _ptr(w), w_off,
                                          _same(rows, h, shared, wa, w, out), width, eps, int(center), _ptr(out), _stream()))


@_launch
def add_group_norm(x: torch.Tensor, w: torch.Tensor | None, groups: int, eps: float, out: torch.Tensor | None,
                   a: "torch.Tensor | ChosenRows | None" = None, b: torch.Tensor | None = None, a_mult: float = 1.0, center: bool = False):
    """x += a_mult * a + b (in place; a in the activation type, b 32-bit, both optional), then out = group_rms(x) * w (out None:
    adds only; w None: out is the sum itself in the activation type); center: every group's mean is taken off first (layer norm without bias)."""
    lib = load_library()
    if type(a) is ChosenRows:
        weight = w if out is not None else None
        if (groups == 1 or out is None) and b is None and (out is None or w is not None) and a.fits(x, weight, out):
            return _chosen_norm(x, a, a_mult, None, weight, 0.0, eps, center and out is not None, out)
        a = a.sum()
    n, width = x.shape
    assert x.dtype == torch.float32 and x.is_contiguous()
    assert a is None or (a.shape == x.shape and a.is_contiguous())
    assert b is None or (b.shape == x.shape and b.is_contiguous() and b.dtype == torch.float32)
    assert out is None or (out.shape == x.shape and out.is_contiguous() and (w is None or w.numel() == width))
    ref = out if out is not None else a
    assert ref is not None, "nothing to do"
    _check(lib.nvs_add_group_norm(_ptr(x), _ptr(a), a_mult, _ptr(b), None, n, _ptr(w) if out is not None else None, _same(ref, a, w, out),
                                  width, groups, eps, int(center), _ptr(out), _stream()))


@_launch
def group_norm_rows(x: torch.Tensor, rows: torch.Tensor | None, nrows: int, w: torch.Tensor, groups: int, eps: float, out: torch.Tensor,
                    center: bool = False):
    """out[r] = group_rms(x[rows[r]]) * w (rows None: row r); center: as add_group_norm."""
    lib = load_library()
    assert x.dtype == torch.float32 and x.is_contiguous() and out.is_contiguous() and out.shape == (nrows, x.shape[1])
    assert rows is None or (rows.dtype == torch.int32 and rows.numel() >= nrows)
    assert rows is not None or nrows <= x.shape[0]
    _check(lib.nvs_add_group_norm(_ptr(x), None, 1.0, None, _ptr(rows), nrows, _ptr(w), _same(out, w), x.shape[1], groups, eps, int(center),
                                  _ptr(out), _stream()))


@_launch
def sandwich_norm(x: torch.Tensor, a: "torch.Tensor | ChosenRows | None", wa: torch.Tensor | None, w: torch.Tensor | None, eps: float,
                  out: torch.Tensor | None, a2: torch.Tensor | None = None, a_mult: float = 1.0, a2_mult: float = 1.0, w_off: float = 1.0):
    """x += rms(a_mult * a + a2_mult * a2) * (w_off + wa) (in place; a None: no add), then out = rms(x) * (w_off + w) (out None: no
    second norm)."""
    lib = load_library()
    if type(a) is ChosenRows:
        weight = w if out is not None else None
        if a2 is None and wa is not None and a.fits(x, wa, weight, out):
            return _chosen_norm(x, a, a_mult, wa, weight, w_off, eps, False, out)
        a = a.sum()
    n, width = x.shape
    assert x.dtype == torch.float32 and x.is_contiguous()
    assert a is None or (a.shape == x.shape and a.is_contiguous() and wa is not None and wa.numel() == width)
    assert a2 is None or (a is not None and a2.shape == x.shape and a2.is_contiguous())
    assert out is None or (out.shape == x.shape and out.is_contiguous() and w is not None and w.numel() == width)
    ref = out if out is not None else a
    assert ref is not None, "nothing to do"
    _check(lib.nvs_sandwich_norm(_ptr(x), _ptr(a), a_mult, _ptr(a2), a2_mult, _ptr(wa) if a is not None else None, None, n,
                                 _ptr(w) if out is not None else None, w_off, _same(ref, a, a2, wa if a is not None else None,
                                                                                   w if out is not None else None, out), width, eps, None, _ptr(out), _stream()))


@_launch
def offset_norm_rows(x: torch.Tensor, rows: torch.Tensor | None, nrows: int, w: torch.Tensor, eps: float, out: torch.Tensor, w_off: float = 1.0,
                     a: torch.Tensor | None = None, wa: torch.Tensor | None = None):
    """out[r] = rms(x[rows[r]]) * (w_off + w) (rows None: row r); with a and wa: of x[rows[r]] + rms(a[rows[r]]) * (w_off + wa) (x stays)."""
    lib = load_library()
    assert a is None or (rows is not None and a.shape == x.shape and a.is_contiguous() and wa.numel() == x.shape[1])
    sums = torch.empty(nrows, x.shape[1], dtype=torch.float32, device=x.device) if a is not None else None
    assert x.dtype == torch.float32 and x.is_contiguous() and out.is_contiguous() and out.shape == (nrows, x.shape[1])
    assert rows is None or (rows.dtype == torch.int32 and rows.numel() >= nrows)
    assert rows is not None or nrows <= x.shape[0]
    _check(lib.nvs_sandwich_norm(_ptr(x), _ptr(a), 1.0, None, 1.0, _ptr(wa), _ptr(rows), nrows, _ptr(w), w_off, _same(out, w, a, wa), x.shape[1],
                                 eps, _ptr(sums), _ptr(out), _stream()))


@_launch
def branch_norm(x: torch.Tensor, a: torch.Tensor | None, w: torch.Tensor, ls: torch.Tensor | None, eps: float, out: torch.Tensor | None,
                chosen: "tuple | None" = None):
    """x += rms(y) * w * ls (in place; ls None: no scale), y = a (may be None) + with chosen = (rows, plan, weights) of a routed layer the
    weighted sum of every token's choices; out (may be None) receives the new x in the activation type."""
    lib = load_library()
    n, width = x.shape
    rows, plan, wts = chosen if chosen is not None else (None, None, None)
    assert x.dtype == torch.float32 and x.is_contiguous() and w.numel() == width and (ls is None or ls.numel() == width)
    assert a is None or (a.shape == x.shape and a.is_contiguous())
    assert out is None or (out.shape == x.shape and out.is_contiguous())
    top = 0
    if rows is not None:
        top = wts.shape[1]
        assert rows.stride(1) == 1 and rows.shape[1] == width and wts.dtype == torch.float32 and wts.is_contiguous()
        assert wts.shape[0] == n and plan.pair_row.shape == (n, top)
    _check(lib.nvs_branch_norm(_ptr(x), _ptr(a), _ptr(rows), rows.stride(0) if rows is not None else 0, _ptr(plan.pair_row) if plan else None,
                               _ptr(wts), top, _same(w, a, rows, ls, out), n, _ptr(w), _ptr(ls), width, eps, _ptr(out), _stream()))


@_launch
def gated_memory_scan(proj: torch.Tensor, v_col: int, k_col: int, q_col: int, i_col: int, f_col: int, i_bias: torch.Tensor,
                      f_bias: torch.Tensor, cap: float, q_scale: float, heads: int, dk: int, dv: int, por: Portions, S: torch.Tensor,
                      M: torch.Tensor, y: torch.Tensor, den: torch.Tensor):
    """The matrix memory with exponential gates (see include/nvl_seq.h): S [nslots, heads, dv + 1, dk] and M [nslots, heads] are the
    state; y [n, heads * dv] receives the numerators, den [n, heads] the divisors."""
    lib = load_library()
    n = por.n
    assert proj.shape[0] == n and proj.stride(1) == 1 and i_bias.numel() == heads and f_bias.numel() == heads
    assert S.dtype == torch.float32 and S.is_contiguous() and tuple(S.shape[1:]) == (heads, dv + 1, dk)
    assert M.dtype == torch.float32 and M.is_contiguous() and tuple(M.shape[1:]) == (heads,) and M.shape[0] == S.shape[0]
    assert y.dtype == torch.float32 and y.is_contiguous() and y.shape == (n, heads * dv)
    assert den.dtype == torch.float32 and den.is_contiguous() and den.shape == (n, heads)
    need = 0 if torch.cuda.is_current_stream_capturing() else lib.nvs_gated_memory_scan_workspace(heads, dk, dv, por.nseq, por.max_q)
    ws = torch.empty(need, dtype=torch.float32, device=proj.device) if need else None
    _check(lib.nvs_gated_memory_scan(_ptr(proj), proj.stride(0), v_col, k_col, q_col, i_col, f_col, _same(proj, i_bias, f_bias), _ptr(i_bias),
                                     _ptr(f_bias), cap, q_scale, heads, dk, dv, _ptr(por.cu_q), _ptr(por.ctx0), _ptr(por.slot), por.nseq, n,
                                     por.max_q, _ptr(S), _ptr(M), _ptr(y), _ptr(den), _ptr(ws), need, _stream()))


@_launch
def scale_softcap(logits: torch.Tensor, scale: float, cap: float) -> torch.Tensor:
    """32-bit cap * tanh(logits * scale / cap) (cap <= 0: logits * scale)."""
    lib = load_library()
    assert logits.is_contiguous()
    out = torch.empty(logits.shape, dtype=torch.float32, device=logits.device)
    _check(lib.nvs_scale_softcap(_ptr(logits), _code(logits), scale, cap, logits.numel(), _ptr(out), _stream()))
    return out


class Rotation:
    """How the leading `dims` entries of a vector turn with the position: 32-bit frequencies of the pairs (device), the pairing
    ((2i, 2i+1), or (i, i + dims / 2) with `halves`) and a factor on cos and sin."""
    __slots__ = ("freq", "dims", "halves", "mag")

    def __init__(self, freq: torch.Tensor, halves: bool = False, mag: float = 1.0):
        assert freq.dtype == torch.float32 and freq.is_contiguous()
        self.freq, self.dims, self.halves, self.mag = freq, 2 * freq.numel(), bool(halves), float(mag)


@_launch
def latent_prep(proj: torch.Tensor, q_col: int, q_rank: int, q_norm: torch.Tensor, cq: torch.Tensor, eps: float, kv_col: int = -1,
                kv_rank: int = 0, rot_dim: int = 0, kv_norm: torch.Tensor | None = None, pos: torch.Tensor | None = None,
                rot: Rotation | None = None, block_size: int = 0, slots: torch.Tensor | None = None, k_cache: torch.Tensor | None = None,
                v_cache: torch.Tensor | None = None, turn: torch.Tensor | None = None):
    """Norms of the query latent (-> cq [n, q_rank]) and, with kv_col >= 0, of the key/value latent, the rotation of the shared key
    part and the store of both into the paged cache: k_cache [slots, 1, kv_rank + rot_dim], v_cache [slots, 1, kv_rank] (the
    latent again, page-transposed like every value cache). turn [n, rot.dims / 2, 2] 32-bit: receives all tokens' cosines and sines."""
    lib = load_library()
    n = proj.shape[0]
    assert proj.stride(1) == 1 and cq.shape == (n, q_rank) and cq.is_contiguous() and q_norm.numel() == q_rank
    if kv_col >= 0:
        assert kv_norm.numel() == kv_rank and slots.dtype == torch.int32 and slots.numel() >= n
        assert pos.dtype == torch.int64 and pos.numel() >= n and pos.is_contiguous()
        assert k_cache.is_contiguous() and v_cache.is_contiguous() and k_cache.shape[0] % block_size == 0
        assert tuple(k_cache.shape[1:]) == (1, kv_rank + rot_dim) and tuple(v_cache.shape[1:]) == (1, kv_rank)
        assert rot is None or (rot.freq.is_cuda and rot.dims <= rot_dim)
    args = (_ptr(proj), proj.stride(0), _same(proj, q_norm, cq, kv_norm, k_cache, v_cache), q_col, q_rank, _ptr(q_norm),
            _ptr(cq), kv_col, kv_rank, rot_dim, _ptr(kv_norm), _ptr(pos), _ptr(rot.freq) if rot else None,
            rot.dims if rot else 0, int(rot.halves) if rot else 0, rot.mag if rot else 1.0, eps, block_size, _ptr(slots),
            _ptr(k_cache), _ptr(v_cache))
    if turn is None or not turn.numel():
        _check(lib.nvs_latent_prep(*args, n, _stream()))
    else:
        _check(lib.nvs_latent_prep_turn(*args, _ptr(turn), n, _stream()))


_HEAD_SIZES = (64, 128, 192, 256)


def latent_heads_fit(x: torch.Tensor, w: torch.Tensor, K: int, N: int, tail: int = 0) -> bool:
    """Whether latent_heads takes a step of x's rows (K -> N entries per head, `tail` entries behind): what it can take, and of few rows only those that have
    a part behind, whose launch is saved. MI355X, us, a batched product (and the rotation) / here: 16 heads, 128 -> 192 + 64: 16 rows 9.3 / 7.4, 256: 14.5 / 10.5, 4,000:
    29 / 24, 14,000: 95 / 57; 4 heads, 128 -> 256 + 64: 64 rows 8.5 / 10.0, 1,000: 8.5 / 11.2, 14,000: 31 / 26; 16 heads, 192 -> 128: 64 rows 5.4 / 6.5, 1,000: 6.3 / 7.8,
    4,000: 12.4 / 12.8, 14,000: 46 / 29; 32 heads, 4,000: 23 / 19."""
    if x.shape[0] * w.shape[0] < 65536 and not (tail and K * N <= 128 * 192):
        return False
    return (x.is_cuda and x.dtype == w.dtype == torch.bfloat16 and K in _HEAD_SIZES and N in _HEAD_SIZES and (K + tail) % 8 == 0 and (N + tail) % 8 == 0
            and tail % 2 == 0 and w.is_contiguous() and w.data_ptr() % 16 == 0)


@_launch
def latent_heads(x: torch.Tensor, w: torch.Tensor, y: torch.Tensor, turned: bool, tail: int = 0, rot: Rotation | None = None, turn: torch.Tensor | None = None):
    """y[t, a, :N] = W_a x[t, a, :K]: w [H, N, K], with `turned` [H, K, N]. The `tail` entries behind x's K go behind y's N, the leading rot.dims of them turned
    by `turn` (latent_prep)."""
    lib = load_library()
    n, H, K = x.shape[0], x.shape[1], x.shape[2] - tail
    N = y.shape[2] - tail
    assert w.shape == ((H, K, N) if turned else (H, N, K)) and w.is_contiguous() and y.shape[:2] == (n, H) and x.stride(2) == y.stride(2) == 1
    assert rot is None or turn.shape == (n, rot.dims // 2, 2) and turn.is_contiguous() and turn.dtype == torch.float32
    assert x.dtype == w.dtype == y.dtype == torch.bfloat16
    _check(lib.nvs_latent_heads(_ptr(x), x.stride(0), x.stride(1), _ptr(w), int(turned), K, N, _ptr(y), y.stride(0), y.stride(1), H, tail,
                                rot.dims if rot else 0, int(rot.halves) if rot else 0, _ptr(turn), n, _stream()))


def latent_prompt_fit(x: torch.Tensor, uk: torch.Tensor, tail: int, rot: Rotation | None, k_cache: torch.Tensor, v_cache: torch.Tensor, block_size: int, por: Portions) -> bool:
    """Whether latent_prompt takes a step of x's rows: the sizes it is built for, where window_attn would take the same kernel.
    MI355X, whole prompts, us, all calls one by one / the queries' product here / the values' too: width 1,024, one of 17 tokens 790 / 744 / 629, one of 300 947 / 905 / 791, 9 of
    1,100 to 2,048 3270 / 3024 / 2899; width 4,096, 7 of 1,100 to 2,000 6620 / 6367 / 6358."""
    H, d, r = uk.shape
    return (x.is_cuda and x.dtype == uk.dtype == k_cache.dtype == torch.bfloat16 and (d, r, tail) == (128, 192, 64) and uk.is_contiguous()
            and (uk.data_ptr() | k_cache.data_ptr() | v_cache.data_ptr()) % 16 == 0 and (rot is None or rot.dims % 16 == 0)
            and bool(load_library().nvs_latent_prompt_fits(por.n, por.nseq, H, block_size)))


@_launch
def latent_prompt(q: torch.Tensor, uk: torch.Tensor, uv: torch.Tensor | None, rot: Rotation | None, turn: torch.Tensor | None, gate: torch.Tensor | None, k_cache, v_cache,
                  block_tables: torch.Tensor, block_size: int, por: Portions, scale: float, window: int, out: torch.Tensor):
    """latent_heads and window_attn of a step of prompts in one kernel: q [n, H, 128 + 64], uk [H, 128, 192], gate [n, H], out [n, H * 192]. uv [H, 128, 192]: the
    latent_heads behind it too, out [n, H * 128]."""
    lib = load_library()
    n, H = q.shape[0], q.shape[1]
    assert q.shape == (por.n, H, 192) and q.stride(2) == 1 and q.stride(1) == 192 and uk.shape == (H, 128, 192) and uk.is_contiguous()
    assert uv is None or (uv.shape == (H, 128, 192) and uv.is_contiguous())
    assert out.shape == (n, H * (192 if uv is None else 128)) and out.is_contiguous() and (gate is None or (gate.shape == (n, H) and gate.stride(1) == 1))
    assert rot is None or turn.shape == (n, rot.dims // 2, 2) and turn.is_contiguous() and turn.dtype == torch.float32
    assert block_tables.dtype == torch.int32 and block_tables.stride(1) == 1 and block_tables.shape[0] >= por.nseq
    assert tuple(k_cache.shape[1:]) == (1, 256) and tuple(v_cache.shape[1:]) == (1, 192)
    assert _same(q, uk, uv, gate, k_cache, v_cache, out) == _code(q) and q.dtype == torch.bfloat16
    _check(lib.nvs_latent_prompt(_ptr(q), q.stride(0), _ptr(uk), _ptr(uv), _ptr(turn) if rot else None, rot.dims if rot else 0, int(rot.halves) if rot else 0, _ptr(gate),
                                 gate.stride(0) if gate is not None else 0, _ptr(k_cache), _ptr(v_cache), _ptr(block_tables), block_tables.stride(0), block_size, _ptr(por.cu_q), _ptr(por.ctx0), por.nseq,
                                 n, H, scale, window, _ptr(out), _stream()))


@_launch
def rotate_heads(inp: torch.Tensor, out: torch.Tensor, pos: torch.Tensor, rot: Rotation | None):
    """inp, out [n, H, width] views (unit stride along the last axis): out = inp with the leading rot.dims entries of every head rotated."""
    lib = load_library()
    n, H, width = inp.shape
    assert out.shape == inp.shape and inp.stride(2) == 1 and out.stride(2) == 1 and pos.dtype == torch.int64 and pos.numel() >= n
    assert rot is None or rot.dims <= width
    _check(lib.nvs_rotate_heads(_ptr(inp), inp.stride(0), inp.stride(1), _ptr(out), out.stride(0), out.stride(1), _same(inp, out), H, width,
                                _ptr(pos), _ptr(rot.freq) if rot else None, rot.dims if rot else 0, int(rot.halves) if rot else 0,
                                rot.mag if rot else 1.0, n, _stream()))


@_launch
def decay_scan(proj: torch.Tensor, v_col: int, k_col: int, q_col: int, decay: torch.Tensor, heads: int, dk: int, dv: int,
               por: Portions, S: torch.Tensor, y: torch.Tensor):
    """Per head S = decay S + k v^T, y = S^T q on SiLU of the named columns of proj; S [nslots, heads, dv, dk], y [n, heads * dv]."""
    lib = load_library()
    n = por.n
    assert proj.shape[0] == n and proj.stride(1) == 1
    assert decay.dtype == torch.float32 and decay.numel() == heads and decay.is_contiguous()
    assert S.dtype == torch.float32 and S.is_contiguous() and tuple(S.shape[1:]) == (heads, dv, dk)
    assert y.dtype == torch.float32 and y.is_contiguous() and y.shape == (n, heads * dv)
    need = 0 if torch.cuda.is_current_stream_capturing() else lib.nvs_ssd_scan_workspace(heads, dv, dk, por.nseq, por.max_q)
    ws = torch.empty(need, dtype=torch.float32, device=proj.device) if need else None
    _check(lib.nvs_decay_scan(_ptr(proj), proj.stride(0), v_col, k_col, q_col, _code(proj), _ptr(decay), heads, dk, dv, _ptr(por.cu_q),
                              _ptr(por.ctx0), _ptr(por.slot), por.nseq, n, por.max_q, _ptr(S), _ptr(y), _ptr(ws), need, _stream()))


@_launch
def glu_act(gu: torch.Tensor, ff: int, out: torch.Tensor, kind: int = 0, limit: float = 0.0, alpha: float = 1.0):
    """gu [n, 2 ff] = [gate | up] -> out [n, ff]. kind 0: silu(g) u; kind 1: min(g, limit) sigmoid(alpha g) (clamp(u) + 1);
    kind 2: gu [n, ff], no gate: the tanh form of GELU."""
    lib = load_library()
    n = gu.shape[0]
    assert gu.shape[1] == (1 if kind == 2 else 2) * ff and gu.stride(1) == 1 and out.shape == (n, ff) and out.is_contiguous()
    _check(lib.nvs_glu_act(_ptr(gu), gu.stride(0), _same(gu, out), ff, kind, limit, alpha, n, _ptr(out), _stream()))


def _few_rows(x: torch.Tensor, w: torch.Tensor, glu: bool) -> bool:
    """Whether x w^T goes to nvs_linear_rows: whole 128-byte pieces of k, few rows and not too many of w. MI355X, us here / the library's, bf16: 64 rows,
    1024 x 1024 3.6 / 8.6, 1024 x 3072 4.9 / 10.0, 4096 x 1024 4.5 / 8.6, 4096 x 4096 12.3 / 14.7, 6144 x 1024 5.8 / 8.8, 12288 x 2048 13.8 / 12.9,
    24576 x 4096 54.8 / 47.9; 256 rows, 1024 x 1024 4.2 / 8.3, 4096 x 4096 19.5 / 22.2, 6144 x 1024 12.8 / 12.3; 128 rows of it 7.5 / 9.5; 16 rows,
    12288 x 2048 11.7 / 11.6, 32768 x 4096 57.9 / 60.3 (its 268 MB out of memory). The activation on the way saves its launch (4 us and its passes): more is taken. 32-bit: 330 rows,
    1024 x 1024 10.3 / 11.8, 4096 x 1024 33.6 / 41.3, 3084 x 1024 30.9 / 23.8; 512 rows, 1024 x 2048 21.3 / 21.5, 4096 x 1024 42.9 / 36.2."""
    if x.dim() != 2 or w.dim() != 2:
        return False
    (m, k), (n, wide) = x.shape, w.shape
    if wide != k or n == 0 or k == 0 or x.stride(0) < k or x.device != w.device:          # (rows that share entries too: nvs_linear_rows refuses them)
        return False
    if w.dtype == torch.bfloat16:
        if k % 64 or x.stride(0) % 8 or not (m <= 16 or m <= 256 and n <= 4096 or m <= 128 and n <= 6144 or
                                             glu and (m <= 32 or m * n <= 64 * 12288 or m <= 256 and n <= 8192)):
            return False
    elif w.dtype != torch.float32 or k % 32 or x.stride(0) % 4 or not (m <= 16 or m <= 512 and n <= 2048 or m <= 384 and n <= (6144 if glu else 4096)):
        return False
    return w.is_cuda and x.dtype == w.dtype and x.stride(1) == 1 and w.is_contiguous() and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0


def _linear_rows(x: torch.Tensor, w: torch.Tensor, b: torch.Tensor | None, act: int, limit: float, alpha: float, out: torch.Tensor) -> torch.Tensor:
    lib = load_library()
    m, k = x.shape
    _check(lib.nvs_linear_rows(_ptr(x), x.stride(0), _ptr(w), _ptr(b), _same(x, w, b, out), m, out.shape[1], k, act, limit, alpha, _ptr(out),
                               out.stride(0), _stream()))
    return out


TILES_FROM = 768


def tiles_rule(n: int, N: int, K: int) -> bool:
    """Whether x w^T of n rows, N features and K entries each goes to the tiles of 256 rows x 256 features (256 of them are a pass, left-over ones of at most 128 go in
    halves). MI355X, us here / the library's, between the other launches of a prompt step: weights come from memory there, and a product of few tiles that looks 10 % better
    repeated by itself is 20 % worse. What decides is how full the passes are. Not full, here and there: 13,550 rows, 4096 x 4096 329 / 340, 6144 x 4096 478 / 632, 12288 x 4096 912 / 1037,
    4096 x 12288 951 / 1187, 2312 x 1024 74 / 106; 12,285, 6144 x 2048 223 / 319; 3,000, 24576 x 4096 428 / 573. Short reductions: 2,000 rows, 4096 x 256 13 / 19, 3072 x 384 14 / 18.
    Less than a pass leaves compute units idle, or with half a tile each, which wait for their operands: 1,300 rows, 4096 x 2048 39 / 34, x 4096 69 / 55, x 12288 189 / 140; 2,000, 4096 x 3072 60 / 53;
    3,000, 2048 x 6144 108 / 77; 900, 6144 x 1536 35 / 28; at K 1024 not: 2,000, 4096 26 / 27, 8,190, 1024 24 / 27. So with rows that end early in a tile: 1,300, 24576 x 4096 236 / 221 (but 900,
    16384 x 4096 94 / 106). The library is slower at features that are no multiple of 128: 6,600 rows, 1040 x 2048 48 / 44 (two fifths of a pass), 8,190 49 / 51, 12,285 55 / 70; 1824 x 4096, 3,000 rows 68 / 58,
    6,600 93 / 102; 13,550, 656 x 1024 32 / 38. Multiples of 128 that are none of 256 fill its tiles and not these: 640 x 1024, 12,285 rows 31 / 28, 13,550 32 / 37; x 4096 by itself 81 / 56 and 82 / 74.
    Whole passes take as long here and there, 2 to 3 % longer here by themselves (16,380 rows, 4096 x 4096 373 / 366, 24576 x 4096 2206 / 2152, 2048 x 6144 277 / 288), but kernels of both kinds in turn cost each
    other that much, so they are not told apart. Steps of 16,384 rows in ms, all here / whole passes by the library: two layers of Qwen3-8B 9.58 / 9.56, nokipel 4096 11.70 / 11.62, 2048 3.71 / 3.73,
    foduzen 4096 10.88 / 10.84, lobidra 2048 4.47 / 4.51, ligidra 2048 5.06 / 5.11, Qwen3-0.6B 17.19 / 17.04; of 12,288: 7.30 / 7.58, 9.00 / 9.11, - , 8.27 / 8.23; of 4,096: 2.63 / 2.68, 3.56 / 3.56, 1.29 / 1.27, 2.93 / 2.93."""
    tiles = -(-n // 256) * -(-N // 256)
    if n < TILES_FROM or tiles < 96:
        return False
    if K <= 512:
        return True
    rest = tiles % 256
    use = n * N / ((tiles // 256 + (0.5 if 0 < rest <= 128 else rest > 128)) * 256 ** 3)          # the passes' share that is rows and features
    if N % 128:
        return K <= 1024 or (use >= 0.5 if K <= 2048 else tiles > 160 and use >= 0.7)
    if N % 256:
        return use >= (0.5 if K <= 1024 else 0.75)
    if tiles <= 128:
        return K <= 1024
    if K > 1024 and n < 2000 and use < 0.85:
        return False
    rest = rest or 256
    return rest >= 224 if tiles <= 256 else tiles > 512 or rest <= 128 or rest >= 192


def tiles_reach(rows: int, ldx: int, weights: int, ldo: int) -> bool:
    """Whether the tiles' 32-bit offsets reach all of rows x ldx entries, the weights, and results ldo entries apart (csrc/seq/tiles_reach.h)."""
    return max(rows * ldx, weights) * 2 < 0xC0000000 - 8192 and ldo < 1 << 22


def _only_the_result(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether a product's result is all that is asked of it, so that a kernel's launch may stand in for F.linear: nobody differentiates it in either direction (forward mode
    goes on under no_grad), maps over it, traces, compiles or watches it, or has autocast choose its type, and the tensors are plain ones of the device that launches go to."""
    return (not _grad_enabled() and not _transformed() and _forward_ad._current_level < 0 and _dispatch_modes() == 0 and not _tracing() and not _compiling()
            and not _autocast("cuda") and type(x) in _PLAIN and type(w) in _PLAIN and x.get_device() == torch.cuda.current_device())


# (looked up once: the call above is made for every product of a step of many rows, 1.2 us)
_PLAIN, _forward_ad = (torch.Tensor, torch.nn.Parameter), torch.autograd.forward_ad
_grad_enabled, _transformed, _dispatch_modes = torch.is_grad_enabled, torch._C._are_functorch_transforms_active, torch._C._len_torch_dispatch_stack
_tracing, _compiling, _autocast = torch.jit.is_tracing, torch.compiler.is_compiling, torch.is_autocast_enabled


def linear_tiles_fits(x: torch.Tensor, w: torch.Tensor) -> bool:
    """What nvs_linear_tiles takes."""
    if x.dim() != 2 or w.dim() != 2:
        return False
    (n, k), (N, wide), (ld, unit) = x.shape, w.shape, x.stride()
    return (k == wide and k % 64 == 0 and k >= 128 and N % 8 == 0 and unit == 1 and ld % 8 == 0 and ld >= k and x.dtype == w.dtype == torch.bfloat16 and x.is_cuda
            and x.device == w.device and w.is_contiguous() and tiles_reach(n, ld, N * k, N) and _only_the_result(x, w) and (x.data_ptr() | w.data_ptr()) % 16 == 0)


def many_rows(x: torch.Tensor, w: torch.Tensor, b: torch.Tensor | None = None) -> bool:
    return (x.dim() == 2 and w.dim() == 2 and tiles_rule(x.shape[0], *w.shape) and linear_tiles_fits(x, w)
            and (b is None or type(b) in _PLAIN and b.dtype == x.dtype and b.device == x.device and b.is_contiguous() and b.shape == w.shape[:1] and b.data_ptr() % 16 == 0))


SOME_ROWS_TO = 1024


def rows_rule(m: int, N: int, K: int, captured: bool = False) -> bool:
    """Whether x w^T of m rows beyond a decode step's goes to nvs_linear_rows: its tiles of 64 x 64 are one pass (those of a column tile stay on one of eight XCDs, 32 of them at a
    time), and a call of it takes the host 3 us, one of the library's product 20. MI355X, us of the GPU, weights from memory, here / the library's: 320 rows, 1024 x 1024 5.7 / 8.6,
    x 2048 7.4 / 9.3, x 3072 9.3 / 11.8, 2304 x 1024 7.8 / 9.0, 2048 x 2048 10.0 / 10.9; 512 rows, 2048 x 2048 11.0 / 11.5, x 6144 26.1 / 27.6; 1,000 rows, 1024 x 1024 8.0 / 9.3, x 2048
    11.1 / 11.4, x 3072 14.5 / 15.3; more than a pass 400 rows, 2304 x 1024 13.0 / 9.3, 767 rows, 1040 x 1024 12.2 / 9.4. Two passes of a short reduction still take less than the
    library's call does the host (320 rows, 4096 x 1024 13.4 / 10.2, 512: 14.0 / 11.2), for which such steps wait: waits_for_host, and `captured` where they do not. The two ways round
    alike but add in another order, so a captured step and the same step launched one by one need not have the same bits."""
    passes = -(-(-(-N // 64)) // 8) * -(-m // 64) / 32
    return passes <= 1 and m > 256 or passes <= 2 and K <= 1024 and not captured          # (up to 256 rows: _few_rows, whose line was measured there)


HOST_BOUND_CONTEXT = 2304


def waits_for_host() -> bool:
    """Whether the GPU waits for the host in an eager step of some hundred rows, by what the step says of itself. MI355X, us a step among others, products of up to two passes and gate|up by
    the library / here: Qwen3-0.6B, 300 rows 3606 / 2595, 356: 3683 / 2623; behind contexts, 10 portions of 30 rows behind 512, 1,024, 2,048 tokens 3642 3583 3586 / 2548 2733 3285; attention
    is the longer part from there on: behind 2,560, 2,816, 3,072: 3537 3564 3600 / 3542 3663 3797; one of 320 behind 2,048, 2,560: 3477 3503 / 3432 3709; 20 of 25 and one of 500 behind 2,048: 3370 3499 / 3412 3551. The other families at width 1,024,
    300 to 500 rows: 504 to 887 / 510 to 842 (foduzen 640 / 583, nokipel 633 / 578, pefazen 670 / 600, lobidra 717 / 661, ligidra 884 / 827, reselorn 634 / 530), behind contexts of 3,000
    to 8,000 tokens 677 to 1286 / 568 to 1286, none slower by more than two runs of it differ; so in steps of 40 to 250 and 600 to 1,000 rows. Decode steps read all their contexts."""
    if torch.cuda.is_current_stream_capturing():
        return False
    ctx = get_context()
    if ctx.portions is not None:
        return ctx.portions.max_q > 1
    return ctx.context_lens is None and ctx.max_seqlen_k <= HOST_BOUND_CONTEXT


def some_rows(x: torch.Tensor, w: torch.Tensor, b: torch.Tensor | None = None) -> bool:
    if x.dim() != 2 or w.dim() != 2:
        return False
    (m, k), (N, wide), (ld, unit) = x.shape, w.shape, x.stride()
    return (x.is_cuda and m > 0 and N > 0 and k == wide and k > 0 and k % 64 == 0 and unit == 1 and ld % 8 == 0 and ld >= k and x.dtype == w.dtype == torch.bfloat16
            and rows_rule(m, N, k, k > 1024 or not waits_for_host()) and x.device == w.device and w.is_contiguous() and _only_the_result(x, w)
            and (x.data_ptr() | w.data_ptr()) % 16 == 0
            and (b is None or type(b) in _PLAIN and b.dtype == x.dtype and b.device == x.device and b.is_contiguous() and b.shape == w.shape[:1]))


def linear_rows(x: torch.Tensor, w: torch.Tensor, b: torch.Tensor | None = None) -> torch.Tensor:
    return _linear_rows(x, w, b, -1, 0.0, 0.0, torch.empty(x.shape[0], w.shape[0], dtype=x.dtype, device=x.device))


def _linear_many(x: torch.Tensor, w: torch.Tensor, b: torch.Tensor | None = None) -> torch.Tensor:
    m = x.shape[0]
    if m >= TILES_FROM and many_rows(x, w, b):         # (asked first: short steps wait for the host)
        return linear_tiles(x, w, b)
    if m <= SOME_ROWS_TO and some_rows(x, w, b):
        return linear_rows(x, w, b)
    return torch.nn.functional.linear(x, w, b)


@_launch
def linear(x: torch.Tensor, w: torch.Tensor, b: torch.Tensor | None = None) -> torch.Tensor:
    """x [n, K] times w [N, K]^T (+ b): few rows and many here, others by the vendor library."""
    if not _few_rows(x, w, False) or not (b is None or b.dtype == x.dtype and b.is_contiguous() and b.shape == w.shape[:1]):
        return _linear_many(x, w, b)
    return _linear_rows(x, w, b, -1, 0.0, 0.0, torch.empty(x.shape[0], w.shape[0], dtype=x.dtype, device=x.device))


def linear_tiles(x: torch.Tensor, w: torch.Tensor, b: torch.Tensor | None = None, out: torch.Tensor | None = None) -> torch.Tensor:
    """x w^T (+ b) in tiles of 256 rows: x [n, K], w [N, K], b [N]."""
    lib = load_library()
    n, K = x.shape
    assert x.dtype == w.dtype == torch.bfloat16 and x.stride(1) == 1 and w.is_contiguous() and w.shape[1] == K
    assert b is None or b.dtype == x.dtype and b.is_contiguous() and b.shape == w.shape[:1]
    if out is None:
        out = torch.empty(n, w.shape[0], dtype=x.dtype, device=x.device)
    assert out.shape == (n, w.shape[0]) and out.stride(1) == 1 and out.dtype == x.dtype
    _check(lib.nvs_linear_tiles(_ptr(x), x.stride(0), _ptr(w), _ptr(b), w.shape[0], K, n, _ptr(out), out.stride(0), _stream()))
    return out


def silu_linear_rows(n: int, ff: int, K: int) -> int:
    """Rows per tile of silu_linear, 0 where the vendor library's product and the activation behind it are the faster way. MI355X, us there / here at 64 / 256 rows, ff 3072, K 1024:
    500 rows 18.7 / 13.7 / 14.9, 800: 20.3 / 20.1 / 15.4, 1300: 26.5 / 22.1 / 25.1, 2000: 36.2 / 33.1 / 26.3, 4000: 67 / 61 / 46, 14600: 202 / 204 / 155; ff 768, K 1024: 800:
    13.0 / 13.5 / 14.8, 2000: 16.2 / 17.1 / 15.0, 4000: 22.7 / 21.9 / 16.5; ff 2048, K 2048: 800: 23.7 / 28.1 / 25.1, 1300: 30 / 34 / 26, 4000: 60 / 71 / 51; ff 8192, K 3072: 600: 61 / 89 / 63,
    1000: 87 / 103 / 72, 9000: 721 / 907 / 618; ff 12288, K 4096: 600: 118 / 134 / 128, 1000: 179 / 198 / 143, 14600: 2282 / 2965 / 1984. One pass that is half to three quarters full, long
    reductions, there / 256: ff 3072, K 4096, 1300: 67 / 78; ff 1536, 2700: 64 / 75, K 3072 53 / 59; ff 512, 9100, K 2560 50 / 53, K 2048 43 / 45; ff 6144, K 1536, 600: 31 / 36 (500: 29 / 24). Short ones of which 64 rows make one pass and 256 half of
    one or a little more than one, 64 / 256: K 512, ff 3072, 600: 9.7 / 10.6 (768: 13.1 / 10.7), ff 1536, 1300: 9.8 / 10.6, ff 12288, 600: 25.3 / 26.2; K 1024, ff 12288, 600: 41.1 / 42.0."""
    columns = -(-2 * ff // 256)
    high = -(-n // 256)
    tiles = high * columns
    if K % 64:
        return 0
    if ff % 8 or K < 128:                    # (not for the tiles of 256 rows that the figures are of: those before them)
        return 0 if K > 2560 else 256 if tiles >= 208 and (tiles >= 216 * -(-tiles // 256) or tiles >= 768) else 64 if K <= 1024 and tiles >= 72 else 0
    low = -(-n // 64) * columns              # tiles of 64 rows: two at a time on every compute unit are a pass
    if K <= 1024 and (128 < tiles and low <= 512 or 256 < tiles <= 320 and low <= 1024) or K <= 512 and tiles >= 72 and low <= 256:
        return 64
    if 128 < tiles <= 200 and (tiles <= (176 if K >= 4096 else 160) and (K >= 3072 or K >= 2560 and n >= 3000) or K > 1024 and n < 768 and n < (0.8 if tiles <= 160 else 0.6) * 256 * high):
        return 0
    return 256 if tiles >= 96 and (n >= 768 or K <= 1536) or tiles >= 48 and n >= 500 and K <= 1024 else 0


def silu_short_steps(n: int, K: int) -> bool:
    """Whether gate|up and SiLU of fewer rows than silu_linear_rows gives tiles of 256 rows take those all the same: short reductions in steps that wait for the host, whose calls of the
    library's product and the activation take 25 us, this one 6 (waits_for_host, where the steps are; as there, bits need not be those of a captured step). MI355X, us of the GPU, weights
    from memory, the product and the activation / here, 320 and 640 rows, where neither rule before it takes them: K 128, ff 768 - 7.3 / - 7.2, 1536: 7.2 9.3 / 7.2 7.3; K 512, ff 768 - 10.4
    / - 11.0, 1536: 10.3 12.7 / 11.0 11.1, 3072: 12.6 / 11.2; K 1024, ff 768 - 12.0 / - 15.8, 1536: 11.7 14.4 / 15.7 15.9, 3072: 16.4 / 19.9; 64 and 128 rows, K 1024, ff 6144 - 17.8 / - 20.9."""
    return 64 <= n < TILES_FROM and 128 <= K <= 1024 and K % 64 == 0 and waits_for_host()


def silu_linear_fits(x: torch.Tensor, w: torch.Tensor) -> bool:
    if x.dim() != 2 or w.dim() != 2:
        return False
    (n, k), (N, wide), ld = x.shape, w.shape, x.stride(0)
    return (x.dtype == w.dtype == torch.bfloat16 and x.is_cuda and x.device == w.device and x.stride(1) == 1 and ld % 8 == 0 and ld >= k == wide and N % 2 == 0 and w.is_contiguous()
            and (n + 255) * ld < 8 << 32 and N * k < 8 << 32 and (x.data_ptr() | w.data_ptr()) % 16 == 0)


def silu_linear(x: torch.Tensor, w: torch.Tensor, tm: int, out: torch.Tensor | None = None) -> torch.Tensor:
    """silu(g) u of [g | u] = x w^T: x [n, K], w [2 ff, K] = [gate | up], tiles of tm rows."""
    lib = load_library()
    n, K = x.shape
    ff = w.shape[0] // 2
    assert x.dtype == w.dtype == torch.bfloat16 and x.stride(1) == 1 and w.is_contiguous() and w.shape == (2 * ff, K)
    if out is None:
        out = torch.empty(n, ff, dtype=x.dtype, device=x.device)
    assert out.shape == (n, ff) and out.stride(1) == 1 and out.dtype == x.dtype
    _check(lib.nvs_silu_linear(_ptr(x), x.stride(0), _ptr(w), ff, K, n, tm, _ptr(out), out.stride(0), _stream()))
    return out


@_launch
def linear_act(x: torch.Tensor, w: torch.Tensor, ff: int, kind: int = 0, limit: float = 0.0, alpha: float = 1.0) -> torch.Tensor:
    """glu_act of x times w^T, w [2 ff, K] = [gate | up] (kind 2: [ff, K])."""
    assert w.shape[0] == (1 if kind == 2 else 2) * ff
    out = torch.empty(x.shape[0], ff, dtype=x.dtype, device=x.device)
    if _few_rows(x, w, True):
        return _linear_rows(x, w, None, kind, limit, alpha, out)
    if kind == 0 and silu_linear_fits(x, w):
        tm = silu_linear_rows(x.shape[0], ff, x.shape[1]) or (256 if silu_short_steps(x.shape[0], x.shape[1]) else 0)
        if tm:
            return silu_linear(x, w, tm, out)
    glu_act(_linear_many(x, w), ff, out, kind, limit, alpha)
    return out


@_launch
def moe_route(z: torch.Tensor, total: int, correction: torch.Tensor | None, top: int, count: int, keep: int, scale: float,
              sigmoid: bool = False, renorm: bool = True):
    """z [n, >= total] 32-bit router logits -> (ids [n, top] int32, weights [n, top] 32-bit). Scores are a softmax over the entries,
    or with `sigmoid` every entry's own sigmoid; weights are the chosen scores, divided by their sum with `renorm`, times scale."""
    lib = load_library()
    n = z.shape[0]
    assert z.dtype == torch.float32 and z.stride(1) == 1 and z.shape[1] >= total
    assert correction is None or (correction.dtype == torch.float32 and correction.numel() == total and correction.is_contiguous())
    ids = torch.empty(n, top, dtype=torch.int32, device=z.device)
    wts = torch.empty(n, top, dtype=torch.float32, device=z.device)
    _check(lib.nvs_moe_route(_ptr(z), z.stride(0), _ptr(correction), n, total, top, count, keep, scale, int(sigmoid), int(renorm), _ptr(ids),
                             _ptr(wts), _stream()))
    return ids, wts


def _router_fits(x: torch.Tensor, router: torch.Tensor, bias: torch.Tensor | None) -> bool:
    n, k = x.shape
    if x.dtype not in (torch.bfloat16, torch.float32) or n == 0 or k == 0 or x.stride(0) < k or x.device != router.device:
        return False
    wide = x.dtype == torch.float32
    return (router.shape[0] <= (48 if wide else 64) and k % (32 if wide else 64) == 0 and x.stride(1) == 1 and x.stride(0) * x.element_size() % 16 == 0
            and x.data_ptr() % 16 == 0 and router.is_contiguous() and router.data_ptr() % 16 == 0 and (bias is None or bias.is_contiguous()))


@_launch
def moe_router(x: torch.Tensor, router: torch.Tensor, bias: torch.Tensor | None, total: int, correction: torch.Tensor | None, top: int, count: int,
               keep: int, scale: float, sigmoid: bool = False, renorm: bool = True):
    """moe_route of the 32-bit logits x router^T (+ bias); a router of total + 1 rows ends with the shared expert's gate. Returns
    (ids, weights, gate [n, 1] or None). One kernel for up to 64 entries (48 beside 32-bit rows, whose products take five times the matrix pipe's time)
    and rows of whole 128-byte pieces. MI355X, us, copy + library product + moe_route / here, 33 entries, k 1024 and 4096: bf16, 64 rows 17 / 9 and
    20 / 13, 2000 rows 23 / 9 and 37 / 17, 13,550 rows 58 / 14 and 138 / 30; 32-bit, 64 rows 12.7 / 10.7 and 16.6 / 15.2, 13,550 rows 43 / 24 and
    88 / 68 (64 entries 42 / 35 and 87 / 97)."""
    n, k = x.shape
    entries = router.shape[0]
    assert router.dtype == torch.float32 and router.shape[1] == k and total <= entries <= total + 1
    if not _router_fits(x, router, bias):
        z = torch.nn.functional.linear(x.float(), router, bias)
        ids, wts = moe_route(z, total, correction, top, count, keep, scale, sigmoid, renorm)
        return ids, wts, z[:, total:] if entries > total else None
    lib = load_library()
    assert bias is None or (bias.dtype == torch.float32 and bias.numel() == entries)
    assert correction is None or (correction.dtype == torch.float32 and correction.numel() == total and correction.is_contiguous())
    ids = torch.empty(n, top, dtype=torch.int32, device=x.device)
    wts = torch.empty(n, top, dtype=torch.float32, device=x.device)
    gate = torch.empty(n, 1, dtype=torch.float32, device=x.device) if entries > total else None
    need = lib.nvs_moe_router_workspace(n, entries, k, _code(x))
    ws = torch.empty(need, dtype=torch.float32, device=x.device) if need else None
    _check(lib.nvs_moe_router(_ptr(x), x.stride(0), _code(x), _ptr(router), _ptr(bias), entries, k, _ptr(correction), n, total, top, count, keep, scale,
                              int(sigmoid), int(renorm), _ptr(ids), _ptr(wts), _ptr(gate), _ptr(ws), need, _stream()))
    return ids, wts, gate


@_launch
def moe_table_route(tokens: torch.Tensor, table: torch.Tensor, weight: float):
    """tokens [n] int64, table [vocab, top] int32 -> (ids [n, top] = table[tokens], weights [n, top] = weight)."""
    lib = load_library()
    n, top = tokens.numel(), table.shape[1]
    assert tokens.dtype == torch.int64 and tokens.is_contiguous() and table.dtype == torch.int32 and table.is_contiguous()
    ids = torch.empty(n, top, dtype=torch.int32, device=tokens.device)
    wts = torch.empty(n, top, dtype=torch.float32, device=tokens.device)
    _check(lib.nvs_moe_table_route(_ptr(tokens), _ptr(table), n, top, weight, _ptr(ids), _ptr(wts), _stream()))
    return ids, wts


class MoePlan:
    __slots__ = ("tile_expert", "row_token", "pair_row", "cap", "tm")


def _moe_groups(pairs: int, experts: int, width: int, ff: int, tm: int) -> float:
    """Workgroups of the two products at tiles of tm rows (256 weight rows each), weighted by the lengths of their reductions."""
    tiles = min(experts, pairs) * max(1.0, pairs / experts / tm + 0.5)
    return tiles * (-(-2 * ff // 256) * width + -(-width // 256) * ff) / (width + ff)


def moe_tile_rows(pairs: int, experts: int, width: int, ff: int, dtype: torch.dtype) -> int:
    """Rows per tile of a step's plan. It follows the rows an expert gets on average: a tile reads all weights of its features, so few
    rows want the smallest tile and many the largest. The figures of 256 rows are of moe_gemm_pipe_kernel; the 16-bit plans that gemm_tiles_kernel
    runs instead are moe_plan_rows' below. MI355X, gate|up + down of 32 gated experts, us at tiles of 16 / 64 / 128 / 256 rows:
    width 4096, ff 3072: 8 rows 428 / 436 / 471 / 609; 32: 598 / 455 / 489 / 622; 64: 838 / 580 / 507 / 640; 250: 2256 / 1003 / 879 / 928;
    1694: 12546 / 4674 / 4103 / 3634. Width 2048: 16 rows 126 / 133 / 149 / 178; 32: 141 / 135 / 155 / 181; 500: 1028 / 456 / 420 / 408.
    Width 1024, ff 768 (few and short tiles: two small workgroups per compute unit cover each other's start and end better than one large
    one fills it): 34 rows 40 / 44 / 50 / 66; 68: 52 / 48 / 53 / 70; 500: - / 111 / 118 / 114; 700: - / 146 / 160 / 155; 1400: - / 275 / 265 / 239; 1750: - / 304 / 306 / 275; 32 of
    ff 512: 700 - / 96 / 89 / 100, 1400 - / 181 / 175 / 145; eight of ff 1024: 1000 - / 82 / 86 / 89, 2000 - / 115 / 115 / 97.
    32-bit: width 1024, 32 rows 80 / 126 / 228, 500: 830 / 836 / 912; width 2048, 32 rows 312 / 371 / 679, 125: 888 / 839 / 1100.
    Few workgroups leave most of the chip idle, and then the smaller tile is the faster one: 64-row workgroups on half of the compute units or fewer
    lose to 16 rows, 128-row ones to 64 below about 150, 256-row ones to 128 until the chip is full. Gated, 16 / 64 / 128 / 256 rows: one expert of 2048 x 2048, 64 rows 23 / 58 / 66 / 99,
    400: 48 / 59 / 68 / 112, 700: - / 61 / 74 / 113, 4000: - / 127 / 121 / 137, 8000: - / 243 / 221 / 200; two of 4096 x 3072, 100 rows each 70 / 92 / 100 / 162, 1000: - / 188 /
    178 / 197; four of 8192 x 1024, 2000 rows each - / 502 / 422 / 379. A down product of a short reduction prefers 64 rows until there are many: eight of 2048 x 512, 2000 rows
    each - / 150 / 173 / 179; 32 of 2048 x 768, 300 rows each - / 143 / 138 / 150, 500: - / 256 / 232 / 230, 1000: - / 467 / 428 / 414; of 2048 x 512, 500: - / 142 / 147 / 157, 1400: - / 399 / 350 / 301. 32-bit, two of 2048 x 1024, 100 rows each 46 / 197 / 370.
    Rows that are no whole 128-byte pieces take the kernels that load their own operands, at the heights measured for those."""
    per = pairs // experts
    piece = 64 if dtype == torch.bfloat16 else 32
    if width % piece or ff % piece:
        return 128 if per >= 256 else 64 if per >= 64 else 16

    def groups(tm):
        return _moe_groups(pairs, experts, width, ff, tm)

    if per < 512 and groups(64) < 130:
        return 16
    if dtype != torch.bfloat16:
        return 64 if per >= (96 if width >= 2048 else 512) else 16
    if width < 2048:
        if per >= 640 and groups(256) >= 380:
            return 256
        return 64 if per >= 56 else 16
    if per >= 448 and groups(256) >= (270 if ff >= 1024 else 480):
        return 256
    return 128 if per >= 64 and groups(128) >= (150 if ff >= 1024 else 1000) else 64 if per >= 24 else 16


def moe_plan_rows(pairs: int, experts: int, width: int, ff: int, dtype: torch.dtype) -> int:
    """Rows per tile of a step's plan, where 16-bit tiles of 256 rows are gemm_tiles_kernel's: moe_tile_rows, but 256 rows from 128 per expert on.
    Half of the experts fill a second tile of 128 rows there; its weights are read again and it takes as long as a full one, while the larger tile's
    workgroup takes the next tile's operands under the end of its last. MI355X, plan, gate|up, down and the weighted sum, us at 64 / 128 / 256 rows,
    rows per expert 90, 130, 180, 250, 450 (16-bit, gated):
    32 of 4096 x 3072: 100 591 / 520 / 552; 150 728 / 689 / 560; 200 868 / 705 / 572; 250 963 / 857 / 729; 375 1302 / 1143 / 941;
    32 of 2048 x 1536: 177 / 167 / 170; 234 / 207 / 176; 248 / 208 / 183; 301 / 258 / 218; 350 rows 350 / 311 / 261;
    32 of 2048 x 768: 106 / 98 / 103; 123 / 140 / 106; 157 / 133 / 111; 178 / 150 / 129; 240 / 203 / 173;
    32 of 1024 x 768: 61 / 60 / 61; 67 / 76 / 63; 85 / 77 / 66; 104 / 94 / 86; 136 / 118 / 98; 8 of 1024 x 1024: - ; 42 / 48 / 42; 43 / 49 / 43; 46 / 49 / 44; -;
    8 of 2048 x 512: 47 / 54 / 45; 49 / 56 / 47; 51 / 57 / 48; 54 / 58 / 50; 59 / 64 / 55, 1500 rows 130 / 134 / 108.
    Tiles of 128 rows stay where all of them run at once and their reduction is long: two of 4096 x 3072, 250 rows 132 / 119 / 128, 450 141 / 122 / 131, 900
    204 / 185 / 156; four of 8192 x 1024, 250 rows 173 / 153 / 157, 600 233 / 209 / 205; eight of 4096 x 1024, 180 rows 115 / 101 / 106, 250 127 / 120 / 113;
    eight of 2048 x 1536, 180 rows 94 / 77 / 80, 250 96 / 107 / 82 (one of 2048 x 2048, 1500 rows 78 / 78 / 69). Where moe_tile_rows says 16, few
    workgroups have anything to do, and that stays the fastest (one of 2048 x 2048, 250 rows, 16 / 64 / 128 / 256: 38 / 61 / 70 / 60)."""
    rows, per = moe_tile_rows(pairs, experts, width, ff, dtype), pairs // experts
    if rows == 16 or dtype != torch.bfloat16 or width % 64 or ff % 64 or min(width, ff) < 128 or per < 128:
        return rows
    long = ff >= 1024 and (width >= 4096 or (width >= 2048 and per < 256))
    return 128 if long and _moe_groups(pairs, experts, width, ff, 128) < 170 else 256


@_launch
def moe_plan(ids: torch.Tensor, experts: int, tm: int) -> MoePlan:
    """Pairs (token, choice) sorted by expert into tiles of tm rows (ids >= experts get no row)."""
    lib = load_library()
    n, top = ids.shape
    assert ids.dtype == torch.int32 and ids.is_contiguous()
    p = MoePlan()
    p.tm, p.cap = tm, lib.nvs_moe_rows(n * top, experts, tm)
    p.tile_expert = torch.empty(p.cap // tm, dtype=torch.int32, device=ids.device)
    p.row_token = torch.empty(p.cap, dtype=torch.int32, device=ids.device)
    p.pair_row = torch.empty(n, top, dtype=torch.int32, device=ids.device)
    need = lib.nvs_moe_plan_scratch(n * top, experts)
    scratch = torch.empty(need, dtype=torch.int32, device=ids.device) if need else None
    _check(lib.nvs_moe_plan_wide(_ptr(ids), n, top, experts, tm, _ptr(p.tile_expert), _ptr(p.row_token), _ptr(p.pair_row), _ptr(scratch),
                                 need, _stream()))
    return p


@_launch
def moe_gemm(x: torch.Tensor, w: torch.Tensor, plan: MoePlan, glu: bool, out: torch.Tensor, relu2: bool = False):
    """glu: w [experts, 2 nout, K], rows gathered by token, out = silu(gate) * up; relu2: w [experts, nout, K], rows gathered by
    token, out = max(w x, 0)^2; neither: w [experts, nout, K], x holds the planned rows."""
    lib = load_library()
    assert not (glu and relu2)
    nout, K = (w.shape[1] // 2 if glu else w.shape[1]), w.shape[2]
    assert w.is_contiguous() and x.stride(1) == 1 and x.shape[1] == K and out.shape == (plan.cap, nout) and out.stride(1) == 1
    assert glu or relu2 or x.shape[0] == plan.cap
    _check(lib.nvs_moe_gemm(_ptr(x), x.stride(0), _ptr(w), _same(x, w, out), 1 if glu else (2 if relu2 else 0), nout, K, _ptr(plan.tile_expert), _ptr(plan.row_token),
                            plan.cap, plan.tm, _ptr(out), out.stride(0), _stream()))


@_launch
def moe_combine(rows: torch.Tensor, plan: MoePlan, wts: torch.Tensor, h: torch.Tensor, shared: torch.Tensor | None,
                shared_gate: torch.Tensor | None, out: torch.Tensor | None, res: torch.Tensor | None = None):
    """out[t] = sum_k wts[t, k] * (row of the pair, or h[t] for a pass-through choice) + sigmoid(shared_gate[t]) * shared[t]. With res
    [n, width] (32-bit): res += that sum, and out (may be None) is the new res in the activation type."""
    lib = load_library()
    n, width = h.shape
    top = wts.shape[1]
    assert rows.stride(1) == 1 and rows.shape[1] == width and h.stride(1) == 1
    assert (out is None and res is not None) or (out.shape == (n, width) and out.is_contiguous())
    assert res is None or (res.dtype == torch.float32 and res.shape == (n, width) and res.is_contiguous())
    assert wts.dtype == torch.float32 and wts.is_contiguous() and plan.pair_row.shape == (n, top)
    assert shared is None or (shared.shape == (n, width) and shared.is_contiguous())
    assert shared_gate is None or (shared is not None and shared_gate.dtype == torch.float32 and shared_gate.shape[0] == n)
    _check(lib.nvs_moe_combine(_ptr(rows), rows.stride(0), _ptr(plan.pair_row), _ptr(wts), top, _ptr(h), h.stride(0), _ptr(shared),
                               _ptr(shared_gate), shared_gate.stride(0) if shared_gate is not None else 0, _same(rows, h, shared, out), n,
                               width, _ptr(res), _ptr(out), _stream()))
