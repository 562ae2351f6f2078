"""Projections of a decode step's few tokens on the HIP kernel (csrc/linear_rows.hip, through
libmi_model.so, the C ABI in include/mi_model.h), each with what surrounds it in the same launch:

  rope_tables  cos and sin of the step's positions           (model.py:151-155)
  linear     [residual +] ([rmsnorm] x W^T + bias)           (model.py:81-84,107,204-207)
  mlp        [residual +] SwiGLU MLP of [rmsnorm] x          (model.py:112-138; two launches)
  qkv_rope   rmsnorm, q/k/v projection, rotary embedding and the paged cache write (model.py:92,96)

The weights are read in nn.Linear's own layout.  `linear_fits` / `mlp_fits` say which sizes the
kernel takes.  No CPU path and no fallback: a missing library or a call outside the sizes raises.
"""
import ctypes
import os
from pathlib import Path

import torch

from . import _lib
from .fa2 import _pool_strides

LIB_PATH = Path(os.environ.get("MI_MODEL_LIB", Path(__file__).resolve().parent / "libmi_model.so"))

MAX_ROWS = 64        # tokens per call
MAX_NORM_ROWS = 16   # with the norm of x in the same launch
MAX_IN = 2048        # in features (a work-group's waves hold whole rows of x)
HEAD_DIM = 128
_PLAIN = (torch.Tensor, torch.nn.Parameter)

_p, _i32, _i64, _f32 = ctypes.c_void_p, ctypes.c_int32, ctypes.c_int64, ctypes.c_float
# name -> (restype, argtypes); mirrors include/mi_model.h
SIGNATURES = {
    "mi_model_last_error": (ctypes.c_char_p, []),
    "mi_model_linear": (_i32, [_i32, _p, _i64, _p, _f32, _p, _p, _p, _i64, _p, _i64, _i32, _i32,
                               _i32, _p]),
    "mi_model_rope_table": (_i32, [_i32, _p, _p, _p, _p, _i32, _i32, _p]),
    "mi_model_mlp_workspace_size": (ctypes.c_size_t, [_i32, _i32, _i32]),
    "mi_model_mlp": (_i32, [_i32, _p, _i64, _p, _f32, _p, _p, _p, _i64, _p, _i64, _i32, _i32, _i32,
                            _p, ctypes.c_size_t, _p]),
    "mi_model_qkv_rope": (_i32, [_i32, _p, _i64, _p, _f32, _p, _p, _p, _p, _i64, _p, _p, _i64, _p,
                                 _p, _p, _i32, _i32, _i32, _i32, _i32, _p]),
}

_library = None


def load():
    """Load libmi_model.so once; raise if it is missing."""
    global _library
    if _library is None:
        if not LIB_PATH.exists():
            raise ImportError(
                f"{LIB_PATH} not found: build it with `python my-inference-engine_amd/build_lib.py`")
        lib = ctypes.CDLL(str(LIB_PATH))
        for name, (res, args) in SIGNATURES.items():
            fn = getattr(lib, name)
            fn.restype = res
            fn.argtypes = args
        _library = lib
    return _library


def _check(status):
    if status != _lib.OK:
        raise _lib.MiFa2Error(
            f"libmi_model status {status}: {load().mi_model_last_error().decode()}")


def _rows(t, name, dtype):
    assert t.is_cuda and t.dtype == dtype, f"{name}: a {dtype} GPU tensor"
    assert t.dim() == 2 and t.stride(1) == 1, f"{name}: [rows, n] with unit column stride"
    # one row: its stride is never used, and torch may report any value there
    return t.data_ptr(), t.stride(0) if t.shape[0] > 1 else t.shape[1]


def _weight(w, shape, dtype):
    assert w.is_cuda and w.dtype == dtype and tuple(w.shape) == shape and w.is_contiguous(), \
        f"a contiguous {dtype} GPU weight of shape {shape}"
    return w.data_ptr()


def _readable(t):
    """t's rows as the kernel reads them: unit column stride, 16-byte aligned rows."""
    return (t.stride(-1) == 1 and t.data_ptr() % 16 == 0
            and (t.shape[0] == 1 or (t.stride(0) % 8 == 0 and 0 < t.stride(0) < 1 << 23
                                     and t.stride(0) >= t.shape[1])))


def _held(t, x):
    """Whether parameter t is held as the kernels read it for rows like x: x's type and device,
    contiguous, 16-byte aligned, a plain tensor (no subclass with operations of its own)."""
    return (type(t) in _PLAIN and t.dtype == x.dtype and t.get_device() == x.get_device()
            and t.is_contiguous() and t.data_ptr() % 16 == 0)


def weight_fits(w, x, out_features):
    """Whether w is an [out_features, in] weight the kernel reads for rows like x."""
    if not _held(w, x) or w.dim() != 2:
        return False
    n, k = w.shape
    return n == out_features and n % 16 == 0 and n > 0 and k % 32 == 0 and 0 < k <= MAX_IN


def bias_fits(b, x, out_features):
    """Whether b is None or a bias of out_features the kernel reads for rows like x."""
    return b is None or (_held(b, x) and b.shape == (out_features,))


def linear_fits(x, w, norm=None):
    """Whether `linear` takes x [rows, in] and w [out, in] (and norm, an RMSNorm weight)."""
    if norm is not None and not (_held(norm, x) and norm.shape == x.shape[1:]):
        return False
    rows, k = x.shape
    return (type(x) in _PLAIN and 1 <= rows <= (MAX_ROWS if norm is None else MAX_NORM_ROWS)
            and x.dtype in _lib.DTYPES and weight_fits(w, x, w.shape[0])
            and w.shape[1] == k and _readable(x))


def mlp_fits(x, gate_up_w, down_w, norm=None):
    """Whether `mlp` takes x [rows, hidden] and these weights (and norm, an RMSNorm weight)."""
    hidden, inter = down_w.shape
    return (linear_fits(x, gate_up_w, norm) and x.shape[1] == hidden and hidden % 16 == 0
            and inter % 32 == 0 and 0 < inter <= 1 << 18 and gate_up_w.shape[0] == 2 * inter
            and _held(down_w, x))


def linear_pays(rows, w):
    """Whether `linear` on [rows, in] is at least as fast as the library's GEMM (us, library and here, bf16;
    fp16 alike).  Up to 16 rows: from 768 in features on (896 x 32,000 14.6 and 13.5, 2,048 x 151,936
    150 and 122; 512 x 32,000 10.5 and 12.1).  More rows: where the weight is larger than the 256 MB
    last-level cache, whose stream bounds both (1,536 x 151,936 at 17, 32, 40 rows 103 and 90, 105 and
    96, 106 and 100; 1,536 x 64,000 at 32 33.8 and 35.3), up to 40 rows (48: 98 and 102)."""
    return (rows <= 16 and w.shape[1] >= 768) or (
        rows <= 40 and w.numel() * w.element_size() >= 1 << 28)


def mlp_pays(rows, hidden):
    """The same for `mlp`: up to 32 rows, and up to 64 where hidden <= 1536 (1,536 x 8,960 at 16, 32, 64
    rows 41 and 24, 41 and 29, 48 and 37; 1,792 x 4,864 at 32 and 33 24.8 and 22.5, 26.0 and 28.0;
    2,048 x 8,192 at 33 35.2 and 38.2)."""
    return rows <= (MAX_ROWS if hidden <= 1536 else 32)


def linear(x, w, bias=None, residual=None, norm_weight=None, eps=0.0, out=None):
    """x [rows, in], w [out, in] -> [rows, out].  residual [rows, out] may be `out` (in place)."""
    R, K = x.shape
    N = w.shape[0]
    if out is None:
        out = torch.empty((R, N), device=x.device, dtype=x.dtype)
    dt = x.dtype
    xp, xs = _rows(x, "x", dt)
    op, os_ = _rows(out, "out", dt)
    assert out.shape == (R, N) and (residual is None or residual.shape == (R, N))
    rp, rs = _rows(residual, "residual", dt) if residual is not None else (None, 0)
    with _lib.on_device(x.device) as stream:
        _check(load().mi_model_linear(
            _lib.DTYPES[dt], xp, xs, _weight(norm_weight, (K,), dt) if norm_weight is not None
            else None, float(eps), _weight(w, (N, K), dt),
            _weight(bias, (N,), dt) if bias is not None else None, rp, rs, op, os_, R, N, K, stream))
    return out


def rope_tables(starts, T, inv_freq):
    """starts [B] int32, inv_freq [64] (16-bit) -> cos, sin [B, 1, T, 128] in inv_freq's dtype for
    positions starts[b] .. starts[b] + T - 1 (model.py:151-155)."""
    B, dev = starts.shape[0], starts.device
    assert starts.is_cuda and starts.dtype == torch.int32 and starts.is_contiguous()
    assert inv_freq.device == dev and inv_freq.dtype in _lib.DTYPES and inv_freq.is_contiguous()
    assert inv_freq.shape == (HEAD_DIM // 2,)
    cos, sin = (torch.empty((B, 1, T, HEAD_DIM), device=dev, dtype=inv_freq.dtype) for _ in range(2))
    with _lib.on_device(dev) as stream:
        _check(load().mi_model_rope_table(_lib.DTYPES[inv_freq.dtype], starts.data_ptr(),
                                          inv_freq.data_ptr(), cos.data_ptr(), sin.data_ptr(), B, T,
                                          stream))
    return cos, sin


def mlp(x, gate_up_w, down_w, residual=None, norm_weight=None, eps=0.0, out=None):
    """x [rows, hidden], gate_up_w [2 * inter, hidden], down_w [hidden, inter] -> [rows, hidden].
    out may be residual and x."""
    R, H = x.shape
    inter = down_w.shape[1]
    dt = x.dtype
    if out is None:
        out = torch.empty((R, H), device=x.device, dtype=dt)
    lib = load()
    xp, xs = _rows(x, "x", dt)
    op, os_ = _rows(out, "out", dt)
    assert out.shape == (R, H) and (residual is None or residual.shape == (R, H))
    rp, rs = _rows(residual, "residual", dt) if residual is not None else (None, 0)
    # every call has its own (from torch's caching allocator, in stream order): nothing is shared
    ws = torch.empty(lib.mi_model_mlp_workspace_size(R, H, inter), dtype=torch.uint8,
                     device=x.device)
    with _lib.on_device(x.device) as stream:
        _check(lib.mi_model_mlp(
            _lib.DTYPES[dt], xp, xs, _weight(norm_weight, (H,), dt) if norm_weight is not None
            else None, float(eps), _weight(gate_up_w, (2 * inter, H), dt),
            _weight(down_w, (H, inter), dt), rp, rs, op, os_, R, H, inter, ws.data_ptr(),
            ws.numel(), stream))
    return out


def qkv_rope(x, norm_weight, eps, w, bias, cos, sin, slot_mapping, k_pool, v_pool, heads_q,
             heads_kv):
    """x [rows, hidden], w [(heads_q + 2 heads_kv) * 128, hidden], cos/sin [rows, 128],
    slot_mapping [rows] int32, k_pool/v_pool [slots, heads_kv, 128] (one layer of KVCache.buf).
    Returns the rotated queries [rows, heads_q * 128]; k and v go to the rows' cache slots."""
    R, H = x.shape
    dt = x.dtype
    n_out = (heads_q + 2 * heads_kv) * HEAD_DIM
    xp, xs = _rows(x, "x", dt)
    cp, cs = _rows(cos, "cos", dt)
    sp, ss = _rows(sin, "sin", dt)
    assert cos.shape == (R, HEAD_DIM) and sin.shape == (R, HEAD_DIM) and cs == ss
    assert slot_mapping.is_cuda and slot_mapping.dtype == torch.int32
    assert slot_mapping.shape == (R,) and slot_mapping.is_contiguous()
    assert k_pool.is_cuda and k_pool.dtype == dt and v_pool.dtype == dt and k_pool.dim() == 3
    assert k_pool.shape == v_pool.shape and k_pool.stride() == v_pool.stride()
    assert k_pool.shape[1:] == (heads_kv, HEAD_DIM) and k_pool.stride(2) == 1
    q = torch.empty((R, heads_q * HEAD_DIM), device=x.device, dtype=dt)
    with _lib.on_device(x.device) as stream:
        _check(load().mi_model_qkv_rope(
            _lib.DTYPES[dt], xp, xs, _weight(norm_weight, (H,), dt), float(eps),
            _weight(w, (n_out, H), dt), _weight(bias, (n_out,), dt) if bias is not None else None,
            cp, sp, cs, slot_mapping.data_ptr(), q.data_ptr(), heads_q * HEAD_DIM,
            k_pool.data_ptr(), v_pool.data_ptr(), _pool_strides(k_pool), k_pool.shape[0], R, H,
            heads_q, heads_kv, stream))
    return q
