"""ctypes binding of libdip_hip.so (the gfx950 DIP decode kernels).

Every function here validates dtype / device / shape / contiguity on the host,
passes raw device pointers plus torch's current HIP stream to the C ABI
declared in include/dip_hip.h, and raises ``RuntimeError`` on any non-zero
status.  There is no fallback: if the library is not built, importing this
module raises ``ImportError``.

Workspaces are cached per (device, tag) as zero-filled byte tensors; every
call returns the parts that must start at zero (arrival counters) to zero
before it ends, and every call that shares one is ordered on the same stream (the module layer runs layers one after the
other, like the reference's SharedBuffers, dip_stream_predispatch.py:123-138).
"""
from __future__ import annotations

import ctypes
import os
import threading
from pathlib import Path

import torch

_HERE = Path(__file__).resolve().parent
LIB_PATH = Path(os.environ.get("DIP_HIP_LIB", _HERE / "libdip_hip.so"))
HEADER_PATH = _HERE.parent / "include" / "dip_hip.h"

if not LIB_PATH.exists():
    raise ImportError(
        f"{LIB_PATH} is not built; run `python dynamic-input-pruning_amd/build.py` "
        "(or __graft_entry__.build()) first")

lib = ctypes.CDLL(str(LIB_PATH))

_p = ctypes.c_void_p
_i64 = ctypes.c_int64
_i32 = ctypes.c_int
_sz = ctypes.c_size_t

_SIGS = {
    "dip_status_string": ([_i32], ctypes.c_char_p),
    "dip_version": ([], _i32),
    "dip_topk_max_n": ([], _i64),
    "dip_int4_gemv": ([_p, _p, _p, _p, _i64, _i64, _i32, _p], _i32),
    "dip_topk_workspace_size": ([_i64], _sz),
    "dip_topk_select": ([_p, _p, _i64, _i64, _p, _sz, _p], _i32),
    "dip_topk_meta": ([_p, _p, _p], _i32),
    "dip_gate_silu_topk": ([_p, _p, _p, _p, _p, _i64, _i64, _i64, _p, _sz, _p], _i32),
    "dip_int4_gather_gemv": ([_p, _p, _p, _p, _p, _i64, _i64, _i64, _p], _i32),
    "dip_up_gather_h": ([_p, _p, _p, _p, _p, _p, _i64, _i64, _i64, _p], _i32),
    "dip_gather_down_workspace_size": ([_i64, _i64], _sz),
    "dip_int4_gather_down": ([_p, _p, _p, _p, _p, _i64, _i64, _i64, _p, _sz, _p], _i32),
    "dip_ca_fused_gemv": ([_p, _p, _p, _p, _p, _p, _p, _p, _p, _i64, _p, _i64, _i64, _i64, _i64,
                           _p], _i32),
    "dip_ca_down": ([_p, _p, _p, _p, _p, _p, _p, _p, _i64, _i64, _i64, _i64, _p, _sz, _p], _i32),
    "dip_ca_assemble": ([_p, _p, _p, _p, _p, _p, _p, _i64, _i64, _p], _i32),
    "dip_dequant_rows": ([_p, _p, _p, _p, _i64, _i64, _i64, _i32, _p], _i32),
    "dip_dequant_t": ([_p, _p, _p, _i64, _i64, _p], _i32),
    "dip_mlp_workspace_size": ([_i64, _i64, _i64], _sz),
    "dip_mlp_decode": ([_p, _p, _p, _p, _p, _p, _p, _p, _p, _p, _p, _p, _i64, _i64, _i64, _p,
                        _sz, _p, _p], _i32),
    "dip_mlp_state_size": ([], _sz),
    "dip_mlp_decode_noalloc": ([_p, _p, _p, _p, _p, _p, _p, _p, _p, _p, _p, _p, _i64, _i64, _i64,
                                _p, _p], _i32),
    "dip_mlp_decode_rmsnorm": ([_p, _p, _p, _p, _p, _p, _p, _p, _p, _p, ctypes.c_float, _p, _p,
                                _p, _p, _p, _p, _i64, _i64, _i64, _p, _sz, _p, _p], _i32),
    "dip_gate_silu_topk_spec": ([_p, _p, _p, _p, _p, _p, _p, _p, _i64, _i64, _i64, _p, _sz, _p,
                                 _p], _i32),
    "dip_int4_gather_down_by_channel": ([_p, _p, _p, _p, _p, _p, _p, _i64, _i64, _i64, _p, _sz,
                                         _p], _i32),
    "dip_scales_group_major": ([_p, _p, _i64, _i64, _p], _i32),
    "dip_quantize_int4": ([_p, _i32, _p, _p, _i64, _i64, _p], _i32),
    "dip_transpose_down_int4": ([_p, _p, _p, _p, _i64, _i64, _p], _i32),
    "dip_host_gather_rows": ([_p, _p, _p, _i64, _i64, _i64, _i32], _i32),
    "dip_host_gather_rows_multi": ([_p, _p, _p, _i64, _p, _i64, _i64, _i32], _i32),
    "dip_host_stream_rows": ([_p, _p, _p, _p, _i64, _p, _i64, _i64, _i64, _i32, _p, _p], _i32),
    "dip_int4_gemm_swiglu": ([_p, _p, _p, _p, _p, _p, _i64, _i64, _i64, _p], _i32),
    "dip_swiglu": ([_p, _p, _p, _i64, _p], _i32),
    "dip_stream_rows": ([_p, _p, _p, _i64, _p, _p, _i64, _i64, _p], _i32),
    "dip_int4_gemm": ([_p, _p, _p, _p, _i64, _i64, _i64, _p], _i32),
    "dip_int4_gemm_t_workspace_size": ([_i64, _i64, _i64], _sz),
    "dip_int4_gemm_t": ([_p, _p, _p, _p, _i64, _i64, _i64, _p, _sz, _p], _i32),
    "dip_int4_gemv_rmsnorm": ([_p, _p, _p, _p, _p, ctypes.c_float, _p, _p, _i64, _i64, _p],
                              _i32),
    "dip_add_rmsnorm_rows": ([_p, _p, _p, _p, _i64, _i64, ctypes.c_float, _p], _i32),
    "dip_qk_norm_rope_cache_rows": ([_p, _p, _p, _p, _p, _p, _p, _p, _i64, _i64, _i64, _i64, _i64,
                                     ctypes.c_float, _p], _i32),
    "dip_add_rmsnorm": ([_p, _p, _p, _p, _i64, ctypes.c_float, _p], _i32),
    "dip_qk_norm_rope_cache": ([_p, _p, _p, _p, _p, _p, _p, _p, _p, _i64, _i64, _i64, _i64,
                                ctypes.c_float, _p], _i32),
    "dip_decode_attention_workspace_size": ([_i64, _i64, _i64], _sz),
    "dip_decode_attention_fused_max_len": ([], _i64),
    "dip_decode_attention_fused": ([_p, _p, _p, _p, _p, _p, _p, _p, _p, _i64, _i64, _i64, _i64,
                                    ctypes.c_float, ctypes.c_float, _p], _i32),
    "dip_decode_attention": ([_p, _p, _p, _p, _p, _i64, _i64, _i64, _i64, ctypes.c_float, _p, _sz,
                              _p], _i32),
    "dip_set_tuning": ([_i32, _i32], _i32),
    "dip_timeline_read": ([_i32, _p], _i32),
    "dip_get_tuning": ([_i32], _i32),
}
# The argument lists above follow this version of include/dip_hip.h
# (DIP_VERSION); a library built from another one would be called with
# shifted arguments, or lack an entry point, so it is refused here.
ABI_VERSION = 305
if lib.dip_version() != ABI_VERSION:
    raise ImportError(f"{LIB_PATH} reports ABI version {lib.dip_version()}, these bindings "
                      f"are written for {ABI_VERSION}; rebuild the library")
for _name, (_args, _res) in _SIGS.items():
    _fn = getattr(lib, _name)
    _fn.argtypes = _args
    _fn.restype = _res

GROUP_SIZE = 128


def status_string(st: int) -> str:
    return lib.dip_status_string(st).decode()


def _check(st: int, fn: str) -> None:
    if st != 0:
        raise RuntimeError(f"{fn} failed: {status_string(st)} (status {st})")


# ---------------------------------------------------------------------------
# host-side validation
# ---------------------------------------------------------------------------
def _dev(*ts: torch.Tensor) -> torch.device:
    d = ts[0].device
    if d.type != "cuda":
        raise RuntimeError(f"expected tensors on a HIP device, got {d}")
    for t in ts[1:]:
        if t.device != d:
            raise RuntimeError(f"tensors on different devices: {d} vs {t.device}")
    return d


def _want(t: torch.Tensor, dtype: torch.dtype, name: str, shape=None) -> torch.Tensor:
    if not isinstance(t, torch.Tensor):
        raise RuntimeError(f"{name} must be a tensor")
    if t.dtype != dtype:
        raise RuntimeError(f"{name} must be {dtype}, got {t.dtype}")
    if shape is not None and tuple(t.shape) != tuple(shape):
        raise RuntimeError(f"{name} must have shape {tuple(shape)}, got {tuple(t.shape)}")
    if not t.is_contiguous() or t.data_ptr() % 16 != 0:
        t = t.contiguous()
        if t.data_ptr() % 16 != 0:
            t = t.clone()
    return t


def _weights(qw: torch.Tensor, sc: torch.Tensor, name: str):
    if qw.dim() != 2 or sc.dim() != 2:
        raise RuntimeError(f"{name}: qweight and scales must be 2-D")
    rows, half = qw.shape
    cols = half * 2
    if cols % GROUP_SIZE != 0:
        raise RuntimeError(f"{name}: in_features {cols} is not a multiple of {GROUP_SIZE}")
    # resident weights pass as they are: the checks of _want, without its calls
    if (qw.dtype is torch.int8 and sc.dtype is torch.bfloat16
            and sc.shape == (rows, cols // GROUP_SIZE) and qw.is_contiguous()
            and sc.is_contiguous() and not (qw.data_ptr() | sc.data_ptr()) & 15):
        return qw, sc, rows, cols
    qw = _want(qw, torch.int8, f"{name}.qweight")
    sc = _want(sc, torch.bfloat16, f"{name}.scales", (rows, cols // GROUP_SIZE))
    return qw, sc, rows, cols


def _stream(device: torch.device) -> int:
    # the handle alone: a Stream object costs 2 us of a small call's 15
    if device.index is None:
        return torch.cuda.current_stream(device).cuda_stream
    return torch._C._cuda_getCurrentRawStream(device.index)


def _ptr(t):
    return None if t is None else t.data_ptr()


_ws_lock = threading.Lock()
_ws_cache: dict = {}


def workspace(device: torch.device, nbytes: int, tag: str) -> torch.Tensor:
    """Zero-filled device workspace of at least `nbytes`, cached per
    (device, tag).  Growing replaces it with a larger zeroed buffer."""
    key = (device.index if device.index is not None else torch.cuda.current_device(), tag)
    with _ws_lock:
        buf = _ws_cache.get(key)
        if buf is None or buf.numel() < nbytes:
            buf = torch.zeros(max(nbytes, 256), dtype=torch.uint8, device=device)
            _ws_cache[key] = buf
        return buf


# ---------------------------------------------------------------------------
# ops
# ---------------------------------------------------------------------------
def int4_gemv(qweight, scales, x, act: int = 0, out=None):
    """out[r] = bf16(sum (q*s)[r,:] . x); act=1 applies bf16(silu(.))."""
    qweight, scales, rows, cols = _weights(qweight, scales, "int4_gemv")
    dev = _dev(qweight, scales, x)
    x = _want(x.reshape(-1), torch.bfloat16, "x", (cols,))
    if out is None:
        out = torch.empty(rows, dtype=torch.bfloat16, device=dev)
    elif (out.dtype != torch.bfloat16 or out.numel() != rows or not out.is_contiguous()
          or out.device != dev or out.data_ptr() % 16 != 0):
        raise RuntimeError(f"out must be a contiguous, 16-byte aligned bf16 tensor of {rows} "
                           "values on the weights' device")
    _check(lib.dip_int4_gemv(_ptr(qweight), _ptr(scales), _ptr(x), _ptr(out), rows, cols,
                             int(act), _stream(dev)), "dip_int4_gemv")
    return out


# Input widths the GEMV's RMSNorm prologue is built for (the staged-x widths).
NORM_GEMV_COLS = frozenset((2560, 4096, 5120))


def int4_gemv_rmsnorm(qweight, scales, h, add, norm_w, eps: float, h_out=None, out=None):
    """out = GEMV of bf16(norm_w * bf16(v * rsqrt(mean(v^2) + eps))) with
    v = bf16(h + add); v also goes to h_out when given (h_out must be a
    different buffer from h and add)."""
    qweight, scales, rows, cols = _weights(qweight, scales, "int4_gemv_rmsnorm")
    dev = _dev(qweight, scales, h, norm_w)
    _bf16_vec(h, cols, "h")
    _bf16_vec(norm_w, cols, "norm_w")
    for name, t in (("add", add), ("h_out", h_out)):
        if t is not None:
            _bf16_vec(t, cols, name)
            if t.device != dev:
                raise RuntimeError(f"{name} must be on the weights' device")
    if out is None:
        out = torch.empty(rows, dtype=torch.bfloat16, device=dev)
    else:
        _bf16_vec(out, rows, "out")
    _check(lib.dip_int4_gemv_rmsnorm(_ptr(qweight), _ptr(scales), _ptr(h), _ptr(add),
                                     _ptr(norm_w), float(eps), _ptr(h_out), _ptr(out), rows,
                                     cols, _stream(dev)), "dip_int4_gemv_rmsnorm")
    return out


def int4_gemm(qweight, scales, x, out=None):
    """out [M, N] = bf16(x [M, K] @ (q*s)^T) on bf16 MFMA (prompt projections)."""
    qweight, scales, rows, cols = _weights(qweight, scales, "int4_gemm")
    dev = _dev(qweight, scales, x)
    if x.dtype != torch.bfloat16 or x.shape[-1] != cols:
        raise RuntimeError(f"x must be bf16 [..., {cols}]")
    x2 = x if x.dim() == 2 else x.reshape(-1, cols)
    if not x2.is_contiguous() or x2.data_ptr() % 16:
        x2 = x2.contiguous().clone() if x2.data_ptr() % 16 else x2.contiguous()
    m = x2.shape[0]
    shape = (*x.shape[:-1], rows)
    if out is None:
        out = torch.empty(shape, dtype=torch.bfloat16, device=dev)
    elif (out.dtype != torch.bfloat16 or out.numel() != m * rows or not out.is_contiguous()
          or out.device != dev):
        raise RuntimeError(f"out must be a contiguous bf16 tensor of {m} x {rows} values")
    _check(lib.dip_int4_gemm(_ptr(qweight), _ptr(scales), _ptr(x2), _ptr(out), m, rows, cols,
                             _stream(dev)), "dip_int4_gemm")
    return out if out.shape == shape else out.view(shape)


def int4_gemm_swiglu(gate_qw, gate_sc, up_qw, up_sc, x):
    """swiglu(int4_gemm(gate, x), int4_gemm(up, x)) in one launch."""
    gate_qw, gate_sc, rows, cols = _weights(gate_qw, gate_sc, "int4_gemm_swiglu.gate")
    up_qw, up_sc, rows2, cols2 = _weights(up_qw, up_sc, "int4_gemm_swiglu.up")
    if (rows2, cols2) != (rows, cols):
        raise RuntimeError("gate and up differ in shape")
    dev = _dev(gate_qw, gate_sc, up_qw, up_sc, x)
    if x.dtype != torch.bfloat16 or x.shape[-1] != cols:
        raise RuntimeError(f"x must be bf16 [..., {cols}]")
    x2 = _want(x.reshape(-1, cols), torch.bfloat16, "x")
    out = torch.empty(*x.shape[:-1], rows, dtype=torch.bfloat16, device=dev)
    _check(lib.dip_int4_gemm_swiglu(_ptr(gate_qw), _ptr(gate_sc), _ptr(up_qw), _ptr(up_sc),
                                    _ptr(x2), _ptr(out), x2.shape[0], rows, cols, _stream(dev)),
           "dip_int4_gemm_swiglu")
    return out


def int4_gemm_t_splits(m: int, out_features: int, in_features: int) -> int:
    """The parts of K that dip_int4_gemm_t adds up in its workspace."""
    nbytes = lib.dip_int4_gemm_t_workspace_size(m, out_features, in_features)
    return max(1, nbytes // (4 * m * out_features))


def int4_gemm_t(qweight_t, scales_t, x, out=None):
    """out [M, N] = bf16(x [M, K] @ bf16(q*s)) for W stored as K rows of N
    (the transposed down matrix), on bf16 MFMA."""
    qweight_t, scales_t, k_rows, n = _weights(qweight_t, scales_t, "int4_gemm_t")
    dev = _dev(qweight_t, scales_t, x)
    if x.dtype != torch.bfloat16 or x.shape[-1] != k_rows:
        raise RuntimeError(f"x must be bf16 [..., {k_rows}]")
    x2 = x.reshape(-1, k_rows)
    if not x2.is_contiguous() or x2.data_ptr() % 16:
        x2 = x2.contiguous().clone() if x2.data_ptr() % 16 else x2.contiguous()
    m = x2.shape[0]
    if out is None:
        out = torch.empty(m, n, dtype=torch.bfloat16, device=dev)
    elif (out.dtype != torch.bfloat16 or out.numel() != m * n or not out.is_contiguous()
          or out.device != dev):
        raise RuntimeError(f"out must be a contiguous bf16 tensor of {m} x {n} values")
    nbytes = lib.dip_int4_gemm_t_workspace_size(m, n, k_rows)
    # scratch that nothing has to clear: the caching allocator's, so calls on
    # several streams or in a captured graph each have their own
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev) if nbytes else None
    _check(lib.dip_int4_gemm_t(_ptr(qweight_t), _ptr(scales_t), _ptr(x2), _ptr(out), m, n, k_rows,
                               _ptr(ws), 0 if ws is None else ws.numel(), _stream(dev)),
           "dip_int4_gemm_t")
    return out.view(*x.shape[:-1], n)


def topk_select(s: torch.Tensor, k: int, out=None):
    """int32 [k] indices, bit-exact with topk_ops::topk_select."""
    dev = _dev(s)
    s = _want(s.reshape(-1), torch.bfloat16, "s")
    n = s.numel()
    k = int(k)
    if k < 0:
        raise RuntimeError("k must be >= 0")
    if n > lib.dip_topk_max_n():
        raise RuntimeError(f"top-k supports n <= {lib.dip_topk_max_n()}, got {n}")
    if out is None:
        out = torch.empty(k, dtype=torch.int32, device=dev)
    nbytes = lib.dip_topk_workspace_size(n)
    ws = workspace(dev, nbytes, "topk")
    _check(lib.dip_topk_select(_ptr(s), _ptr(out), n, k, _ptr(ws), ws.numel(), _stream(dev)),
           "dip_topk_select")
    return out


def topk_meta(device=None) -> dict:
    """Thresholds and tier sizes of the last top-k run on `device`
    (t_lo, t_strict as fp32; count_a, count_b)."""
    dev = torch.device(device) if device is not None else torch.device("cuda")
    ws = workspace(dev, lib.dip_topk_workspace_size(0), "topk")
    m = torch.empty(16, dtype=torch.uint8, device=dev)
    _check(lib.dip_topk_meta(_ptr(ws), _ptr(m), _stream(dev)), "dip_topk_meta")
    f = m[:8].view(torch.float32).cpu()
    i = m[8:].view(torch.int32).cpu()
    return dict(t_lo=float(f[0]), t_strict=float(f[1]), count_a=int(i[0]), count_b=int(i[1]))


def gate_silu_topk(qweight, scales, x, k, g=None, idx=None):
    """g = bf16(silu(gate(x))) then idx = topk(|g|, k) (int32, reference
    order), both on the device with no host synchronisation."""
    qweight, scales, rows, cols = _weights(qweight, scales, "gate")
    dev = _dev(qweight, scales, x)
    x = _want(x.reshape(-1), torch.bfloat16, "x", (cols,))
    k = int(k)
    if not 0 <= k:
        raise RuntimeError("k must be >= 0")
    if rows > lib.dip_topk_max_n():
        raise RuntimeError(f"top-k supports n <= {lib.dip_topk_max_n()}, got {rows}")
    if g is None:
        g = torch.empty(rows, dtype=torch.bfloat16, device=dev)
    if idx is None:
        idx = torch.empty(k, dtype=torch.int32, device=dev)
    ws = workspace(dev, lib.dip_topk_workspace_size(rows), "topk")
    _check(lib.dip_gate_silu_topk(_ptr(qweight), _ptr(scales), _ptr(x), _ptr(g), _ptr(idx), rows,
                                  cols, k, _ptr(ws), ws.numel(), _stream(dev)),
           "dip_gate_silu_topk")
    return g, idx


def _indices(idx: torch.Tensor, name="indices") -> torch.Tensor:
    if idx.dtype == torch.int64:
        idx = idx.to(torch.int32)
    return _want(idx.reshape(-1), torch.int32, name)


def int4_gather_gemv(qweight, scales, x, indices, out=None):
    qweight, scales, rows, cols = _weights(qweight, scales, "int4_gather_gemv")
    dev = _dev(qweight, scales, x, indices)
    x = _want(x.reshape(-1), torch.bfloat16, "x", (cols,))
    indices = _indices(indices)
    k = indices.numel()
    if out is None:
        out = torch.empty(k, dtype=torch.bfloat16, device=dev)
    _check(lib.dip_int4_gather_gemv(_ptr(qweight), _ptr(scales), _ptr(x), _ptr(indices),
                                    _ptr(out), rows, cols, k, _stream(dev)),
           "dip_int4_gather_gemv")
    return out


def up_gather_h(qweight, scales, x, indices, g, out=None):
    """h[j] = bf16(g[indices[j]] * bf16(up[indices[j]] . x))."""
    qweight, scales, rows, cols = _weights(qweight, scales, "up_gather_h")
    dev = _dev(qweight, scales, x, indices, g)
    x = _want(x.reshape(-1), torch.bfloat16, "x", (cols,))
    g = _want(g.reshape(-1), torch.bfloat16, "g", (rows,))
    indices = _indices(indices)
    k = indices.numel()
    if out is None:
        out = torch.empty(k, dtype=torch.bfloat16, device=dev)
    _check(lib.dip_up_gather_h(_ptr(qweight), _ptr(scales), _ptr(x), _ptr(indices), _ptr(g),
                               _ptr(out), rows, cols, k, _stream(dev)), "dip_up_gather_h")
    return out


def int4_gather_down(down_t, scales, h, indices=None, out=None):
    """y[o] = bf16(sum_j h[j] * (q*s)[row_j, o]); row_j = indices[j] or j."""
    down_t, scales, rows, out_f = _weights(down_t, scales, "int4_gather_down")
    dev = _dev(down_t, scales, h)
    h = _want(h.reshape(-1), torch.bfloat16, "h_sel")
    k = h.numel()
    if indices is not None:
        indices = _indices(indices)
        if indices.numel() != k:
            raise RuntimeError("indices and h_sel must have the same length")
    elif k > rows:
        raise RuntimeError(f"h_sel has {k} entries but down_t_sel has {rows} rows")
    if out is None:
        out = torch.empty(out_f, dtype=torch.bfloat16, device=dev)
    nbytes = lib.dip_gather_down_workspace_size(k, out_f)
    ws = workspace(dev, nbytes, "down")
    _check(lib.dip_int4_gather_down(_ptr(down_t), _ptr(scales), _ptr(h), _ptr(indices),
                                    _ptr(out), rows, out_f, k, _ptr(ws), ws.numel(),
                                    _stream(dev)), "dip_int4_gather_down")
    return out


def int4_gather_down_by_channel(down_t, scales, h_full, indices, out=None, h_out=None,
                                scales_gm=None):
    """y[o] = bf16(sum_j h_full[indices[j]] * (q*s)[indices[j], o]) with h
    indexed by channel (the decode step's form); h_out[j] (if given) gets
    h_full[indices[j]].  indices=None: every row in order (indices[j] = j,
    k = rows).  scales_gm: the group-major copy of scales
    (scales_group_major), read instead of scales when given."""
    down_t, scales, rows, out_f = _weights(down_t, scales, "int4_gather_down_by_channel")
    scales_gm = _scales_gm(scales_gm, scales)
    dev = _dev(down_t, scales, h_full, *(() if indices is None else (indices,)))
    h_full = _want(h_full.reshape(-1), torch.bfloat16, "h_full", (rows,))
    if indices is None:
        k = rows
    else:
        indices = _indices(indices)
        k = indices.numel()
    if h_out is not None:
        h_out = _want(h_out, torch.bfloat16, "h_out", (k,))
    if out is None:
        out = torch.empty(out_f, dtype=torch.bfloat16, device=dev)
    nbytes = lib.dip_gather_down_workspace_size(k, out_f)
    ws = workspace(dev, nbytes, "down")
    _check(lib.dip_int4_gather_down_by_channel(_ptr(down_t), _ptr(scales), _ptr(scales_gm),
                                               _ptr(h_full), _ptr(indices), _ptr(out),
                                               _ptr(h_out), rows,
                                               out_f, k, _ptr(ws), ws.numel(), _stream(dev)),
           "dip_int4_gather_down_by_channel")
    return out


def ca_fused_gemv(res_qw, res_sc, str_qw, str_sc, x, src, row, g=None, gid=None, out=None):
    res_qw, res_sc, res_rows, cols = _weights(res_qw, res_sc, "ca_fused_gemv.res")
    str_qw, str_sc, str_rows, cols2 = _weights(str_qw, str_sc, "ca_fused_gemv.str")
    if cols2 != cols:
        raise RuntimeError("resident and streamed rows differ in width")
    dev = _dev(res_qw, str_qw, x, src, row)
    x = _want(x.reshape(-1), torch.bfloat16, "x", (cols,))
    src = _indices(src, "src")
    row = _indices(row, "row")
    k = src.numel()
    if row.numel() != k:
        raise RuntimeError("src and row must have the same length")
    if g is not None:
        g = _want(g.reshape(-1), torch.bfloat16, "g")
        gid = _indices(gid, "gid")
    if out is None:
        out = torch.empty(k, dtype=torch.bfloat16, device=dev)
    g_len = g.numel() if g is not None else 0
    _check(lib.dip_ca_fused_gemv(_ptr(res_qw), _ptr(res_sc), _ptr(str_qw), _ptr(str_sc),
                                 _ptr(x), _ptr(src), _ptr(row), _ptr(g), _ptr(gid), g_len,
                                 _ptr(out), res_rows, str_rows, cols, k, _stream(dev)),
           "dip_ca_fused_gemv")
    return out


def ca_down(res_qw, res_sc, str_qw, str_sc, h, src, row, out=None):
    res_qw, res_sc, res_rows, out_f = _weights(res_qw, res_sc, "ca_down.res")
    str_qw, str_sc, str_rows, out_f2 = _weights(str_qw, str_sc, "ca_down.str")
    if out_f2 != out_f:
        raise RuntimeError("resident and streamed rows differ in width")
    dev = _dev(res_qw, str_qw, h, src, row)
    h = _want(h.reshape(-1), torch.bfloat16, "h")
    src = _indices(src, "src")
    row = _indices(row, "row")
    k = h.numel()
    if out is None:
        out = torch.empty(out_f, dtype=torch.bfloat16, device=dev)
    nbytes = lib.dip_gather_down_workspace_size(k, out_f)
    ws = workspace(dev, nbytes, "down")
    _check(lib.dip_ca_down(_ptr(res_qw), _ptr(res_sc), _ptr(str_qw), _ptr(str_sc), _ptr(h),
                           _ptr(src), _ptr(row), _ptr(out), res_rows, str_rows, out_f, k,
                           _ptr(ws), ws.numel(), _stream(dev)), "dip_ca_down")
    return out


def ca_assemble(id2slot: torch.Tensor, idx: torch.Tensor):
    """Returns (combined int32 [k], src int32 [k], row int32 [k],
    miss_ids int32 [k] (first n_miss valid), counts int32 [2] = n_hit, n_miss)."""
    dev = _dev(id2slot, idx)
    id2slot = _want(id2slot.reshape(-1), torch.int64, "id2slot")
    idx = _indices(idx, "idx")
    k = idx.numel()
    combined = torch.empty(k, dtype=torch.int32, device=dev)
    src = torch.empty_like(combined)
    row = torch.empty_like(combined)
    miss = torch.empty_like(combined)
    counts = torch.empty(2, dtype=torch.int32, device=dev)
    _check(lib.dip_ca_assemble(_ptr(id2slot), _ptr(idx), _ptr(combined), _ptr(src), _ptr(row),
                               _ptr(miss), _ptr(counts), id2slot.numel(), k, _stream(dev)),
           "dip_ca_assemble")
    return combined, src, row, miss, counts


def swiglu(g, u):
    """bf16(bf16(silu(g)) * u) of two contiguous bf16 tensors of one shape."""
    dev = _dev(g, u)
    g = _want(g, torch.bfloat16, "g")
    u = _want(u, torch.bfloat16, "u", g.shape)
    out = torch.empty_like(g)
    _check(lib.dip_swiglu(_ptr(g), _ptr(u), _ptr(out), g.numel(), _stream(dev)), "dip_swiglu")
    return out


def dequant_t(qweight, scales):
    """The transpose of bf16(q*s), contiguous [cols, rows] (rows a multiple of
    8)."""
    qweight, scales, rows, cols = _weights(qweight, scales, "dequant_t")
    dev = _dev(qweight, scales)
    out = torch.empty(cols, rows, dtype=torch.bfloat16, device=dev)
    _check(lib.dip_dequant_t(_ptr(qweight), _ptr(scales), _ptr(out), rows, cols, _stream(dev)),
           "dip_dequant_t")
    return out


def dequant_rows(qweight, scales, indices=None, mode: int = 0):
    """mode 0: float32 q*s; mode 1: bf16(q*s) (qlinear.dequantize)."""
    qweight, scales, rows, cols = _weights(qweight, scales, "dequant_rows")
    dev = _dev(qweight, scales)
    if indices is not None:
        indices = _indices(indices)
        n = indices.numel()
    else:
        n = rows
    out = torch.empty(n, cols, dtype=torch.float32 if mode == 0 else torch.bfloat16,
                      device=dev)
    _check(lib.dip_dequant_rows(_ptr(qweight), _ptr(scales), _ptr(indices), _ptr(out), n, rows,
                                cols, int(mode), _stream(dev)), "dip_dequant_rows")
    return out


def quantize_int4(w: torch.Tensor):
    """Device int4 g128 quantization, bit-exact with the reference quantizer."""
    dev = _dev(w)
    if w.dim() != 2 or w.shape[1] % GROUP_SIZE:
        raise RuntimeError("w must be 2-D with in_features a multiple of 128")
    bf = w.dtype == torch.bfloat16
    w = w.contiguous() if bf else w.float().contiguous()
    rows, cols = w.shape
    qw = torch.empty(rows, cols // 2, dtype=torch.int8, device=dev)
    sc = torch.empty(rows, cols // GROUP_SIZE, dtype=torch.bfloat16, device=dev)
    _check(lib.dip_quantize_int4(_ptr(w), int(bf), _ptr(qw), _ptr(sc), rows, cols, _stream(dev)),
           "dip_quantize_int4")
    return qw, sc


def transpose_down_int4(down_qw, down_sc):
    """down [out, inter/2] int4 -> down_t [inter, out/2] int4 on the device."""
    down_qw, down_sc, out_f, inter = _weights(down_qw, down_sc, "down")
    dev = _dev(down_qw, down_sc)
    tq = torch.empty(inter, out_f // 2, dtype=torch.int8, device=dev)
    ts = torch.empty(inter, out_f // GROUP_SIZE, dtype=torch.bfloat16, device=dev)
    _check(lib.dip_transpose_down_int4(_ptr(down_qw), _ptr(down_sc), _ptr(tq), _ptr(ts), out_f,
                                       inter, _stream(dev)), "dip_transpose_down_int4")
    return tq, ts


def scales_group_major(scales: torch.Tensor) -> torch.Tensor:
    """The group-major copy [groups, rows] of a [rows, groups] bf16 scale
    matrix (dip_scales_group_major): the layout the decode step's down stage
    reads down_t's scales in when given one."""
    if scales.dtype != torch.bfloat16 or scales.dim() != 2 or not scales.is_contiguous():
        raise RuntimeError("scales must be a contiguous 2-D bf16 tensor")
    rows, groups = scales.shape
    out = torch.empty(groups, rows, dtype=torch.bfloat16, device=scales.device)
    _check(lib.dip_scales_group_major(_ptr(scales), _ptr(out), rows, groups,
                                      _stream(scales.device)), "dip_scales_group_major")
    return out


def _scales_gm(scales_gm, scales):
    """scales_gm checked against its row-major scales (None passes)."""
    if scales_gm is None:
        return None
    rows, groups = scales.shape
    if (scales_gm.dtype != torch.bfloat16 or tuple(scales_gm.shape) != (groups, rows)
            or not scales_gm.is_contiguous() or scales_gm.device != scales.device):
        raise RuntimeError(f"scales_gm must be a contiguous bf16 [{groups}, {rows}] tensor on "
                           f"{scales.device} (scales_group_major of the scales)")
    return scales_gm


def mlp_workspace_bytes(hidden: int, inter: int, k: int) -> int:
    return lib.dip_mlp_workspace_size(hidden, inter, k)


def mlp_state(device) -> torch.Tensor:
    """A zeroed per-layer decode state for mlp_decode (speculative up rows)."""
    n = lib.dip_mlp_state_size()
    return torch.zeros(n // 4, dtype=torch.int32, device=device)


def mlp_decode(gate_qw, gate_sc, up_qw, up_sc, down_t_qw, down_t_sc, x, k, *, y=None, g=None,
               idx=None, h=None, ws=None, state=None, down_t_sc_gm=None):
    """One resident DIP MLP decode step; returns (y, g, idx, h).

    state: this layer's mlp_state() tensor, kept across calls.  With it the
    step overlaps the top-k with up rows of the channels the last call ranked
    highest (same outputs, bit for bit); without it the step runs stage by
    stage.  down_t_sc_gm: scales_group_major(down_t_sc), which the down
    stage then reads (same outputs, bit for bit)."""
    gate_qw, gate_sc, inter, hidden = _weights(gate_qw, gate_sc, "gate")
    up_qw, up_sc, inter2, hidden2 = _weights(up_qw, up_sc, "up")
    down_t_qw, down_t_sc, inter3, hidden3 = _weights(down_t_qw, down_t_sc, "down_t")
    if not (inter == inter2 == inter3 and hidden == hidden2 == hidden3):
        raise RuntimeError("gate/up/down_t shapes disagree")
    dev = _dev(gate_qw, up_qw, down_t_qw, x)
    x = _want(x.reshape(-1), torch.bfloat16, "x", (hidden,))
    k = int(k)
    if not 0 <= k <= inter:
        raise RuntimeError(f"k={k} outside [0, {inter}]")
    if y is None:
        y = torch.empty(hidden, dtype=torch.bfloat16, device=dev)
    if g is None:
        g = torch.empty(inter, dtype=torch.bfloat16, device=dev)
    if idx is None:
        idx = torch.empty(k, dtype=torch.int32, device=dev)
    if h is None:
        h = torch.empty(k, dtype=torch.bfloat16, device=dev)
    nbytes = lib.dip_mlp_workspace_size(hidden, inter, k)
    if ws is None:
        ws = workspace(dev, nbytes, "mlp")
    elif ws.numel() < nbytes:
        raise RuntimeError("workspace too small")
    if state is not None:
        if (state.device != dev or state.dtype != torch.int32 or not state.is_contiguous()
                or state.numel() * 4 < lib.dip_mlp_state_size()):
            raise RuntimeError("state must be this device's mlp_state() tensor")
    down_t_sc_gm = _scales_gm(down_t_sc_gm, down_t_sc)
    _check(lib.dip_mlp_decode(_ptr(gate_qw), _ptr(gate_sc), _ptr(up_qw), _ptr(up_sc),
                              _ptr(down_t_qw), _ptr(down_t_sc), _ptr(down_t_sc_gm), _ptr(x),
                              _ptr(y), _ptr(g),
                              _ptr(idx), _ptr(h), hidden, inter, k, _ptr(ws), ws.numel(),
                              None if state is None else _ptr(state), _stream(dev)),
           "dip_mlp_decode")
    return y, g, idx, h


def mlp_decode_noalloc(gate_qw, gate_sc, up_qw, up_sc, down_t_qw, down_t_sc, x, k, *, y, g,
                       idx, h, state=None, down_t_sc_gm=None):
    """mlp_decode with the workspace in the library's per-GPU scratch array
    (dip_mlp_decode_noalloc): the caller passes every output, nothing is
    allocated.  Calls that overlap on one GPU race on the scratch array."""
    gate_qw, gate_sc, inter, hidden = _weights(gate_qw, gate_sc, "gate")
    up_qw, up_sc, inter2, hidden2 = _weights(up_qw, up_sc, "up")
    down_t_qw, down_t_sc, inter3, hidden3 = _weights(down_t_qw, down_t_sc, "down_t")
    if not (inter == inter2 == inter3 and hidden == hidden2 == hidden3):
        raise RuntimeError("gate/up/down_t shapes disagree")
    dev = _dev(gate_qw, up_qw, down_t_qw, x)
    k = int(k)
    if not 0 <= k <= inter:
        raise RuntimeError(f"k={k} outside [0, {inter}]")
    x = x.reshape(-1)
    for t, dt, name, shape in ((x, torch.bfloat16, "x", (hidden,)), (y, torch.bfloat16, "y", (hidden,)),
                               (g, torch.bfloat16, "g", (inter,)), (idx, torch.int32, "idx", (k,)),
                               (h, torch.bfloat16, "h", (k,))):
        # used in place: a copy would allocate (and outputs would land in it)
        if (not isinstance(t, torch.Tensor) or t.dtype != dt or tuple(t.shape) != shape
                or t.device != dev or not t.is_contiguous() or t.data_ptr() % 16):
            raise RuntimeError(f"{name} must be a contiguous 16-byte aligned {dt} tensor of "
                               f"shape {shape} on {dev}")
    if state is not None:
        if (state.device != dev or state.dtype != torch.int32 or not state.is_contiguous()
                or state.numel() * 4 < lib.dip_mlp_state_size()):
            raise RuntimeError("state must be this device's mlp_state() tensor")
    down_t_sc_gm = _scales_gm(down_t_sc_gm, down_t_sc)
    _check(lib.dip_mlp_decode_noalloc(_ptr(gate_qw), _ptr(gate_sc), _ptr(up_qw), _ptr(up_sc),
                                      _ptr(down_t_qw), _ptr(down_t_sc), _ptr(down_t_sc_gm),
                                      _ptr(x), _ptr(y), _ptr(g),
                                      _ptr(idx), _ptr(h), hidden, inter, k,
                                      None if state is None else _ptr(state), _stream(dev)),
           "dip_mlp_decode_noalloc")
    return y, g, idx, h


# ---------------------------------------------------------------------------
# one-token decode steps of a Qwen3 decoder layer (whole-model decode loop)
# ---------------------------------------------------------------------------
def _bf16_vec(t: torch.Tensor, n: int, name: str) -> torch.Tensor:
    if t.dtype != torch.bfloat16 or not t.is_contiguous() or t.numel() != n:
        raise RuntimeError(f"{name} must be a contiguous bf16 tensor of {n} values")
    return t


def _pos_tensor(pos: torch.Tensor, dev) -> torch.Tensor:
    if pos.dtype != torch.int64 or pos.numel() < 1 or pos.device != dev:
        raise RuntimeError("pos must be an int64 tensor on the device")
    return pos


def _add_rmsnorm(h, add, weight, out, eps: float, rows: int, n: int):
    dev = _dev(h, weight, out)
    _bf16_vec(h, rows * n, "h")
    _bf16_vec(weight, n, "weight")
    _bf16_vec(out, rows * n, "out")
    if add is not None:
        _dev(add)
        if add.device != dev:
            raise RuntimeError("add must be on h's device")
        _bf16_vec(add, rows * n, "add")
    _check(lib.dip_add_rmsnorm_rows(_ptr(h), _ptr(add), _ptr(weight), _ptr(out), rows, n,
                                    float(eps), _stream(dev)), "dip_add_rmsnorm")
    return out


def add_rmsnorm(h, add, weight, out, eps: float):
    """In place h = bf16(h + add) (when add is given), then
    out = bf16(weight * bf16(h * rsqrt(mean(h^2) + eps)))."""
    return _add_rmsnorm(h, add, weight, out, eps, 1, h.numel())


def add_rmsnorm_rows(h, add, weight, out, eps: float):
    """add_rmsnorm of each row of h [rows, n] (a prompt's tokens)."""
    return _add_rmsnorm(h, add, weight, out, eps, *h.shape)


def _qk_check(qkv, q_norm_w, k_norm_w, cos, sin, q_out, k_cache, v_cache, n_heads, n_kv_heads,
              tokens):
    dev = _dev(qkv, q_out, k_cache, v_cache)
    hd = q_norm_w.numel()
    if k_cache.dim() != 3 or k_cache.shape != v_cache.shape or k_cache.shape[0] != n_kv_heads \
            or k_cache.shape[2] != hd:
        raise RuntimeError("k_cache / v_cache must be [n_kv_heads, max_len, head_dim]")
    max_len = k_cache.shape[1]
    _bf16_vec(qkv, tokens * (n_heads + 2 * n_kv_heads) * hd, "qkv")
    _bf16_vec(q_norm_w, hd, "q_norm_w")
    _bf16_vec(k_norm_w, hd, "k_norm_w")
    _bf16_vec(cos, max_len * hd, "cos")
    _bf16_vec(sin, max_len * hd, "sin")
    _bf16_vec(q_out, tokens * n_heads * hd, "q_out")
    _bf16_vec(k_cache, n_kv_heads * max_len * hd, "k_cache")
    _bf16_vec(v_cache, n_kv_heads * max_len * hd, "v_cache")
    for t in (q_norm_w, k_norm_w, cos, sin):
        if t.device != dev:
            raise RuntimeError("all tensors must be on one device")
    return dev, hd, max_len


def qk_norm_rope_cache(qkv, q_norm_w, k_norm_w, cos, sin, pos, q_out, k_cache, v_cache,
                       n_heads: int, n_kv_heads: int, eps: float):
    """q/k head RMSNorm + rotary embedding at `pos` for one token's q|k|v;
    q -> q_out, k and v -> row pos of the [n_kv_heads, max_len, head_dim]
    caches."""
    dev, hd, max_len = _qk_check(qkv, q_norm_w, k_norm_w, cos, sin, q_out, k_cache, v_cache,
                                 n_heads, n_kv_heads, 1)
    _pos_tensor(pos, dev)
    _check(lib.dip_qk_norm_rope_cache(_ptr(qkv), _ptr(q_norm_w), _ptr(k_norm_w), _ptr(cos),
                                      _ptr(sin), _ptr(pos), _ptr(q_out), _ptr(k_cache),
                                      _ptr(v_cache), n_heads, n_kv_heads, hd, max_len,
                                      float(eps), _stream(dev)), "dip_qk_norm_rope_cache")
    return q_out


def qk_norm_rope_cache_rows(qkv, q_norm_w, k_norm_w, cos, sin, q_out, k_cache, v_cache,
                            n_heads: int, n_kv_heads: int, eps: float):
    """qk_norm_rope_cache for the tokens of a prompt: row t of qkv [tokens, ..]
    at position t, q to row t of q_out, k and v to row t of the caches."""
    tokens = qkv.shape[0]
    dev, hd, max_len = _qk_check(qkv, q_norm_w, k_norm_w, cos, sin, q_out, k_cache, v_cache,
                                 n_heads, n_kv_heads, tokens)
    _check(lib.dip_qk_norm_rope_cache_rows(_ptr(qkv), _ptr(q_norm_w), _ptr(k_norm_w), _ptr(cos),
                                           _ptr(sin), _ptr(q_out), _ptr(k_cache), _ptr(v_cache),
                                           tokens, n_heads, n_kv_heads, hd, max_len, float(eps),
                                           _stream(dev)), "dip_qk_norm_rope_cache_rows")
    return q_out


def decode_attention_workspace_bytes(n_heads: int, head_dim: int, max_len: int) -> int:
    return lib.dip_decode_attention_workspace_size(n_heads, head_dim, max_len)


def decode_attention(q, k_cache, v_cache, pos, out, scale: float, ws=None):
    """Grouped-query attention of one token (q [n_heads, head_dim]) over
    rows 0..pos of the [n_kv_heads, max_len, head_dim] caches -> out."""
    dev = _dev(q, k_cache, v_cache, out)
    if k_cache.dim() != 3 or k_cache.shape != v_cache.shape:
        raise RuntimeError("k_cache / v_cache must be [n_kv_heads, max_len, head_dim]")
    nkv, max_len, hd = k_cache.shape
    nh = q.numel() // hd
    _bf16_vec(q, nh * hd, "q")
    _bf16_vec(out, nh * hd, "out")
    _bf16_vec(k_cache, nkv * max_len * hd, "k_cache")
    _bf16_vec(v_cache, nkv * max_len * hd, "v_cache")
    _pos_tensor(pos, dev)
    nbytes = decode_attention_workspace_bytes(nh, hd, max_len)
    if ws is None:
        ws = workspace(dev, nbytes, "attention")
    elif ws.numel() < nbytes or ws.device != dev:
        raise RuntimeError("attention workspace too small")
    _check(lib.dip_decode_attention(_ptr(q), _ptr(k_cache), _ptr(v_cache), _ptr(pos), _ptr(out),
                                    nh, nkv, hd, max_len, float(scale), _ptr(ws), ws.numel(),
                                    _stream(dev)), "dip_decode_attention")
    return out


def decode_attention_fused_max_len() -> int:
    return lib.dip_decode_attention_fused_max_len()


def decode_attention_fused(qkv, q_norm_w, k_norm_w, cos, sin, pos, k_cache, v_cache, out,
                           n_heads: int, n_kv_heads: int, eps: float, scale: float):
    """qk_norm_rope_cache followed by decode_attention in one launch (caches
    of at most decode_attention_fused_max_len() rows)."""
    dev = _dev(qkv, k_cache, v_cache, out)
    hd = q_norm_w.numel()
    if k_cache.dim() != 3 or k_cache.shape != v_cache.shape or k_cache.shape[0] != n_kv_heads \
            or k_cache.shape[2] != hd:
        raise RuntimeError("k_cache / v_cache must be [n_kv_heads, max_len, head_dim]")
    max_len = k_cache.shape[1]
    _bf16_vec(qkv, (n_heads + 2 * n_kv_heads) * hd, "qkv")
    _bf16_vec(q_norm_w, hd, "q_norm_w")
    _bf16_vec(k_norm_w, hd, "k_norm_w")
    _bf16_vec(cos, max_len * hd, "cos")
    _bf16_vec(sin, max_len * hd, "sin")
    _bf16_vec(out, n_heads * hd, "out")
    _bf16_vec(k_cache, n_kv_heads * max_len * hd, "k_cache")
    _bf16_vec(v_cache, n_kv_heads * max_len * hd, "v_cache")
    for t in (q_norm_w, k_norm_w, cos, sin):
        if t.device != dev:
            raise RuntimeError("all tensors must be on one device")
    _pos_tensor(pos, dev)
    _check(lib.dip_decode_attention_fused(_ptr(qkv), _ptr(q_norm_w), _ptr(k_norm_w), _ptr(cos),
                                          _ptr(sin), _ptr(pos), _ptr(k_cache), _ptr(v_cache),
                                          _ptr(out), n_heads, n_kv_heads, hd, max_len,
                                          float(eps), float(scale), _stream(dev)),
           "dip_decode_attention_fused")
    return out


def mlp_decode_rmsnorm(gate_qw, gate_sc, up_qw, up_sc, down_t_qw, down_t_sc, res, add, norm_w,
                       eps: float, k, *, res_out=None, x_out=None, y=None, g=None, idx=None,
                       h=None, ws=None, state=None, down_t_sc_gm=None):
    """mlp_decode on x = RMSNorm(res + add) * norm_w, the norm folded into the
    gate launch; the updated residual goes to res_out (if given) and x to
    x_out.  Returns (y, g, idx, h, x_out)."""
    gate_qw, gate_sc, inter, hidden = _weights(gate_qw, gate_sc, "gate")
    dev = _dev(gate_qw, res, norm_w)
    _bf16_vec(res, hidden, "res")
    _bf16_vec(norm_w, hidden, "norm_w")
    for name, t in (("add", add), ("res_out", res_out), ("x_out", x_out)):
        if t is not None:
            _bf16_vec(t, hidden, name)
            if t.device != dev:
                raise RuntimeError(f"{name} must be on the weights' device")
    k = int(k)
    if not 0 <= k <= inter:
        raise RuntimeError(f"k={k} outside [0, {inter}]")
    if x_out is None:
        x_out = torch.empty(hidden, dtype=torch.bfloat16, device=dev)
    if y is None:
        y = torch.empty(hidden, dtype=torch.bfloat16, device=dev)
    if g is None:
        g = torch.empty(inter, dtype=torch.bfloat16, device=dev)
    if idx is None:
        idx = torch.empty(k, dtype=torch.int32, device=dev)
    if h is None:
        h = torch.empty(k, dtype=torch.bfloat16, device=dev)
    nbytes = lib.dip_mlp_workspace_size(hidden, inter, k)
    if ws is None:
        ws = workspace(dev, nbytes, "mlp")
    elif ws.numel() < nbytes:
        raise RuntimeError("workspace too small")
    if state is not None and (state.device != dev or state.dtype != torch.int32
                              or state.numel() * 4 < lib.dip_mlp_state_size()):
        raise RuntimeError("state must be this device's mlp_state() tensor")
    down_t_sc_gm = _scales_gm(down_t_sc_gm, down_t_sc)
    _check(lib.dip_mlp_decode_rmsnorm(
        _ptr(gate_qw), _ptr(gate_sc), _ptr(up_qw), _ptr(up_sc), _ptr(down_t_qw), _ptr(down_t_sc),
        _ptr(down_t_sc_gm), _ptr(res), _ptr(add), _ptr(norm_w), float(eps), _ptr(res_out), _ptr(x_out), _ptr(y),
        _ptr(g), _ptr(idx), _ptr(h), hidden, inter, k, _ptr(ws), ws.numel(),
        None if state is None else _ptr(state), _stream(dev)), "dip_mlp_decode_rmsnorm")
    return y, g, idx, h, x_out


TUNE = {"rowdot_wgs_per_cu": 0, "topk_stamps": 1, "spec_margin": 2, "row_tiers": 4}


TIMELINE_KERNELS = {"gate": 0, "topk_spec_up": 1, "down_partials": 2, "down_reduce": 3}
STAMP_BLOCKS, STAMP_WAVES = 2048, 16


def timeline_read(kernel: str):
    """The last launch's per-workgroup stamps of one decode kernel (the
    timeline build of the library only; dip_timeline_read): (start [blocks],
    end [blocks, waves], xcc [blocks]) as numpy arrays in s_memrealtime ticks
    (100 MHz), end entries older than their workgroup's start being waves that
    did not reach the end of this launch."""
    import numpy as np
    buf = np.zeros(STAMP_BLOCKS + STAMP_BLOCKS * STAMP_WAVES + STAMP_BLOCKS // 2 + 1,
                   dtype=np.uint64)
    _check(lib.dip_timeline_read(TIMELINE_KERNELS[kernel], buf.ctypes.data), "dip_timeline_read")
    start = buf[:STAMP_BLOCKS].astype(np.int64)
    end = buf[STAMP_BLOCKS:STAMP_BLOCKS * (1 + STAMP_WAVES)].astype(np.int64).reshape(
        STAMP_BLOCKS, STAMP_WAVES)
    tail = buf[STAMP_BLOCKS * (1 + STAMP_WAVES):].view(np.uint32)
    xcc = tail[:STAMP_BLOCKS].astype(np.int64)
    blocks = int(min(tail[STAMP_BLOCKS], STAMP_BLOCKS))
    return start[:blocks], end[:blocks], xcc[:blocks]


def set_tuning(name: str, value: int) -> None:
    """Launch tuning knob (speed only; see DIP_TUNE_* in include/dip_hip.h)."""
    _check(lib.dip_set_tuning(TUNE[name], int(value)), f"dip_set_tuning({name}={value})")


def get_tuning(name: str) -> int:
    return lib.dip_get_tuning(TUNE[name])


# DIP_TUNE="knob=value,knob=value" applies launch tuning at import (profiling
# and sweeps run unmodified programs this way).
for _kv in filter(None, os.environ.get("DIP_TUNE", "").split(",")):
    _k, _v = _kv.split("=")
    set_tuning(_k.strip(), int(_v))


def host_gather_rows(src: torch.Tensor, ids: torch.Tensor, dst: torch.Tensor,
                     threads: int = 8) -> None:
    """dst[i] = src[ids[i]] row-wise on the host (pinned index_select of
    dip_ca.py:148-153) with `threads` native threads."""
    if src.device.type != "cpu" or dst.device.type != "cpu" or ids.device.type != "cpu":
        raise RuntimeError("host_gather_rows works on host tensors")
    if not (src.is_contiguous() and dst.is_contiguous()):
        raise RuntimeError("host_gather_rows needs contiguous src/dst")
    ids = ids.to(torch.int32).contiguous()
    n = ids.numel()
    row_bytes = src[0].numel() * src.element_size() if src.shape[0] else 0
    if dst.shape[0] < n or dst[0].numel() * dst.element_size() != row_bytes:
        raise RuntimeError("dst too small or row size mismatch")
    _check(lib.dip_host_gather_rows(_ptr(src), _ptr(ids), _ptr(dst), n, row_bytes, src.shape[0],
                                    int(threads)), "dip_host_gather_rows")


def _host_pieces(srcs, dsts, n):
    """Row sizes of matching host matrices (same row count in srcs, at least
    n rows in dsts)."""
    if len(srcs) != len(dsts) or not srcs:
        raise RuntimeError("need matching, non-empty src/dst lists")
    rows = srcs[0].shape[0]
    rbs = []
    for s, d in zip(srcs, dsts):
        if s.device.type != "cpu" or d.device.type != "cpu":
            raise RuntimeError("host row gathers work on host tensors")
        if not (s.is_contiguous() and d.is_contiguous()):
            raise RuntimeError("host row gathers need contiguous src/dst")
        if s.shape[0] != rows:
            raise RuntimeError("every source needs the same row count")
        rb = s[0].numel() * s.element_size() if rows else 0
        if d.shape[0] < n or (n and d[0].numel() * d.element_size() != rb):
            raise RuntimeError("dst too small or row size mismatch")
        rbs.append(rb)
    return rows, rbs


def _ptr_array(ts):
    return (ctypes.c_void_p * len(ts))(*[t.data_ptr() for t in ts])


def host_gather_rows_multi(srcs, ids: torch.Tensor, dsts, threads: int = 8) -> None:
    """dsts[p][i] = srcs[p][ids[i]] for every matrix p (same row count) in
    one pass of the native host thread pool: the index_selects of one miss
    set (dip_ca.py:148-153)."""
    if ids.device.type != "cpu":
        raise RuntimeError("host_gather_rows_multi works on host tensors")
    ids = ids.to(torch.int32).contiguous()
    n = ids.numel()
    rows, rbs = _host_pieces(srcs, dsts, n)
    src_arr, dst_arr = _ptr_array(srcs), _ptr_array(dsts)
    rb_arr = (ctypes.c_int64 * len(rbs))(*rbs)
    _check(lib.dip_host_gather_rows_multi(ctypes.addressof(src_arr), ctypes.addressof(dst_arr),
                                          ctypes.addressof(rb_arr), len(rbs), _ptr(ids), n, rows,
                                          int(threads)), "dip_host_gather_rows_multi")


def stream_rows(srcs, ids: torch.Tensor, count: torch.Tensor, dsts) -> bool:
    """dsts[p][i] = srcs[p][ids[i]] for i < count[0], read by the device from
    the pinned host matrices srcs (ids and count: int32 on the device), queued
    on the current stream.  False, with nothing queued, where a source is not
    pinned."""
    dev = _dev(*dsts, ids, count)
    if ids.dtype != torch.int32 or count.dtype != torch.int32 or not ids.is_contiguous():
        raise RuntimeError("ids and count must be contiguous int32 tensors")
    rows, rbs = srcs[0].shape[0], []
    max_rows = ids.numel()
    if len(dsts) != len(srcs):
        raise RuntimeError("need one device destination per source")
    for s, d in zip(srcs, dsts):
        if s.device.type != "cpu" or not s.is_contiguous() or not d.is_contiguous():
            raise RuntimeError("stream_rows copies contiguous host rows to contiguous device rows")
        rb = s.stride(0) * s.element_size()
        if s.shape[0] != rows or d.stride(0) * d.element_size() != rb:
            raise RuntimeError("row count or row size mismatch")
        if d.shape[0] < max_rows:
            raise RuntimeError("device destination too small")
        rbs.append(rb)
    src_arr, dst_arr = _ptr_array(srcs), _ptr_array(dsts)
    rb_arr = (ctypes.c_int64 * len(rbs))(*rbs)
    st = lib.dip_stream_rows(ctypes.addressof(src_arr), ctypes.addressof(dst_arr),
                             ctypes.addressof(rb_arr), len(rbs), _ptr(ids), _ptr(count), max_rows,
                             rows, _stream(dev))
    if st == -4:  # DIP_ERR_UNSUPPORTED
        return False
    _check(st, "dip_stream_rows")
    return True


def host_stream_rows(srcs, ids: torch.Tensor, pinned, dsts, chunk_rows: int = 2048,
                     threads: int = 8, stream=None, timing: bool = False):
    """Gather rows srcs[p][ids] into the pinned host staging pinned[p] and
    copy them to the device tensors dsts[p] (rows 0 .. n-1), chunk by chunk
    so that a chunk's copy overlaps the next chunk's gather: the miss stream
    of dip_ca.py:146-156.  The first half of the pieces is copied on
    `stream` (default: the current stream of dsts' device), the rest on the
    library's second copy stream, which `stream` then waits for.  Returns
    once the copies are queued; with timing, waits for them and returns the
    summed copy time in ms (per chunk, the longer of the two streams), else
    None."""
    if ids.device.type != "cpu":
        raise RuntimeError("host_stream_rows takes host ids")
    ids = ids.to(torch.int32).contiguous()
    n = ids.numel()
    rows, rbs = _host_pieces(srcs, pinned, n)
    if len(dsts) != len(srcs):
        raise RuntimeError("need one device destination per source")
    dev = dsts[0].device
    for d, rb in zip(dsts, rbs):
        if d.device != dev or d.device.type != "cuda" or not d.is_contiguous():
            raise RuntimeError("destinations must be contiguous tensors on one GPU")
        if d.shape[0] < n or (n and d[0].numel() * d.element_size() != rb):
            raise RuntimeError("device destination too small or row size mismatch")
    if stream is None:
        stream = torch.cuda.current_stream(dev)
    src_arr, pin_arr, dst_arr = _ptr_array(srcs), _ptr_array(pinned), _ptr_array(dsts)
    rb_arr = (ctypes.c_int64 * len(rbs))(*rbs)
    ms = ctypes.c_float(0.0)
    _check(lib.dip_host_stream_rows(ctypes.addressof(src_arr), ctypes.addressof(pin_arr),
                                    ctypes.addressof(dst_arr), ctypes.addressof(rb_arr), len(rbs),
                                    _ptr(ids), n, rows, int(chunk_rows), int(threads),
                                    ctypes.c_void_p(stream.cuda_stream),
                                    ctypes.byref(ms) if timing else None),
           "dip_host_stream_rows")
    return float(ms.value) if timing else None
