"""int4 g128 symmetric format (drop-in for the reference's qlinear.py format
helpers, qlinear.py:25-88).

    qweight : int8 [out_features, in_features // 2]   two int4 per byte,
              low nibble = even column, high nibble = odd column
    scales  : bf16 [out_features, in_features // 128]

``dequantize`` on device tensors runs the HIP dequant kernel (bf16(q*s), the
same rounding as the reference); on host tensors it uses torch ops, which is
how the reference uses it at load time (e.g. the one-time down transpose).
``QuantLinear`` is the reference's projection layer (qlinear.py:67-88).  On
the GPU it reads the packed weight once instead of writing and re-reading a
bf16 copy: the int4 GEMV for one token, the int4 MFMA GEMM for prompts of up
to GEMM_MAX_TOKENS tokens (gate, up and the SwiGLU of an MLP in one launch up
to GATE_UP_MAX_TOKENS); longer prompts take the reference's dequant + F.linear
route.  Both kernels take the weights as exact fp32 q*s (the
reference rounds them to bf16 first), so they differ from dequant + F.linear
by rounding only.
``_replace_linears_with_quant`` and ``load_quantized_qwen3`` build the
reference's int4 baseline model (qlinear.py:91-166) with every weight
resident on one device.
"""
from __future__ import annotations

import functools
from pathlib import Path

import torch
import torch.nn as nn
import torch.nn.functional as F

GROUP_SIZE = 128
_QUANT_SUBSTRINGS = ("q_proj", "k_proj", "v_proj", "o_proj", "gate_proj", "up_proj", "down_proj")
# Input widths the int4 GEMV kernel is built for (its dispatch table:
# 32-column chunks split over 4..32 lanes per row).
_GEMV_COLS = frozenset((128, 256, 512, 1024, 1536, 2048, 2560, 3072, 4096, 5120, 6144, 8192))
# Prompts of up to this many tokens run the int4 MFMA GEMM (weights read
# once as nibbles) where _gemm_serves; longer ones dequantize once and use the
# library GEMM, which wins once the bf16 copy is amortised over enough tokens
# (us, int4 GEMM / both steps of the library route, each in a graph over layers
# that do not fit the caches: 25600 x 5120, 512 tokens 197 / 201, 704 tokens 247 /
# 263, 900 tokens 322 / 270; 12288 x 4096, 512 tokens 70 / 72, 576 tokens 91 / 80;
# 9728 x 2560, 512 tokens 44 / 47, 640 tokens 58 / 50).
GEMM_MAX_TOKENS = 512
# Up to this many rows it takes any input, rounded to bf16; beyond, plain bf16
# tensors only (_plain_bf16).
_ANY_INPUT_TOKENS = 64
# Gate and up in one launch win a little longer, whatever the shape (us, against
# both library products, their dequantisation and the SwiGLU, at 512 / 704 / 768 /
# 900 tokens: 25600 x 5120 374 / 426, 486 / 545, 512 / 539, 622 / 569; 12288 x 4096
# 145 / 164, 201 / 211, 210 / 201, 250 / 227; 9728 x 2560 74 / 101, 107 / 118, 124 /
# 124, 135 / 143; 3072 x 1024 18 / 41, 23 / 42, 24 / 42, 24 / 45.  Over ten shapes and
# 65 to 768 tokens the one launch is at most 8 % behind, at 17408 x 5120 and 768).
GATE_UP_MAX_TOKENS = 768
# The transposed GEMM's limits, for a K beyond GEMM_T_LONG_ROWS, where the library
# slows down (576 tokens, dequantize and product, us per million weights: 16384 x
# 5120 1.77, 17408 x 5120 2.49, 25600 x 5120 2.59), and for a shorter one.  Within
# them _gemm_t_serves.
GEMM_T_MAX_TOKENS = 768
GEMM_T_SHORT_TOKENS = 512
GEMM_T_LONG_ROWS = 16384
# What the kernels are built for, where the dequantised product has no such limit:
# columns of a row, and rows of a matrix dequantised to its transpose.
_MAX_COLS = 1 << 20
_MAX_DEQUANT_T_ROWS = 65535 * 128


def _gemm_serves(rows: int, out_f: int, in_f: int, cus: int) -> bool:
    """Whether the int4 GEMM beats dequantize + the library for 65 rows or more.
    Its workgroups are 128 weight rows x 64 tokens, the row blocks dealt to 8
    XCDs.  Up to 256 tokens it always does; beyond, where
      * at most one comes to a CU, if no XCD has more of them than CUs (us, GEMM /
        library: 5120 x 8192, 384 tokens, 240 workgroups, 51 / 65; 6400 x 5120, 320
        tokens, 250, 35 of them on an XCD, 63 / 50);
      * more come, and run in rounds of one to a CU, two at least (a CU with one
        waits on memory), if these are full enough: 92 % from K 6144 (5120 x 8192,
        448 tokens, 55 %, 87 / 72; 7424 x 8192, 512, 91 %, 96 / 90; 8704 x 8192, 448,
        93 %, 97 / 100), 72 % of three or more from K 4096 (8704 x 4096, 512, 71 %,
        65 / 59; 10240 x 5120, 448, 73 %, 79 / 78).  Two rounds of a shorter K win or
        lose by a tenth, as the library's steps fall (5632 x 5120, 448 tokens, 56 /
        60, 512 56 / 53), and short rows win (6144 x 2048, 384, 56 %, 26 / 31)."""
    if rows > GEMM_MAX_TOKENS:
        return False
    row_blocks, token_blocks = -(-out_f // 128), -(-rows // 64)
    workgroups = row_blocks * token_blocks
    if rows <= 256:
        return True
    if workgroups <= cus:
        return 8 * -(-row_blocks // 8) * token_blocks <= cus
    rounds = max(2, -(-workgroups // cus))
    full = 0.92 if in_f >= 6144 else 0.72 if in_f >= 4096 and rounds > 2 else 0.0
    return workgroups >= full * cus * rounds


def _gemm_t_serves(rows: int, in_f: int, out_f: int, splits: int, cus: int) -> bool:
    """Whether the transposed int4 GEMM, in `splits` parts of K, beats
    dequantize + the library for 65 rows or more.  Its workgroups (256 columns x
    64 tokens x a part) run in rounds of one to a CU, 11 ns per row of K each, so
    a round that is nearly empty costs a whole one; the parts' sums make another
    pass.  The library takes 1.0 us per million weights (1.2 where K is long) and
    2.3 more per thousand tokens.  (us, kernel / library: 6144 x 5120, 384 tokens,
    two parts in one round, 51 / 55, 448 tokens, one part, 78 / 63; 17408 x 5120,
    384 tokens 124 / 177, 768 tokens 208 / 242; 25600 x 5120, 512 tokens 226 / 345,
    768 tokens 290 / 371, 832 tokens, two rounds, 548 / 403; 12288 x 4096, 512
    tokens 87 / 98; 3072 x 1024, 192 tokens 22 / 16.  Over 28 shapes and 65 to 1024
    tokens the choice is 0.7 % from the faster on average, 28 points of 487 more
    than 4 %, the worst 2048 x 4096, 256 tokens, 28 / 19.)"""
    long = in_f > GEMM_T_LONG_ROWS
    if rows > (GEMM_T_MAX_TOKENS if long else GEMM_T_SHORT_TOKENS):
        return False
    rounds = -(-(-(-out_f // 256) * -(-rows // 64) * splits) // cus)
    kernel = 11e-3 * in_f * rounds / splits
    if splits > 1:
        kernel += 2.0 + 1.5e-6 * splits * rows * out_f
    return kernel < 2.0 + 1e-6 * in_f * out_f * ((1.2 if long else 1.0) + 2.3e-3 * rows)


@functools.lru_cache(maxsize=4096)
def _gemm_route(rows: int, out_f: int, in_f: int, device_index: int) -> bool:
    cus = torch.cuda.get_device_properties(device_index).multi_processor_count
    return in_f <= _MAX_COLS and _gemm_serves(rows, out_f, in_f, cus)


@functools.lru_cache(maxsize=4096)
def _gemm_t_route(rows: int, in_f: int, out_f: int, device_index: int) -> bool:
    import _dip_hip as K
    cus = torch.cuda.get_device_properties(device_index).multi_processor_count
    return (in_f % 8 == 0 and out_f <= _MAX_COLS
            and _gemm_t_serves(rows, in_f, out_f, K.int4_gemm_t_splits(rows, out_f, in_f), cus))


# (bound once: a small prompt's call is host time, 1.3 us of it these checks)
_dispatch_modes = torch._C._len_torch_dispatch_stack
_function_modes = torch._C._len_torch_function_stack
_any_autocast = torch._C._is_any_autocast_enabled
_functorch_wrapped = torch._C._functorch.is_functorch_wrapped_tensor
_forward_ad = torch.autograd.forward_ad
_is_tracing = torch._C._is_tracing
_is_compiling = torch.compiler.is_compiling
_is_grad_enabled = torch.is_grad_enabled


def _torch_watched() -> bool:
    """Whether the torch ops of a call would do more than compute: an active
    dispatch or function mode sees them (a default device, itself such a mode,
    does not count), or autocast gives their results another type than bf16."""
    if _dispatch_modes():
        return True
    if _function_modes():
        from torch.overrides import _get_current_function_mode_stack
        from torch.utils._device import DeviceContext
        if any(type(m) is not DeviceContext for m in _get_current_function_mode_stack()):
            return True
    return (_any_autocast() and torch.is_autocast_enabled("cuda")
            and torch.get_autocast_dtype("cuda") != torch.bfloat16)


def _plain_bf16(x: torch.Tensor) -> bool:
    """Whether x is a plain bf16 tensor on the device that nothing differentiates,
    batches, traces or watches: what a kernel called on its data may take in
    place of torch ops.  (Both refuse a weight on another device.)"""
    return (type(x) is torch.Tensor and x.dtype is torch.bfloat16 and x.is_cuda
            and not (x.requires_grad and _is_grad_enabled())
            and not _functorch_wrapped(x) and _forward_ad._current_level < 0
            and not _is_tracing() and not _is_compiling() and not _torch_watched())


def int4_linear(x: torch.Tensor, qweight: torch.Tensor, scales: torch.Tensor) -> torch.Tensor:
    """x @ (q*s)^T for x [..., in] on the device, in x's dtype: the int4
    GEMV for one token, the int4 MFMA GEMM for up to GEMM_MAX_TOKENS, else
    dequantize + F.linear (the reference's route, qlinear.py:86-88)."""
    import _dip_hip as K
    in_f = qweight.shape[1] * 2
    rows = x.numel() // in_f
    if rows == 1 and in_f in _GEMV_COLS:
        v = x.reshape(-1)
        y = K.int4_gemv(qweight, scales, v if v.dtype is torch.bfloat16 else v.to(torch.bfloat16))
        if y.dtype is not x.dtype:
            y = y.to(x.dtype)
        return y.view(*x.shape[:-1], qweight.shape[0])
    if rows > _ANY_INPUT_TOKENS:
        if (rows <= GEMM_MAX_TOKENS and x.shape[-1] == in_f and _plain_bf16(x)
                and _gemm_route(rows, qweight.shape[0], in_f, x.device.index)):
            return K.int4_gemm(qweight, scales, x)
    elif rows > 1:
        if x.dtype is torch.bfloat16 and x.shape[-1] == in_f:
            return K.int4_gemm(qweight, scales, x)
        y = K.int4_gemm(qweight, scales, x.reshape(rows, in_f).to(torch.bfloat16))
        return y.to(x.dtype).reshape(*x.shape[:-1], qweight.shape[0])
    return F.linear(x, dequantize(qweight, scales).to(x.dtype))


def int4_linear_t(x: torch.Tensor, qweight_t: torch.Tensor, scales_t: torch.Tensor) -> torch.Tensor:
    """x @ bf16(q*s) for a matrix stored as rows of the input dimension (the
    transposed down matrix) on the device, in x's dtype: the int4 MFMA GEMM
    for up to GEMM_T_MAX_TOKENS rows of x (GEMM_T_SHORT_TOKENS for a shorter K)
    where it is the faster, else x @ dequantize (the reference's route,
    dip_stream_predispatch.py:213-215), on the transpose where that can be."""
    import _dip_hip as K
    rows, in_f = x.numel() // x.shape[-1], qweight_t.shape[0]
    if rows <= _ANY_INPUT_TOKENS or (
            rows <= GEMM_T_MAX_TOKENS and _plain_bf16(x)
            and _gemm_t_route(rows, in_f, 2 * qweight_t.shape[1], x.device.index)):
        return K.int4_gemm_t(qweight_t, scales_t, x.to(torch.bfloat16)).to(x.dtype)
    if qweight_t.is_cuda and in_f % 8 == 0 and in_f <= _MAX_DEQUANT_T_ROWS:
        return F.linear(x, K.dequant_t(qweight_t, scales_t).to(x.dtype))
    return x @ dequantize(qweight_t, scales_t).to(x.dtype)


def swiglu(gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    """F.silu(gate) * up, in one launch for plain bf16 tensors on the device
    (the same roundings)."""
    if gate.is_cuda and gate.shape == up.shape and _plain_bf16(gate) and _plain_bf16(up):
        import _dip_hip as K
        return K.swiglu(gate, up)
    return F.silu(gate) * up


def int4_gate_up(x, gate_qw, gate_sc, up_qw, up_sc):
    """F.silu(x @ gate^T) * (x @ up^T), or None where that is not one launch: it
    is for plain bf16 prompts of up to GATE_UP_MAX_TOKENS."""
    import _dip_hip as K
    in_f = gate_qw.shape[1] * 2
    rows = x.numel() // in_f
    if not (1 < rows <= GATE_UP_MAX_TOKENS and x.shape[-1] == in_f and in_f <= _MAX_COLS
            and gate_qw.shape == up_qw.shape and _plain_bf16(x)):
        return None
    return K.int4_gemm_swiglu(gate_qw, gate_sc, up_qw, up_sc, x)


def _unpack_int4(qweight: torch.Tensor) -> torch.Tensor:
    """int8 [R, C/2] -> int8 [R, C] in [-8, 7] (qlinear.py:28-50)."""
    q = qweight.view(torch.uint8) if qweight.dtype == torch.int8 else qweight.to(torch.uint8)
    low = (q & 0x0F).to(torch.int8)
    high = ((q >> 4) & 0x0F).to(torch.int8)
    low = torch.where(low >= 8, low - 16, low)
    high = torch.where(high >= 8, high - 16, high)
    return torch.stack((low, high), dim=-1).reshape(q.shape[0], q.shape[1] * 2)


def dequantize(qweight: torch.Tensor, scales: torch.Tensor) -> torch.Tensor:
    """bf16 [R, C] = bf16(q * s) (qlinear.py:53-64)."""
    if qweight.is_cuda:
        from _dip_hip import dequant_rows
        return dequant_rows(qweight, scales, mode=1)
    q = _unpack_int4(qweight)
    out_f, in_f = q.shape
    qf = q.float().reshape(out_f, in_f // GROUP_SIZE, GROUP_SIZE)
    s = scales.float().reshape(out_f, in_f // GROUP_SIZE, 1)
    return (qf * s).reshape(out_f, in_f).to(torch.bfloat16)


class QuantLinear(nn.Module):
    """INT4 g128 symmetric linear; dequantizes then calls F.linear
    (qlinear.py:67-88)."""

    def __init__(self, in_features: int, out_features: int, bias: bool = False):
        super().__init__()
        self.in_features = in_features
        self.out_features = out_features
        assert in_features % GROUP_SIZE == 0
        self.register_buffer("qweight",
                             torch.empty(out_features, in_features // 2, dtype=torch.int8))
        self.register_buffer("scales",
                             torch.empty(out_features, in_features // GROUP_SIZE,
                                         dtype=torch.bfloat16))
        self.bias = None

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        if x.is_cuda and self.out_features > 0:
            return int4_linear(x, self.qweight, self.scales)
        w = dequantize(self.qweight, self.scales)
        return F.linear(x, w.to(x.dtype))


def _replace_linears_with_quant(model: nn.Module) -> list:
    """Swap every nn.Linear whose qualified name contains one of the seven
    projection names for an empty QuantLinear of the same shape
    (qlinear.py:91-106); returns the swapped names.  lm_head and the
    embeddings stay as they are."""
    swapped = []
    for parent_name, parent in list(model.named_modules()):
        for child_name, child in list(parent.named_children()):
            full = f"{parent_name}.{child_name}" if parent_name else child_name
            if isinstance(child, nn.Linear) and any(s in full for s in _QUANT_SUBSTRINGS):
                setattr(parent, child_name, QuantLinear(child.in_features, child.out_features))
                swapped.append(full)
    return swapped


def load_quantized_qwen3(ckpt_dir, gpu_mem_gib: int = 13, cpu_mem_gib: int = 60,
                         device="cuda:0"):
    """The reference's int4 baseline (qlinear.py:109-166): the model of
    `ckpt_dir/config.json` with QuantLinear projections and the weights of
    model_int4.safetensors.  Returns (model, tokenizer or None).

    The reference splits the model between a small GPU and host memory with
    accelerate's offload hooks (gpu_mem_gib / cpu_mem_gib); one MI355X holds
    a whole int4 Qwen3-32B in HBM, so every tensor is placed on `device` and
    the two sizes are accepted for call compatibility only."""
    from dip_model import build_empty_model, load_tensors, load_tokenizer
    from dip_checkpoint import ST_NAME, read_quant_config
    ckpt_dir = Path(ckpt_dir)
    read_quant_config(ckpt_dir)
    model = build_empty_model(ckpt_dir)
    load_tensors(model, ckpt_dir / ST_NAME, device)
    return model, load_tokenizer(ckpt_dir)
