"""Python entry points of the hand-written gfx950 kernels.

Every function checks shapes, types and devices on the host, then launches on
torch's current HIP stream through the C entry points of `cwm_amd/csrc`.  There is
no CPU path and no library substitute: tensors that are not on a HIP device, or a
missing kernel library, raise an error.

The only library routine on the model's path is the bfloat16 matrix product of many
rows where its tiles fill the chip (`torch.mm`, i.e. hipBLASLt), where
the reference also calls a library
(cwm/fastgen/forward.py:593-606).
"""

from __future__ import annotations

import ctypes
from dataclasses import dataclass
from typing import Optional, Tuple

import numpy as np
import torch

from . import build as _build
from . import attention_plan as _work_lists
from .attention_plan import WIDE_TILES
from .build import KernelBuildError

F32, BF16 = 0, 1


class KernelError(RuntimeError):
    """A kernel entry point refused its arguments."""


def _code(dtype: torch.dtype) -> int:
    if dtype == torch.float32:
        return F32
    if dtype == torch.bfloat16:
        return BF16
    raise KernelError(f"kernels take float32 and bfloat16 tensors, not {dtype}")


def _need_gpu(*tensors: Optional[torch.Tensor]) -> None:
    for t in tensors:
        if t is not None and not t.is_cuda:
            raise KernelError(
                "cwm_amd kernels run on a HIP device only; got a tensor on "
                f"{t.device}. There is no CPU path."
            )


def _ptr(t: Optional[torch.Tensor]) -> ctypes.c_void_p:
    return ctypes.c_void_p(0 if t is None else t.data_ptr())


def _stream() -> ctypes.c_void_p:
    """The current HIP stream of the current device (the raw handle; building a torch
    Stream object for every launch costs several microseconds)."""
    return ctypes.c_void_p(torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice()))


def _check(lib: ctypes.CDLL, status: int) -> None:
    if status != 0:
        raise KernelError(lib.cwm_error_message().decode("utf-8", "replace"))


def _rows_contiguous(t: torch.Tensor, what: str) -> None:
    if t.dim() < 1 or t.stride(-1) != 1:
        raise KernelError(f"{what}: innermost dimension must be contiguous, strides are {t.stride()}")


def _i32(t: torch.Tensor, what: str) -> None:
    if t.dtype != torch.int32 or not t.is_contiguous():
        raise KernelError(f"{what} must be a contiguous int32 tensor, found {t.dtype} with strides {t.stride()}")


# --------------------------------------------------------------------------- #
def embedding(tokens: torch.Tensor, table: torch.Tensor, scale: float = 1.0) -> torch.Tensor:
    """float32 [T, D]: `scale` times the rows of `table` ([V, D], float32 or bfloat16) for int32 `tokens` [T]."""
    _need_gpu(tokens, table)
    _i32(tokens, "tokens")
    if table.dim() != 2 or not table.is_contiguous():
        raise KernelError("embedding table must be a contiguous [V, D] tensor")
    lib = _build.load("rowwise")
    out = torch.empty((tokens.numel(), table.shape[1]), dtype=torch.float32, device=table.device)
    _check(
        lib,
        lib.cwm_embedding(
            _ptr(out), _ptr(table), _code(table.dtype), _ptr(tokens),
            ctypes.c_int(tokens.numel()), ctypes.c_int(table.shape[1]), ctypes.c_int(table.shape[0]), ctypes.c_float(scale), _stream(),
        ),
    )
    return out


def add_rmsnorm(
    h: torch.Tensor,
    delta: Optional[torch.Tensor],
    weight: torch.Tensor,
    eps: float,
    out_dtype: torch.dtype,
    rows: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """`h` (float32 [T, D]) += `delta` in place, then RMSNorm(h) * weight.

    `delta` is [T, D], or float32 partial sums [P, T, D] (a matrix product whose K
    was split) that are added in order.  With `rows` (int32 [R]) only those rows are
    normalised and `h` is not changed (the sum with `delta` is still what is
    normalised).
    """
    _need_gpu(h, delta, weight, rows)
    if h.dtype != torch.float32 or h.dim() != 2 or not h.is_contiguous():
        raise KernelError("the residual stream must be a contiguous float32 [T, D] tensor")
    n_tokens, dim = h.shape
    n_partials = 1
    if delta is not None:
        if delta.dim() == 3:
            if delta.dtype != torch.float32:
                raise KernelError("partial sums must be float32")
            n_partials = delta.shape[0]
        if tuple(delta.shape[-2:]) != tuple(h.shape) or not delta.is_contiguous():
            raise KernelError(f"delta {tuple(delta.shape)} does not match the residual stream {tuple(h.shape)}")
    if weight.shape != (dim,) or not weight.is_contiguous():
        raise KernelError(f"norm weight has shape {tuple(weight.shape)}, expected ({dim},)")
    if rows is not None:
        _i32(rows, "rows")
    n_out = n_tokens if rows is None else rows.numel()
    out = torch.empty((n_out, dim), dtype=out_dtype, device=h.device)
    lib = _build.load("rowwise")
    _check(
        lib,
        lib.cwm_add_rmsnorm(
            _ptr(h), _ptr(delta), ctypes.c_int(_code(delta.dtype) if delta is not None else F32),
            ctypes.c_int(n_partials), ctypes.c_long(n_tokens * dim), _ptr(weight), ctypes.c_int(_code(weight.dtype)), _ptr(out), ctypes.c_int(_code(out_dtype)),
            _ptr(rows), ctypes.c_int(n_out), ctypes.c_int(dim), ctypes.c_float(eps), _stream(),
        ),
    )
    return out


def silu_mul(gate_up: torch.Tensor, out_dtype: Optional[torch.dtype] = None, grouped: bool = False) -> torch.Tensor:
    """[T, 2F] -> [T, F]: silu(gate) * up, computed in float32; gate is the first half
    of a row and up the second, or, with `grouped`, they alternate in groups of 8
    columns (the order in which a product with row-interleaved gate/up weights
    delivers them).  Float32 partial sums [P, T, 2F] of a product with a split K are
    taken too: they are added in order, rounded to `out_dtype` as the product would
    have stored them, and then treated alike."""
    _need_gpu(gate_up)
    if grouped and (gate_up.shape[-1] // 2) % 8 != 0:
        raise KernelError("gate and up in groups of 8 need a width that is a multiple of 8")
    lib = _build.load("rowwise")
    if gate_up.dim() == 3:
        if gate_up.dtype != torch.float32 or gate_up.shape[2] % 2 != 0 or not gate_up.is_contiguous():
            raise KernelError("partial sums for silu_mul must be a contiguous float32 [P, T, 2F] tensor")
        n_part, n_tokens, two_f = gate_up.shape
        if (two_f // 2) % 4 != 0:
            return silu_mul(sum_partials(gate_up, out_dtype or torch.float32), grouped=grouped)
        out = torch.empty((n_tokens, two_f // 2), dtype=out_dtype or torch.float32, device=gate_up.device)
        _check(
            lib,
            lib.cwm_silu_mul_partials(
                _ptr(out), ctypes.c_int(_code(out.dtype)), _ptr(gate_up), ctypes.c_int(n_part),
                ctypes.c_int(n_tokens), ctypes.c_int(two_f // 2), ctypes.c_int(int(grouped)), _stream(),
            ),
        )
        return out
    if gate_up.dim() != 2 or gate_up.shape[1] % 2 != 0 or not gate_up.is_contiguous():
        raise KernelError("silu_mul takes a contiguous [T, 2F] tensor")
    n_tokens, two_f = gate_up.shape
    out = torch.empty((n_tokens, two_f // 2), dtype=gate_up.dtype, device=gate_up.device)
    _check(
        lib,
        lib.cwm_silu_mul(
            _ptr(out), _ptr(gate_up), ctypes.c_int(_code(gate_up.dtype)),
            ctypes.c_int(n_tokens), ctypes.c_int(two_f // 2), ctypes.c_int(int(grouped)), _stream(),
        ),
    )
    return out


def gate_up_silu(
    x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor], grouped: bool, streamed: Optional[torch.Tensor] = None
) -> torch.Tensor:
    """silu(x Wg^T) * (x Wu^T) for the joined weight [2F, D] of a gated feed-forward
    (cwm/fastgen/forward.py:776-781): rows Wg then Wu, or, with `grouped`, alternating
    in groups of 8.  A grouped weight lets a decode batch in bfloat16 finish the
    activation in the product's epilogue; every other case runs the product and the
    activation kernel, with the same roundings."""
    n = weight.shape[0]
    fused = (
        grouped and n % 16 == 0
        and x.is_cuda and x.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16
        and x.shape[0] <= STREAM_EPILOGUE_ROWS and _stream_takes(x, weight)
        and x.shape[1] <= stream_unsplit_k(x.shape[0])  # K fits one group of wavefronts: no split
    )
    tiled = x.is_cuda and x.dim() == 2 and _prefers_tile(x, weight, bias, streamed, fused)
    if fused and not tiled:
        return gemm_bf16_stream(x, weight, bias, torch.bfloat16, glu=True, streamed=streamed)
    if tiled and grouped and x.shape[0] <= TILE_ROWS:
        return gemm_bf16_tile(x, weight, None, torch.bfloat16, glu=True)
    if grouped and not tiled and bias is None and x.is_cuda and x.dim() == 2 and x.shape[0] > STREAM_MAX_ROWS and _prefers_wide(x, weight, glu=True):
        return gemm_bf16_wide(x, weight, glu=True)
    return silu_mul(linear(x, weight, bias, partials_ok=True, streamed=streamed), out_dtype=x.dtype, grouped=grouped)


# --------------------------------------------------------------------------- #
def gemm_f32(
    x: torch.Tensor,
    weight: torch.Tensor,
    bias: Optional[torch.Tensor] = None,
    out_dtype: Optional[torch.dtype] = None,
) -> torch.Tensor:
    """x [M, K] @ weight[N, K]^T (+ bias) in float32: float32 sums of products that are exact, or (float32
    operands, K a multiple of 32) exact to 2^-24 of themselves, on the matrix cores; see csrc/gemm_f32.hip."""
    _need_gpu(x, weight, bias)
    if x.dim() != 2 or weight.dim() != 2 or x.shape[1] != weight.shape[1]:
        raise KernelError(f"gemm: x {tuple(x.shape)} and weight {tuple(weight.shape)} do not fit")
    if _f32_parts_takes(x, weight):  # whatever the number of rows: a row's result does not depend on the others
        return _f32_parts(x, weight, bias, out_dtype, -2 if _f32_parts_alone(x.shape[0], weight.shape[0], x.shape[1]) else -1)
    _rows_contiguous(x, "gemm x")
    _rows_contiguous(weight, "gemm weight")
    m, k = x.shape
    n = weight.shape[0]
    if bias is not None and (bias.shape != (n,) or not bias.is_contiguous()):
        raise KernelError(f"gemm: bias {tuple(bias.shape)} does not fit {n} outputs")
    out_dtype = out_dtype or x.dtype
    out = torch.empty((m, n), dtype=out_dtype, device=x.device)
    lib = _build.load("gemm_f32")
    _check(
        lib,
        lib.cwm_gemm_f32(
            _ptr(x), ctypes.c_int(_code(x.dtype)), ctypes.c_long(x.stride(0) if m > 1 else k),
            _ptr(weight), ctypes.c_int(_code(weight.dtype)), ctypes.c_long(weight.stride(0) if n > 1 else k),
            _ptr(out), ctypes.c_int(_code(out_dtype)), ctypes.c_long(n),
            _ptr(bias), ctypes.c_int(_code(bias.dtype) if bias is not None else F32),
            ctypes.c_int(m), ctypes.c_int(n), ctypes.c_int(k), _stream(),
        ),
    )
    return out


F32_PARTS_STRIDE = 1 << 23  # csrc/gemm_f32.hip: a block's byte offsets from its first row of W fit 32 bits; rows further apart are copied


def gemm_f32_parts(
    x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor] = None, out_dtype: Optional[torch.dtype] = None, block: Optional[int] = None,
) -> torch.Tensor:
    """The product of `gemm_f32` where both operands are float32, K is a multiple of 32 up to 65,536 and rows are 16-byte aligned:
    every value in three exact bfloat16 parts, six of their nine products on the matrix cores.  x's parts are made by a kernel of
    their own, into scratch memory of 6 bytes a value.  `block` (tests): the number of a block of the kernel's list, or -2 for one
    launch without scratch memory (K up to 256)."""
    _need_gpu(x, weight, bias)
    if x.dim() != 2 or weight.dim() != 2 or x.shape[1] != weight.shape[1] or not _f32_parts_takes(x, weight):
        raise KernelError(
            "the float32 product in parts takes float32 x [M, K] and weight [N, K] with K a multiple of 32 and 16-byte aligned rows; "
            f"got {tuple(x.shape)} {x.dtype} and {tuple(weight.shape)} {weight.dtype}"
        )
    return _f32_parts(x, weight, bias, out_dtype, -1 if block is None else block)


def _f32_parts(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor], out_dtype: Optional[torch.dtype], block: int) -> torch.Tensor:
    m, k = x.shape
    n = weight.shape[0]
    if bias is not None and (bias.shape != (n,) or not bias.is_contiguous()):
        raise KernelError(f"gemm: bias {tuple(bias.shape)} does not fit {n} outputs")
    if n > 1 and weight.stride(0) >= F32_PARTS_STRIDE:
        weight = weight.contiguous()
    lib = _build.load("gemm_f32")
    out = torch.empty((m, n), dtype=out_dtype or x.dtype, device=x.device)
    scratch = None if block == -2 else torch.empty(-(-m // 16) * (k // 32 * 3072 + -(-k // 256) * 4), dtype=torch.uint8, device=x.device)
    _check(
        lib,
        lib.cwm_gemm_f32_parts(
            _ptr(x), ctypes.c_long(x.stride(0) if m > 1 else k), _ptr(weight), ctypes.c_long(weight.stride(0) if n > 1 else k), _ptr(out),
            ctypes.c_int(_code(out.dtype)), ctypes.c_long(n), _ptr(bias), ctypes.c_int(_code(bias.dtype) if bias is not None else F32),
            ctypes.c_int(m), ctypes.c_int(n), ctypes.c_int(k), _ptr(scratch), ctypes.c_int(block), _stream(),
        ),
    )
    return out


F32_ALONE_K = 256  # csrc/gemm_f32.hip: ALONE_STEPS
# Blocks of 32 rows and 64 columns up to which it pays that each makes its rows' parts again; of a K above half of that, whose blocks do not
# share a compute unit, a quarter.  Two launches / one, us: K = 64, 1,024 blocks 11.0 / 10.2, 2,048 17.6 / 17.7; K = 128, 512 blocks 11.3 / 8.0, 1,024
# 12.2 to 15.5 / 13.1 to 13.5, 2,048 23.1 / 22.9; K = 256, 256 blocks 13.0 / 9.1, 384 12.6 / 14.7, 512 15.7 / 16.1, 1,024 16.4 / 28.2.
F32_ALONE_BLOCKS = 1024


def _f32_parts_alone(m: int, n: int, k: int) -> bool:
    """Whether a product in parts is one launch, whose blocks make the parts of their rows of x themselves."""
    return k <= F32_ALONE_K and -(-m // 32) * -(-n // 64) <= (F32_ALONE_BLOCKS if 2 * k <= F32_ALONE_K else F32_ALONE_BLOCKS // 4)


def _f32_parts_takes(x: torch.Tensor, weight: torch.Tensor) -> bool:
    if x.dtype != torch.float32 or weight.dtype != torch.float32:
        return False
    (m, k), (x_row, x_one), (w_row, w_one) = x.shape, x.stride(), weight.stride()
    return (
        m > 0 and k % 32 == 0 and 0 < k <= 65536 and x_one == 1 and w_one == 1
        and (m <= 1 or x_row % 4 == 0) and (weight.shape[0] <= 1 or w_row % 4 == 0) and x.data_ptr() % 16 == 0 and weight.data_ptr() % 16 == 0
    )


F32_STREAM_MAX_ROWS = 16
_f32_stream_block_steps: Optional[int] = None


def _f32_stream_takes(x: torch.Tensor, weight: torch.Tensor) -> bool:
    return (
        x.dtype == torch.float32 and weight.dtype == torch.float32
        and x.dim() == 2 and weight.dim() == 2 and x.shape[0] <= F32_STREAM_MAX_ROWS
        and x.shape[1] % 4 == 0 and x.stride(-1) == 1 and weight.stride(-1) == 1
        and (x.shape[0] <= 1 or x.stride(0) % 4 == 0) and (weight.shape[0] <= 1 or weight.stride(0) % 4 == 0)
        and x.data_ptr() % 16 == 0 and weight.data_ptr() % 16 == 0
    )


def gemm_f32_stream(
    x: torch.Tensor,
    weight: torch.Tensor,
    bias: Optional[torch.Tensor] = None,
    out_dtype: Optional[torch.dtype] = None,
    partials_ok: bool = False,
) -> torch.Tensor:
    """float32 x [M <= 16, K] @ float32 weight[N, K]^T with float32 multiply-add, the weight
    streamed once by persistent blocks (the decode-step product of the 32-bit path).  Returns
    [M, N]; with `partials_ok` it may return float32 partial sums [P, M, N] of a split K."""
    global _f32_stream_block_steps
    _need_gpu(x, weight, bias)
    if not _f32_stream_takes(x, weight) or x.shape[1] != weight.shape[1]:
        raise KernelError(
            f"the float32 streaming product takes float32 x [M <= {F32_STREAM_MAX_ROWS}, K] and weight [N, K] with K a multiple "
            f"of 4 and 16-byte aligned rows; got {tuple(x.shape)} {x.dtype} and {tuple(weight.shape)} {weight.dtype}"
        )
    m, k = x.shape
    n = weight.shape[0]
    if bias is not None and (bias.shape != (n,) or not bias.is_contiguous()):
        raise KernelError(f"gemm: bias {tuple(bias.shape)} does not fit {n} outputs")
    out_dtype = out_dtype or torch.float32
    lib = _build.load("gemm_f32_stream")
    if _f32_stream_block_steps is None:
        _f32_stream_block_steps = int(lib.cwm_gemm_f32_stream_steps_per_block())
    steps = (k + 15) // 16
    n_tiles = (n + 15) // 16
    cus = _compute_units(x.device)
    k_split = -(-steps // _f32_stream_block_steps)  # K longer than one block's registers is split
    if partials_ok:
        while n_tiles * k_split < 2 * cus and k_split < 8 and steps >= 2 * k_split * 16:
            k_split *= 2  # too few tiles to fill the chip
    blocks = max(k_split, min(cus, n_tiles * k_split) // k_split * k_split)
    if k_split == 1:
        out = torch.empty((m, n), dtype=out_dtype, device=x.device)
    else:
        out = torch.empty((k_split, m, n), dtype=torch.float32, device=x.device)
    _check(
        lib,
        lib.cwm_gemm_f32_stream(
            _ptr(x), ctypes.c_long(x.stride(0) if m > 1 else k), _ptr(weight), ctypes.c_long(weight.stride(0) if n > 1 else k),
            _ptr(out), ctypes.c_int(_code(out.dtype)), ctypes.c_long(n), ctypes.c_long(m * n),
            _ptr(bias), ctypes.c_int(_code(bias.dtype) if bias is not None else F32),
            ctypes.c_int(m), ctypes.c_int(n), ctypes.c_int(k), ctypes.c_int(k_split), ctypes.c_int(blocks), _stream(),
        ),
    )
    if k_split > 1 and not partials_ok:
        return sum_partials(out, out_dtype)
    return out


def linear(
    x: torch.Tensor,
    weight: torch.Tensor,
    bias: Optional[torch.Tensor] = None,
    out_dtype: Optional[torch.dtype] = None,
    partials_ok: bool = False,
    streamed: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """y = x W^T (+ b).  cwm/fastgen/forward.py:593-606.

    float32 activations or float32 weights: the float32 kernels (`gemm_f32`; up to 16
    rows of float32 on the weight-streaming one, whose sums differ from the other's by rounding).
    bfloat16 activations and weights: matrix cores with float32 accumulation, the
    library product for many rows.  With `partials_ok` the result may be float32
    partial sums [P, M, N] that the caller adds (see `add_rmsnorm`).  `streamed`: the weight's
    streaming copy (`stream_layout`), which the products of few rows read instead where there is one.
    """
    out_dtype = out_dtype or x.dtype
    if x.dtype == torch.float32 or weight.dtype == torch.float32:
        if x.is_cuda and _f32_stream_takes(x, weight):
            return gemm_f32_stream(x, weight, bias, out_dtype, partials_ok)
        return gemm_f32(x, weight, bias, out_dtype)
    return gemm_bf16(x, weight, bias, out_dtype, partials_ok, streamed)


STREAM_MAX_ROWS = 64
_cu_count: dict = {}


_stream_shapes: dict = {}  # rows -> (wavefronts of a block, steps of K a wavefront holds)


def _compute_units(device: torch.device) -> int:
    idx = device.index if device.index is not None else torch.cuda.current_device()
    if idx not in _cu_count:
        _cu_count[idx] = torch.cuda.get_device_properties(idx).multi_processor_count
    return _cu_count[idx]


def _stream_block_shape(m: int) -> Tuple[int, int]:
    """(wavefronts of a block, steps of 32 along K that one wavefront keeps of x in registers) of the streaming
    product for `m` rows, asked of the library: the kernel's register budget is stated there and nowhere else."""
    shape = _stream_shapes.get(m)
    if shape is None:
        lib = _build.load("gemm_bf16_stream")
        shape = _stream_shapes[m] = (lib.cwm_gemm_bf16_stream_waves(ctypes.c_int(m)), lib.cwm_gemm_bf16_stream_steps_per_wave(ctypes.c_int(m)))
    return shape


def stream_unsplit_k(m: int, fused: bool = True) -> int:
    """The longest K that one group of wavefronts of the streaming product holds for `m` rows, so that K is not
    split over blocks: the fused epilogues (rotation + cache write, gated activation) need that.  Products without an
    epilogue are split from 17 rows on as for 64, so that a row's bits are the same."""
    waves, regs = _stream_block_shape(m if m <= 16 or fused else STREAM_MAX_ROWS)
    return 32 * waves * regs


def stream_layout(weight: torch.Tensor) -> torch.Tensor:
    """The streaming copy of a bfloat16 matrix W [N, K]: [tiles of 16 rows, steps of 32 columns, 64, 8], lane
    16 j + r of a step holding W[16 tile + r][32 step + 8 j ..+8] (one operand of the matrix instruction), zeros
    past N and K.  The streaming product reads it 1 KB a wavefront's load, every cache line once."""
    _need_gpu(weight)
    if weight.dtype != torch.bfloat16 or weight.dim() != 2 or weight.stride(1) != 1:
        raise KernelError("a streaming copy is made of a bfloat16 matrix with contiguous rows")
    n, k = weight.shape
    out = torch.empty((-(-n // 16), -(-k // 32), 64, 8), dtype=torch.bfloat16, device=weight.device)
    lib = _build.load("gemm_bf16_stream")
    _check(lib, lib.cwm_gemm_bf16_stream_copy(_ptr(weight), ctypes.c_long(weight.stride(0)), _ptr(out), ctypes.c_int(n), ctypes.c_int(k), _stream()))
    return out


def gemm_bf16_stream(
    x: torch.Tensor,
    weight: torch.Tensor,
    bias: Optional[torch.Tensor] = None,
    out_dtype: Optional[torch.dtype] = None,
    partials_ok: bool = False,
    rope: Optional[tuple] = None,
    glu: bool = False,
    streamed: Optional[torch.Tensor] = None,
    rows_per_input: Optional[int] = None,
    keep_sums: bool = False,
) -> torch.Tensor:
    """bfloat16 x [M <= 64, K] @ weight[N, K]^T with persistent blocks that keep x in
    registers and stream the weight once.  `streamed` is the matrix's streaming copy
    (`stream_layout(weight)`); with it the kernel reads that copy, in whole cache lines and past the
    caches, instead of `weight`.  Returns [M, N]; with `partials_ok` it may
    return float32 partial sums [P, M, N] of a split K for the caller to add (the
    residual-add + RMSNorm kernel takes them); with `keep_sums` it then does so (P = 1) for a K that is not
    split too, instead of a result of a shorter type, so that nothing is rounded between the product and what follows
    (for products that the tiled kernel, which leaves such sums, takes as well).  `rope`
    (positions, seq_of_token, inv_freq, cache, block_table, n_q_heads, n_kv_heads,
    head_dim) makes the epilogue rotate the q and k columns and write k and v into the
    paged cache (see `qkv_rope_write`).  `glu`: the weight's rows are gate and up rows in
    alternating groups of 8 and the result is silu(gate) * up, [M, N / 2] (see
    `gate_up_silu`).  `rows_per_input` (a multiple of 16): x is [G, M, K], and the weight's rows belong to its G inputs in
    turn, that many each (the last one's may be fewer): column n of the result is row n of the weight times input
    n // rows_per_input."""
    _need_gpu(x, weight, bias)
    inputs = 1
    if rows_per_input is not None:
        inputs = x.shape[0]
        if (
            x.dim() != 3 or rows_per_input < 16 or rows_per_input % 16 != 0 or rope is not None or glu or x.stride(0) % 8 != 0
            or not (inputs - 1) * rows_per_input < weight.shape[0] <= inputs * rows_per_input
        ):
            raise KernelError(f"{weight.shape[0]} rows of a weight do not belong to {inputs} inputs in runs of {rows_per_input} (a multiple of 16)")
        input_stride, x = x.stride(0), x[0]
    if x.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16:
        raise KernelError("the streaming product takes bfloat16 operands")
    if x.dim() != 2 or weight.dim() != 2 or x.shape[1] != weight.shape[1]:
        raise KernelError(f"gemm: x {tuple(x.shape)} and weight {tuple(weight.shape)} do not fit")
    m, k = x.shape[0], weight.shape[1]
    n = weight.shape[0]
    if m > STREAM_MAX_ROWS:
        raise KernelError(f"the streaming product takes at most {STREAM_MAX_ROWS} rows, not {m}")
    if bias is not None and (bias.shape != (n,) or not bias.is_contiguous()):
        raise KernelError(f"gemm: bias {tuple(bias.shape)} does not fit {n} outputs")
    out_dtype = out_dtype or torch.bfloat16
    lib = _build.load("gemm_bf16_stream")
    waves = _stream_block_shape(m)[0]
    steps = (k + 31) // 32
    n_tiles = (n + 15) // 16
    cus = _compute_units(x.device)
    k_split = -(-steps * 32 // stream_unsplit_k(m, rope is not None or glu))  # K longer than one group of wavefronts' registers is split
    if (rope is not None or glu) and (k_split != 1 or m > STREAM_EPILOGUE_ROWS):
        raise KernelError("the fused epilogues need at most 32 rows and a K that one group of wavefronts holds")
    if glu:
        partials_ok = False
    if partials_ok:
        while n_tiles * k_split < 2 * cus and k_split < 8 and steps >= 2 * k_split * waves:
            k_split *= 2  # too few tiles to fill the chip
    blocks = max(k_split, min(cus, n_tiles * k_split) // k_split * k_split)
    input_args = (ctypes.c_long(0), ctypes.c_int(0), ctypes.c_int(0))
    if inputs > 1:
        per, most = rows_per_input // 16, max(1, cus // k_split)
        tiles_a_block = -(-n_tiles // most)
        while True:  # as few tiles a block as leave one round of blocks
            a_input, rest = -(-per // tiles_a_block), -(-(n_tiles - (inputs - 1) * per) // tiles_a_block)
            if (inputs - 1) * a_input + rest <= most or tiles_a_block >= per:
                break
            tiles_a_block += 1
        blocks = k_split * ((inputs - 1) * a_input + rest)
        input_args = (ctypes.c_long(input_stride), ctypes.c_int(per), ctypes.c_int(a_input))
    if k_split == 1 and partials_ok and keep_sums and out_dtype != torch.float32 and _tile_wins(x, weight):
        out = torch.empty((1, m, n), dtype=torch.float32, device=x.device)  # the consumer adds float32 sums, here one
    elif k_split == 1:
        out = torch.empty((m, n // 2 if glu else n), dtype=out_dtype, device=x.device)
    else:
        out = torch.empty((k_split, m, n), dtype=torch.float32, device=x.device)
    if streamed is not None:
        if streamed.shape != (n_tiles, steps, 64, 8) or streamed.dtype != torch.bfloat16 or not streamed.is_contiguous() or streamed.device != x.device:
            raise KernelError(f"the streaming copy of a [{n}, {k}] matrix is bfloat16 [{n_tiles}, {steps}, 64, 8], not {tuple(streamed.shape)}")
        w_ptr, w_stride = _ptr(streamed), ctypes.c_long(steps * 512)
    else:
        w_ptr, w_stride = _ptr(weight), ctypes.c_long(weight.stride(0) if n > 1 else k)
    _check(
        lib,
        lib.cwm_gemm_bf16_stream(
            _ptr(x), ctypes.c_long(x.stride(0) if m > 1 else x.shape[1]), w_ptr, w_stride,
            _ptr(out), ctypes.c_int(_code(out.dtype)), ctypes.c_long(out.shape[-1]), ctypes.c_long(m * n),
            _ptr(bias), ctypes.c_int(_code(bias.dtype) if bias is not None else F32),
            ctypes.c_int(m), ctypes.c_int(n), ctypes.c_int(k), ctypes.c_int(k_split), ctypes.c_int(blocks),
            *_rope_args(rope), ctypes.c_int(int(glu)), ctypes.c_int(int(streamed is not None)), *input_args, _stream(),
        ),
    )
    if k_split > 1 and not partials_ok:
        return sum_partials(out, out_dtype)
    return out


def linear_inputs_takes(x: torch.Tensor, weight: torch.Tensor, rows_per_input: int) -> bool:
    """Whether the product of a few rows of several inputs is one launch (`linear_inputs`): as many as the streaming product takes.  Linear
    attention's layer of four products and their low rank of 64 on five inputs, apart (five launches, and four more up to the gated result) and so
    (two), replayed, us by rows 17, 32, 33 and 64: width 512 42 and 19, 46 and 20, 74 and 25, 81 and 27; 2,048 65 and 34, 78 and 43, 108 and 49, 128 and
    68; 3,072 81 and 44, 110 and 58, 125 and 67, 159 and 94; 5,120 122 and 78, 149 and 96, 166 and 111, 231 and 156; 8,192 196 and 149, 233 and 188, 245
    and 203, 322 and 276.  Without the weights' streaming copies no size of these is slower either (8,192, 24 rows 211 and 201)."""
    return (
        x.is_cuda and x.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16 and x.dim() == 3 and x.shape[1] <= STREAM_MAX_ROWS
        and rows_per_input % 16 == 0 and x.is_contiguous() and x.shape[1] * x.shape[2] % 8 == 0 and _stream_takes(x[0], weight)
    )


def linear_inputs(x: torch.Tensor, weight: torch.Tensor, rows_per_input: int, streamed: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Several inputs x [G, M <= 64, K] times the rows of one joined weight that belong to each (`rows_per_input` rows an
    input, the last one's may be fewer), side by side: float32 partial sums [P, M, N] for the caller to add."""
    out = gemm_bf16_stream(x, weight, None, torch.float32, partials_ok=True, streamed=streamed, rows_per_input=rows_per_input)
    return out if out.dim() == 3 else out.unsqueeze(0)


_NO_ROPE_ARGS = [ctypes.c_void_p(0)] * 5 + [ctypes.c_int(0)] * 6


def _rope_args(rope: Optional[tuple]) -> list:
    if rope is None:
        return _NO_ROPE_ARGS
    positions, seq_of_token, inv_freq, cache, block_table, n_q, n_kv, hd = rope
    return [
        _ptr(positions), _ptr(seq_of_token), _ptr(inv_freq), _ptr(cache), _ptr(block_table),
        ctypes.c_int(block_table.shape[1]), ctypes.c_int(cache.shape[3] // hd), ctypes.c_int(cache.shape[0]),
        ctypes.c_int(n_q), ctypes.c_int(n_kv), ctypes.c_int(hd),
    ]


def qkv_rope_write(
    x: torch.Tensor,
    weight: torch.Tensor,
    bias: Optional[torch.Tensor],
    n_q_heads: int,
    n_kv_heads: int,
    head_dim: int,
    positions: torch.Tensor,
    inv_freq: Optional[torch.Tensor],
    cache: torch.Tensor,
    block_table: torch.Tensor,
    seq_of_token: torch.Tensor,
    streamed: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """The joined q/k/v projection of x [T, D] (weight [(Hq + 2 Hkv) * hd, D]), the
    rotation of its q and k columns by each token's position, and the write of the
    rotated keys and of the values into the paged cache
    (cwm/fastgen/forward.py:593-632).  Returns [T, (Hq + 2 Hkv) * hd] with q rotated.
    Decode batches in bfloat16 do all three in the streaming product's epilogue; any
    other case runs the product and then the rotation + cache-write kernel, with the
    same arithmetic."""
    n_out = (n_q_heads + 2 * n_kv_heads) * head_dim
    if weight.shape[0] != n_out:
        raise KernelError(f"q/k/v weight has {weight.shape[0]} rows, expected {n_out}")
    fused = (
        x.is_cuda
        and x.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16 and cache.dtype == torch.bfloat16
        and x.shape[0] <= STREAM_EPILOGUE_ROWS
        and head_dim <= 256
        and _stream_takes(x, weight)
        and x.shape[1] <= stream_unsplit_k(x.shape[0])  # K fits one group of wavefronts: no split
        and not _prefers_tile(x, weight, bias, streamed, True)
    )
    if fused:
        _i32(positions, "positions")
        _i32(seq_of_token, "seq_of_token")
        _i32(block_table, "block_table")
        if inv_freq is not None and (inv_freq.dtype != torch.float32 or inv_freq.numel() != head_dim // 2 or not inv_freq.is_contiguous()):
            raise KernelError(f"the rotary table must be float32 [{head_dim // 2}]")
        if cache.dim() != 4 or cache.shape[1] != 2 or cache.shape[2] != n_kv_heads or cache.shape[3] % head_dim != 0 or not cache.is_contiguous():
            raise KernelError(f"cache {tuple(cache.shape)} does not fit {n_kv_heads} heads of size {head_dim}")
        if positions.numel() != x.shape[0] or seq_of_token.numel() != x.shape[0] or block_table.dim() != 2:
            raise KernelError("positions and seq_of_token must be [T], block_table [B, W]")
        return gemm_bf16_stream(
            x, weight, bias, torch.bfloat16,
            rope=(positions, seq_of_token, inv_freq, cache, block_table, n_q_heads, n_kv_heads, head_dim), streamed=streamed,
        )
    qkv = linear(x, weight, bias, partials_ok=True, streamed=streamed)
    if qkv.dim() == 3:
        # partial sums of a split K: added by the rotation kernel where it can, else by a kernel of their own
        if x.dtype == torch.bfloat16 and cache.dtype == torch.bfloat16 and head_dim % 8 == 0 and head_dim <= 256:
            return rope_kv_write_partials(qkv, n_q_heads, n_kv_heads, head_dim, positions, inv_freq, cache, block_table, seq_of_token)
        qkv = sum_partials(qkv, x.dtype)
    q_out, kv_out = n_q_heads * head_dim, n_kv_heads * head_dim
    q = qkv[:, :q_out].unflatten(1, (n_q_heads, head_dim))
    k = qkv[:, q_out : q_out + kv_out].unflatten(1, (n_kv_heads, head_dim))
    v = qkv[:, q_out + kv_out :].unflatten(1, (n_kv_heads, head_dim))
    rope_kv_write(q, k, v, positions, inv_freq, cache, block_table, seq_of_token)
    return qkv


def rope_kv_write_partials(
    partials: torch.Tensor,
    n_q_heads: int,
    n_kv_heads: int,
    head_dim: int,
    positions: torch.Tensor,
    inv_freq: Optional[torch.Tensor],
    cache: torch.Tensor,
    block_table: torch.Tensor,
    seq_of_token: torch.Tensor,
) -> torch.Tensor:
    """`rope_kv_write` from the float32 partial sums [P, T, (Hq + 2 Hkv) * hd] of the joined q/k/v
    projection: they are added in order and rounded to bfloat16 (the bits `sum_partials` gives), q
    and k are rotated, k and v written to the paged bfloat16 cache.  Returns [T, (Hq + 2 Hkv) * hd]."""
    _need_gpu(partials, positions, inv_freq, cache, block_table, seq_of_token)
    width = (n_q_heads + 2 * n_kv_heads) * head_dim
    if partials.dim() != 3 or partials.dtype != torch.float32 or partials.shape[2] != width or not partials.is_contiguous():
        raise KernelError(f"partial sums must be a contiguous float32 [P, T, {width}] tensor")
    n_part, n_tokens, _ = partials.shape
    if head_dim % 8 != 0 or cache.dtype != torch.bfloat16:
        raise KernelError("the rotation from partial sums takes head sizes of a multiple of 8 and a bfloat16 cache")
    _i32(positions, "positions")
    _i32(seq_of_token, "seq_of_token")
    _i32(block_table, "block_table")
    if inv_freq is not None and (inv_freq.dtype != torch.float32 or inv_freq.numel() != head_dim // 2 or not inv_freq.is_contiguous()):
        raise KernelError(f"the rotary table must be float32 [{head_dim // 2}]")
    if cache.dim() != 4 or cache.shape[1] != 2 or cache.shape[2] != n_kv_heads or cache.shape[3] % head_dim != 0 or not cache.is_contiguous():
        raise KernelError(f"cache {tuple(cache.shape)} does not fit {n_kv_heads} heads of size {head_dim}")
    if positions.numel() != n_tokens or seq_of_token.numel() != n_tokens or block_table.dim() != 2:
        raise KernelError("positions and seq_of_token must be [T], block_table [B, W]")
    out = torch.empty((n_tokens, width), dtype=torch.bfloat16, device=partials.device)
    lib = _build.load("rope_kv")
    _check(
        lib,
        lib.cwm_rope_kv_write_partials(
            _ptr(out), ctypes.c_long(width), _ptr(partials), ctypes.c_int(n_part), ctypes.c_long(n_tokens * width),
            _ptr(positions), _ptr(seq_of_token), _ptr(inv_freq), _ptr(cache), _ptr(block_table),
            ctypes.c_int(block_table.shape[1]), ctypes.c_int(cache.shape[3] // head_dim), ctypes.c_int(cache.shape[0]),
            ctypes.c_int(n_tokens), ctypes.c_int(n_q_heads), ctypes.c_int(n_kv_heads), ctypes.c_int(head_dim), _stream(),
        ),
    )
    return out


def sum_partials(partials: torch.Tensor, out_dtype: torch.dtype) -> torch.Tensor:
    """[P, M, N] float32 -> [M, N]: the partial sums added in order."""
    _need_gpu(partials)
    if partials.dim() != 3 or partials.dtype != torch.float32 or not partials.is_contiguous():
        raise KernelError("partial sums must be a contiguous float32 [P, M, N] tensor")
    p, m, n = partials.shape
    out = torch.empty((m, n), dtype=out_dtype, device=partials.device)
    lib = _build.load("rowwise")
    _check(lib, lib.cwm_sum_partials(_ptr(out), ctypes.c_int(_code(out_dtype)), _ptr(partials), ctypes.c_int(p), ctypes.c_long(m * n), _stream()))
    return out


TILE_MAX_ROWS = 512
_tile_slabs: dict = {}  # (rows, columns, K, blocks) -> slabs of partial results


def _tile_takes(x: torch.Tensor, weight: torch.Tensor) -> bool:
    k, n = x.shape[1], weight.shape[0]
    return (
        x.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16
        and k % 64 == 0 and n % 16 == 0 and 0 < x.shape[0] <= TILE_MAX_ROWS
        and x.stride(-1) == 1 and weight.stride(-1) == 1
        and (x.shape[0] <= 1 or x.stride(0) % 8 == 0) and (n <= 1 or weight.stride(0) % 8 == 0)
        and max(x.stride(0), weight.stride(0)) < (1 << 22)
        and x.data_ptr() % 16 == 0 and weight.data_ptr() % 16 == 0
    )


def gemm_bf16_tile(
    x: torch.Tensor,
    weight: torch.Tensor,
    bias: Optional[torch.Tensor] = None,
    out_dtype: Optional[torch.dtype] = None,
    partials_ok: bool = False,
    glu: bool = False,
    units: Optional[int] = None,
) -> torch.Tensor:
    """bfloat16 x [M <= 512, K] @ weight[N, K]^T with float32 sums: persistent blocks whose tiles
    of 64, 128 or 256 rows reach LDS by direct loads and that share the work by steps of K.  Returns
    [M, N]; with `partials_ok` it may return float32 partial sums [P, M, N] for the caller to add.
    `glu`: the weight's rows are gate and up rows in alternating groups of 8 and the result is
    silu(gate) * up, [M, N / 2] (in the kernel where a block owns whole tiles, else after it).
    `units` (tests) stands in for the number of compute units."""
    _need_gpu(x, weight, bias)
    if x.dim() != 2 or weight.dim() != 2 or x.shape[1] != weight.shape[1] or not _tile_takes(x, weight):
        raise KernelError(
            f"the tiled product takes bfloat16 x [0 < M <= {TILE_MAX_ROWS}, K] and weight [N, K] with K a multiple of 64, N of "
            f"16 and 16-byte aligned rows; got {tuple(x.shape)} {x.dtype} and {tuple(weight.shape)} {weight.dtype}"
        )
    m, k = x.shape
    n = weight.shape[0]
    if bias is not None and (bias.shape != (n,) or not bias.is_contiguous()):
        raise KernelError(f"gemm: bias {tuple(bias.shape)} does not fit {n} outputs")
    out_dtype = out_dtype or torch.bfloat16
    lib = _build.load("gemm_bf16_tile")
    units = units or _compute_units(x.device)
    slabs = _tile_slabs.get((m, n, k, units))
    if slabs is None:
        slabs = _tile_slabs[(m, n, k, units)] = int(lib.cwm_gemm_bf16_tile_slabs(m, n, k, units))
        if slabs < 1:
            raise KernelError(f"the tiled product has no cut for M={m} N={n} K={k}")
    fused_glu = glu and slabs == 1 and bias is None
    if fused_glu:
        out = torch.empty((m, n // 2), dtype=torch.bfloat16, device=x.device)
    elif slabs == 1:
        out = torch.empty((m, n), dtype=torch.float32 if bias is not None else (torch.bfloat16 if glu else out_dtype), device=x.device)
    else:
        out = torch.empty((slabs, m, n), dtype=torch.float32, device=x.device)
    _check(
        lib,
        lib.cwm_gemm_bf16_tile(
            _ptr(x), ctypes.c_long(x.stride(0) if m > 1 else k), _ptr(weight), ctypes.c_long(weight.stride(0) if n > 1 else k),
            _ptr(out), ctypes.c_int(_code(out.dtype)), ctypes.c_long(out.shape[-1]), ctypes.c_long(m * n),
            ctypes.c_int(m), ctypes.c_int(n), ctypes.c_int(k), ctypes.c_int(units), ctypes.c_int(slabs), ctypes.c_int(int(fused_glu)),
            _stream(),
        ),
    )
    if fused_glu:
        return out
    if bias is not None:  # not in the kernel; no model of this architecture has one on a product of this size
        if out.dim() == 3:
            out[0] += bias.float()
        else:
            out = out + bias.float()
    if glu:
        return silu_mul(out if out.dim() == 3 else out.to(torch.bfloat16), out_dtype=torch.bfloat16, grouped=True)
    if out.dim() == 3 and not partials_ok:
        return sum_partials(out, out_dtype)
    return out if out.dim() == 3 or out.dtype == out_dtype else out.to(out_dtype)


# rows up to which the streaming product (x in registers, every epilogue in the kernel) is preferred whatever the matrix
STREAM_FUSED_ROWS = 8
STREAM_EPILOGUE_ROWS = 32  # rows up to which its epilogues go
# From 9 to 32 rows the streaming product from a copy is ahead for matrices of fewer entries than these: it
# rotates, writes the cache and applies the gate in its epilogue, and leaves one to four partial sums where the tiled one, whose
# blocks share tiles of a small matrix, leaves up to 16.  Measured with the kernels that then follow, streamed / tiled, us: q/k/v of
# 3,072 x 2,048 6.5 / 13.1 at 12 rows and 7.9 / 13.5 at 24, of 6,144 x 4,096 14.8 / 20.5 at 12, of 8,192 x 6,144 21.0 / 24.2; gate/up
# of 16,384 x 2,048 14.2 / 16.6 and 15.0 / 17.1, of 28,672 x 4,096 39.1 / 42.0, but of 43,008 x 6,144 83.1 / 80.8; K split over blocks:
# 2,048 x 8,192 11.3 / 13.0 and 12.6 / 14.0, 3,072 x 9,216 15.4 / 17.4 and 16.9 / 18.3, but 4,096 x 14,336 26.6 / 24.8 and 28.1 / 25.9.
STREAM_WHOLE_ENTRIES = 1 << 27
STREAM_SPLIT_ENTRIES = 1 << 25
# Wide results of a short K are the tiled kernel's: its blocks own whole tiles there, while a streaming block pays its sum over
# the wavefronts for one 16-column tile after the other.  Streamed / tiled, us, at 9 rows and at 17: 24,576 x 512 11.0 / 8.7 and
# 9.1 / 8.9, 32,768 x 512 14.3 / 9.6 and 11.0 / 9.2, 32,768 x 768 13.6 / 11.6 and 11.3 / 11.8, 128,256 x 512 46 / 25 and 35 / 26; but 16,384 x
# 256 7.6 / 8.8 and 6.7 / 8.9, 20,480 x 1,024 11.4 / 14.1 and 9.6 / 14.7.  At a K of 1,024, 32,768 columns 16.3 / 15.1 and 12.9 / 14.1,
# 128,256 50 / 44 and 46 / 48.
STREAM_WIDE, STREAM_WIDE_K = 20480, 1024
STREAM_WIDER = 32768  # up to 16 rows the K of 1,024 itself is short from here on
# Matrices of fewer entries than this are streamed from 9 to 32 rows whether they have a copy or not, so that a copy does not
# decide on bits there (as below `TILE_FEW_ROWS_ENTRIES` up to 8 rows).  Streamed row-major / tiled, us, with the norm that follows, at 9 and
# 32 rows: 256 x 512 5.8 / 9.5 and 5.7 / 9.9, 1,024 x 2,048 7.0 / 9.6 and 7.1 / 10.1, 2,048 x 2,048 8.0 / 9.8 and 8.9 / 10.5, 512 x 8,064 7.7 / 12.4 and
# 9.3 / 13.1; above, the copy is what makes it worth while: 1,536 x 4,608 10.4 / 10.9 and 13.0 / 12.0, 2,048 x 6,144 11.2 / 11.5 and 15.1 / 12.9.
STREAM_ANY_ENTRIES = 1 << 22
# The smallest matrices (64 KB, a test model's) stay with the tiled kernel from 9 rows on, with a copy or without: some 2 us a product
# (208 x 128 8.3 instead of 5.9 us) are not worth other bits for what such models give.
STREAM_LEAST_ENTRIES = 1 << 15
TILE_ROWS = 128  # rows up to which the tiled product is the fastest whatever the shape
TILE_TALL_ROWS = 256  # rows of its tallest block: up to there it reads W once
TILE_COLUMNS = 128  # columns of a tall block's tile


# entries of a matrix from which on reading it is what a product of few rows costs (below, a launch more or less counts as much)
TILE_FEW_ROWS_ENTRIES = 1 << 24


def _wide_and_short(m: int, n: int, k: int) -> bool:
    return k < STREAM_WIDE_K and n >= STREAM_WIDE or k == STREAM_WIDE_K and n >= STREAM_WIDER and m <= 16


def _prefers_tile(
    x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor], streamed: Optional[torch.Tensor] = None, fused: bool = False,
) -> bool:
    """Whether this product goes to the tiled kernel (which has no bias of its own): from 33 rows on; from 9 on where
    the matrix is among the smallest (`STREAM_LEAST_ENTRIES`), wide and short, or so large that it pays to read it
    row-major in whole cache lines past the caches, which the streaming kernel can only do with a copy
    (`STREAM_WHOLE_ENTRIES` and `STREAM_SPLIT_ENTRIES` with one, `STREAM_ANY_ENTRIES` without); and for fewer rows
    where the matrix is large and has no streaming copy (a layer's four products of the 32B shape at 8 rows: 159 us tiled,
    187 us streamed from the row-major matrices, 159 us streamed from the copies; at 1 row 163, 178 and 154 us).
    `fused`: whether the streaming product would have an epilogue, which takes a longer K without a split."""
    if bias is not None:
        return False
    m = x.shape[0]
    if m <= STREAM_FUSED_ROWS and (streamed is not None or weight.numel() < TILE_FEW_ROWS_ENTRIES):
        return False
    if STREAM_FUSED_ROWS < m <= STREAM_EPILOGUE_ROWS:
        n, k = weight.shape
        if n * k >= STREAM_LEAST_ENTRIES and not _wide_and_short(m, n, k):
            with_copy = STREAM_WHOLE_ENTRIES if k <= stream_unsplit_k(m, fused) else STREAM_SPLIT_ENTRIES
            if n * k < (STREAM_ANY_ENTRIES if streamed is None else with_copy):
                return False
    return _tile_wins(x, weight)


def _tile_wins(x: torch.Tensor, weight: torch.Tensor) -> bool:
    """Whether the tiled product takes this product and is the fastest for it.  Above 128 rows its blocks of
    256 rows are bound by LDS and matrix cores, and the library is faster wherever its own tiles fill the
    chip.  Measured on the matrices of the 8B, 32B and 70B shapes at 160 and 256 rows: the tiled product,
    which shares K between blocks, is ahead where its tiles are at most half as many as the compute units
    (up to 16,384 columns: 41 against 67 us for the 32B shape's q/k/v product at 256 rows, 89 against 234 us
    for its feed-forward's second product).  With two blocks of rows (up to 512) it was ahead on that second
    product alone (144 against 195 us at 384 rows), which the float32 partial sums that the next kernel then
    reads cost again in a decode step, so more than 256 rows go to the wide kernel or the library (`_prefers_wide`)."""
    m = x.shape[0]
    if m > TILE_TALL_ROWS or not _tile_takes(x, weight):
        return False
    if m <= TILE_ROWS:
        return True
    return 2 * -(-weight.shape[0] // TILE_COLUMNS) <= _compute_units(x.device)


def _wide_takes(x: torch.Tensor, weight: torch.Tensor) -> bool:
    k, n = x.shape[1], weight.shape[0]
    return (
        x.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16
        and k % 64 == 0 and n % 16 == 0 and x.shape[0] > 0
        and x.stride(-1) == 1 and weight.stride(-1) == 1
        and (x.shape[0] <= 1 or x.stride(0) % 8 == 0) and (n <= 1 or weight.stride(0) % 8 == 0)
        and (x.shape[0] <= 1 or x.stride(0) >= k) and (n <= 1 or weight.stride(0) >= k)  # rows that overlap are the library's
        and max(x.stride(0), weight.stride(0)) < (1 << 22)
        and x.data_ptr() % 16 == 0 and weight.data_ptr() % 16 == 0
    )


def _prefers_wide(x: torch.Tensor, weight: torch.Tensor, glu: bool = False) -> bool:
    """Whether a product of more rows than the tiled kernel takes goes to the wide kernel instead of the library: where it is
    expected to be faster, by the costs of both kernels' tiles (csrc/gemm_bf16_wide.hip)."""
    if not _wide_takes(x, weight):
        return False
    return bool(_build.load("gemm_bf16_wide").cwm_gemm_bf16_wide_pays(x.shape[0], weight.shape[0], x.shape[1], _compute_units(x.device), int(glu)))


def _wide_keeps_sums(m: int, n: int, k: int) -> bool:
    """Whether the wide kernel's float32 sums are no further from the exact ones than the library's.  Both add K in its order, with the same bits, but
    where few or very many tiles make the library cut K, and its sums are then shorter: float32 results off float64, library / wide, 130 x 512 x 2,048
    1.3e-7 / 2.7e-7, 2,048 x 10,304 x 6,144 4.4e-7 / 5.0e-7, 600 x 1,024 x 21,504 5.9e-7 / 9.4e-7.  Of 2,162 sizes with a K of 512 to 28,672 none in these
    bounds is.  A bfloat16 result does not show it: rounded, the errors differ by a millionth of themselves."""
    return k <= 1024 or (k <= 2048 and (1 << 17) < m * n <= (1 << 26))


def gemm_bf16_wide(
    x: torch.Tensor, weight: torch.Tensor, out_dtype: Optional[torch.dtype] = None, glu: bool = False, units: Optional[int] = None,
    tile: Optional[int] = None,
) -> torch.Tensor:
    """bfloat16 x [M, K] @ weight[N, K]^T with float32 sums, [M, N] in bfloat16 or float32: persistent blocks whose tiles of
    64 to 256 rows and 128 or 256 columns reach LDS by direct loads.  `glu`: the weight's rows are gate and up rows in
    alternating groups of 8 and the result is silu(gate) * up, [M, N / 2] in bfloat16.  `units` (tests) stands in for the
    number of compute units, `tile` (tests) names one of the kernel's tiles."""
    _need_gpu(x, weight)
    if x.dim() != 2 or weight.dim() != 2 or x.shape[1] != weight.shape[1] or not _wide_takes(x, weight):
        raise KernelError(
            "the wide product takes bfloat16 x [M, K] and weight [N, K] with K a multiple of 64, N of 16 and 16-byte aligned "
            f"rows; got {tuple(x.shape)} {x.dtype} and {tuple(weight.shape)} {weight.dtype}"
        )
    m, k = x.shape
    n = weight.shape[0]
    out = torch.empty((m, n // 2 if glu else n), dtype=torch.bfloat16 if glu else out_dtype or torch.bfloat16, device=x.device)
    lib = _build.load("gemm_bf16_wide")
    _check(
        lib,
        lib.cwm_gemm_bf16_wide(
            _ptr(x), ctypes.c_long(x.stride(0) if m > 1 else k), _ptr(weight), ctypes.c_long(weight.stride(0)), _ptr(out),
            ctypes.c_int(_code(out.dtype)), ctypes.c_long(out.shape[1]), ctypes.c_int(m), ctypes.c_int(n), ctypes.c_int(k),
            ctypes.c_int(units or _compute_units(x.device)), ctypes.c_int(int(glu)), ctypes.c_int(-1 if tile is None else tile), _stream(),
        ),
    )
    return out


def _stream_takes(x: torch.Tensor, weight: torch.Tensor) -> bool:
    k = x.shape[1]
    return (
        k % 8 == 0
        and x.stride(-1) == 1 and weight.stride(-1) == 1
        and (x.shape[0] <= 1 or x.stride(0) % 8 == 0)
        and (weight.shape[0] <= 1 or weight.stride(0) % 8 == 0)
        and x.data_ptr() % 16 == 0 and weight.data_ptr() % 16 == 0
    )


def gemm_bf16(
    x: torch.Tensor,
    weight: torch.Tensor,
    bias: Optional[torch.Tensor] = None,
    out_dtype: Optional[torch.dtype] = None,
    partials_ok: bool = False,
    streamed: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """bfloat16 x [M, K] @ bfloat16 weight[N, K]^T, float32 accumulation.

    Up to 8 rows, and up to 32 for all but the smallest and the largest matrices (`_prefers_tile`): the hand-written
    persistent weight-streaming kernel, x in registers.
    Up to 128 rows (256 for a result of at most 16,384 columns): the hand-written tiled kernel, x and W
    through LDS (it needs K % 64 == 0 and N % 16 == 0; other sizes of up to 64 rows stream).
    More rows: the hand-written wide kernel where it is ahead of the library, mostly where the library's tiles would leave much
    of the chip idle (`_prefers_wide`; it needs the same sizes and no bias), else the library product (hipBLASLt through torch), as the reference calls a
    library here, with a bfloat16 or a float32 result.  Row lengths that are no multiple
    of 8 go to the float32 kernel, which takes any size.
    """
    _need_gpu(x, weight, bias)
    out_dtype = out_dtype or torch.bfloat16
    m = x.shape[0]
    if not _stream_takes(x, weight):
        return gemm_f32(x, weight, bias, out_dtype)
    if _prefers_tile(x, weight, bias, streamed):
        return gemm_bf16_tile(x, weight, None, out_dtype, partials_ok)
    if m <= STREAM_MAX_ROWS:
        return gemm_bf16_stream(x, weight, bias, out_dtype, partials_ok, streamed=streamed, keep_sums=bias is None and m > STREAM_FUSED_ROWS)
    if bias is None and (out_dtype != torch.float32 or _wide_keeps_sums(m, *weight.shape)) and _prefers_wide(x, weight):
        return gemm_bf16_wide(x, weight, out_dtype)
    if out_dtype == torch.float32:
        y = torch.mm(x, weight.t(), out_dtype=torch.float32)  # bfloat16 operands, float32 sums written as they are
        return y if bias is None else y + bias.float()
    if bias is not None:
        return torch.addmm(bias.to(x.dtype), x, weight.t())  # the bias rides in the library's epilogue
    # one call whatever the shape: nothing is timed or tuned inside a step, so the same step gives the same bits
    # in every process.  (Calls on column ranges of a wide output were measured: at most 3% faster at 2,048 rows.)
    return torch.mm(x, weight.t())


# --------------------------------------------------------------------------- #
def rope_kv_write(
    q: torch.Tensor,
    k: Optional[torch.Tensor],
    v: Optional[torch.Tensor],
    positions: torch.Tensor,
    inv_freq: Optional[torch.Tensor],
    cache: Optional[torch.Tensor] = None,
    block_table: Optional[torch.Tensor] = None,
    seq_of_token: Optional[torch.Tensor] = None,
) -> None:
    """Rotate `q` [T, Hq, hd] and `k` [T, Hkv, hd] in place by positions * inv_freq
    (adjacent pairs) and write the rotated keys and `v` into the paged `cache`
    ([pages, 2, Hkv, page * hd]; keys [slot][dim], values [slot / 8][dim][slot % 8])
    at the rows the block table gives.  `q`, `k`, `v`
    may be views into one wider tensor (token stride free, heads contiguous)."""
    _need_gpu(q, k, v, positions, inv_freq, cache, block_table, seq_of_token)
    if q.dim() != 3 or q.stride(2) != 1 or q.stride(1) != q.shape[2]:
        raise KernelError("q must be [T, Hq, hd] with contiguous heads")
    n_tokens, n_q, hd = q.shape
    n_kv = 0
    for name, t in (("k", k), ("v", v)):
        if t is not None:
            if t.dim() != 3 or t.shape[0] != n_tokens or t.shape[2] != hd or t.stride(2) != 1 or t.stride(1) != hd:
                raise KernelError(f"{name} must be [T, Hkv, hd] with contiguous heads")
            if t.dtype != q.dtype:
                raise KernelError("q, k and v must have one type")
            n_kv = t.shape[1]
    _i32(positions, "positions")
    if positions.numel() != n_tokens:
        raise KernelError("one position per token is needed")
    if inv_freq is not None and (inv_freq.dtype != torch.float32 or inv_freq.numel() != hd // 2 or not inv_freq.is_contiguous()):
        raise KernelError(f"the rotary table must be float32 [{hd // 2}]")
    page_size = num_pages = width = 0
    if cache is not None:
        if k is None or v is None or block_table is None or seq_of_token is None:
            raise KernelError("a cache write needs k, v, a block table and the sequence of each token")
        if cache.dim() != 4 or cache.shape[1] != 2 or cache.shape[2] != n_kv or cache.shape[3] % hd != 0 or not cache.is_contiguous():
            raise KernelError(f"cache {tuple(cache.shape)} does not fit {n_kv} heads of size {hd}")
        if cache.dtype != q.dtype:
            raise KernelError("the cache and q, k, v must have one type")
        _i32(block_table, "block_table")
        _i32(seq_of_token, "seq_of_token")
        if block_table.dim() != 2 or seq_of_token.numel() != n_tokens:
            raise KernelError("block_table must be [B, W] and seq_of_token [T]")
        num_pages, page_size, width = cache.shape[0], cache.shape[3] // hd, block_table.shape[1]
    lib = _build.load("rope_kv")
    _check(
        lib,
        lib.cwm_rope_kv_write(
            _ptr(q), ctypes.c_long(q.stride(0)),
            _ptr(k), ctypes.c_long(k.stride(0) if k is not None else 0),
            _ptr(v), ctypes.c_long(v.stride(0) if v is not None else 0),
            ctypes.c_int(_code(q.dtype)), _ptr(positions), _ptr(seq_of_token), _ptr(inv_freq),
            _ptr(cache), _ptr(block_table), ctypes.c_int(width), ctypes.c_int(page_size), ctypes.c_int(num_pages),
            ctypes.c_int(n_tokens), ctypes.c_int(n_q), ctypes.c_int(n_kv if k is not None else 0), ctypes.c_int(hd),
            _stream(),
        ),
    )


def _check_sink(sink: Optional[torch.Tensor], n_q: int) -> None:
    if sink is not None and (sink.dtype != torch.float32 or sink.shape != (n_q,) or not sink.is_contiguous()):
        raise KernelError(f"the sinks must be a contiguous float32 [{n_q}] tensor, one a query head")


def _check_bias(distance_bias: Optional[Tuple[torch.Tensor, torch.Tensor]], n_q: int) -> Tuple[Optional[torch.Tensor], Optional[torch.Tensor]]:
    if distance_bias is None:
        return None, None
    for t in distance_bias:
        _need_gpu(t)
        if t.dtype != torch.float32 or t.shape != (n_q,) or not t.is_contiguous():
            raise KernelError(f"a distance bias is two contiguous float32 [{n_q}] tensors, a slope and a rate a query head")
    return distance_bias


def _check_mask(window: Optional[int], chunk: Optional[int], softcap: Optional[float]) -> None:
    if window is not None and window < 1:
        raise KernelError("a window holds at least the query's own key")
    if chunk is not None and (chunk < 1 or window is not None):
        raise KernelError("a block of keys holds at least one position, and comes instead of a window")
    if softcap is not None and not softcap > 0:
        raise KernelError("a cap on the scores must be positive")


def _check_kept(q: torch.Tensor, window: Optional[int], chunk: Optional[int], keep_first: int, out_scale: Optional[torch.Tensor]) -> None:
    if keep_first < 0 or (keep_first > 0 and (chunk is not None or window is None)):
        raise KernelError("kept first keys go with a window")
    if out_scale is not None and (
        q.dim() != 3 or out_scale.dtype != torch.float32 or tuple(out_scale.shape) != tuple(q.shape[:2]) or not out_scale.is_contiguous()
    ):
        raise KernelError("out_scale must be contiguous float32 [T, Hq]")


def paged_attention_simple(
    q: torch.Tensor,
    cache: torch.Tensor,
    block_table: torch.Tensor,
    positions: torch.Tensor,
    seq_of_token: torch.Tensor,
    window: Optional[int],
    scale: float,
    max_keys: Optional[int] = None,
    sink: Optional[torch.Tensor] = None,
    softcap: Optional[float] = None,
    chunk: Optional[int] = None,
    distance_bias: Optional[Tuple[torch.Tensor, torch.Tensor]] = None,
    keep_first: int = 0,
    out_scale: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """Causal attention of `q` [T, Hq, hd] over the paged cache by the plain kernel:
    float32 arithmetic, a key/value head's query heads sharing its keys and values, long
    key ranges cut into segments that a second kernel joins.  `window`: keys read per
    query, own included (None: all).  `max_keys`: the most keys any token reads (default:
    from the largest position, which costs a copy to the host).  `sink`: float32 [Hq], a term exp(sink) that
    each head's softmax denominator holds beside its keys (no key, no value, not scaled).  `softcap`: scaled scores
    become softcap * tanh(score / softcap) before the softmax.  `chunk` (instead of a window): a query reads the keys of
    its own block of that many positions, counted from 0, up to itself.  `distance_bias` (slope, rate), float32 [Hq]
    each: slope_h * ln(1 + rate_h * (query's position - key's)) comes off the score.  `keep_first` (with a window): a query
    also reads the sequence's first so many keys, however far back.  `out_scale`: float32 [T, Hq], a factor on every
    head's result.  Returns [T, Hq * hd]."""
    _need_gpu(q, cache, block_table, positions, seq_of_token, sink, out_scale)
    _check_kept(q, window, chunk, keep_first, out_scale)
    bias_slope, bias_rate = _check_bias(distance_bias, q.shape[1] if q.dim() == 3 else 0)
    _check_mask(window, chunk, softcap)
    _check_sink(sink, q.shape[1] if q.dim() == 3 else 0)
    if q.dim() != 3 or q.stride(2) != 1 or q.stride(1) != q.shape[2]:
        raise KernelError("q must be [T, Hq, hd] with contiguous heads")
    n_tokens, n_q, hd = q.shape
    if cache.dim() != 4 or cache.shape[1] != 2 or cache.shape[3] % hd != 0 or not cache.is_contiguous():
        raise KernelError(f"cache {tuple(cache.shape)} does not fit heads of size {hd}")
    if cache.dtype != q.dtype:
        raise KernelError("the cache and q must have one type")
    n_kv = cache.shape[2]
    _i32(block_table, "block_table")
    _i32(positions, "positions")
    _i32(seq_of_token, "seq_of_token")
    if positions.numel() != n_tokens or seq_of_token.numel() != n_tokens or block_table.dim() != 2:
        raise KernelError("positions and seq_of_token must be [T], block_table [B, W]")
    out = torch.empty((n_tokens, n_q * hd), dtype=q.dtype, device=q.device)
    lib = _build.load("attention_simple")
    if max_keys is None:
        max_keys = int(positions.max()) + 1 if n_tokens else 1
    if window is not None or chunk is not None:
        max_keys = min(max_keys, window if chunk is None else chunk)
    max_keys = max(1, max_keys)
    partial = None
    if max_keys > lib.cwm_attention_simple_segment_keys():
        partial = torch.empty(n_tokens * n_q * lib.cwm_attention_simple_max_segments() * (hd + 2), dtype=torch.float32, device=q.device)
    _check(
        lib,
        lib.cwm_attention_simple(
            _ptr(q), ctypes.c_long(q.stride(0)), _ptr(out), ctypes.c_long(n_q * hd), _ptr(cache),
            ctypes.c_int(_code(q.dtype)), _ptr(block_table), ctypes.c_int(block_table.shape[1]),
            _ptr(positions), _ptr(seq_of_token), ctypes.c_int(n_tokens), ctypes.c_int(n_q), ctypes.c_int(n_kv),
            ctypes.c_int(hd), ctypes.c_int(cache.shape[3] // hd), ctypes.c_int(cache.shape[0]),
            ctypes.c_int(-1 if window is None else window - 1), ctypes.c_int(chunk or 0), ctypes.c_float(scale),
            ctypes.c_float(softcap or 0.0), ctypes.c_int(max_keys), _ptr(partial), _ptr(sink), _ptr(bias_slope), _ptr(bias_rate),
            ctypes.c_int(keep_first), _ptr(out_scale), _stream(),
        ),
    )
    return out


@dataclass
class _UploadedPlan:
    """A step's attention work lists on the device, and what the launch needs to know of them."""

    work: torch.Tensor  # items of one row tile
    wide: torch.Tensor  # items of `item_tiles` row tiles
    merge: torch.Tensor
    n_work: int
    n_wide: int
    n_merge: int
    n_merge_mid: int  # merge items of at most 32 partials, after those with more
    n_merge_wide: int  # merge items of cut wide items, last in the list
    n_partials: int
    work_keys: int  # keys of an average item of one row tile
    wide_shape: Tuple[int, float]  # key tiles of the longest wide item, and the mean
    item_tiles: int = WIDE_TILES  # row tiles of a wide item


class StaticPlans:
    """The attention work lists of a step that is captured once and replayed: every list has a home of a
    fixed size at a fixed address, which `refresh` fills for each new step (unused places hold null items),
    so that the captured launches stay valid while the sequences grow.  The first, uncaptured run of the step
    finds out which lists the model's layers ask for and makes their homes."""

    def __init__(self, device: torch.device, max_keys: int) -> None:
        self.device = device
        self.max_keys = max_keys  # the most keys a sequence may hold while the capture is in use
        self.homes: dict = {}  # (group, key/value heads, window, chunk, whether keys are cut finer) -> (capacity, device vector, uploaded plan)

    def _padded(self, batch, group: int, n_kv: int, window: Optional[int], capacity, chunk: Optional[int], finer: bool):
        from .attention_plan import build_plan, capacity_until, pad_plan

        wide_cut_below = -(-2 * _compute_units(self.device) // n_kv)
        if capacity is None:
            plan, capacity = capacity_until(batch.q_lens, batch.kv_lens, group, window, wide_cut_below, self.max_keys, chunk, finer)
        else:
            plan = build_plan(batch.q_lens, batch.kv_lens, group, window, wide_cut_below, chunk, finer)
        flat = pad_plan(plan, capacity)
        return plan, capacity, flat

    def plan(self, batch, group: int, n_kv: int, window: Optional[int], chunk: Optional[int], finer: bool) -> "_UploadedPlan":
        key = (group, n_kv, window, chunk, finer)
        home = self.homes.get(key)
        if home is None:
            plan, capacity, flat = self._padded(batch, group, n_kv, window, None, chunk, finer)
            if flat is None:
                raise KernelError("this step's attention work has items that a captured step does not take")
            dev = torch.from_numpy(flat).pin_memory().to(self.device, non_blocking=True)
            a = capacity.work * 6
            uploaded = _UploadedPlan(
                work=dev[:a], wide=dev[a:a], merge=dev[a:], n_work=capacity.work, n_wide=0, n_merge=capacity.merge,
                n_merge_mid=capacity.merge_mid, n_merge_wide=0, n_partials=capacity.work,
                work_keys=int((plan.work[:, 3] - plan.work[:, 2]).mean()) if plan.work.shape[0] else 0, wide_shape=(0, 0.0),
            )
            home = self.homes[key] = (capacity, dev, uploaded)
        return home[2]

    def refresh(self, batch) -> bool:
        """Fill every home with the lists of `batch`; False if one of them has outgrown its home."""
        for (group, n_kv, window, chunk, finer), (capacity, dev, _) in self.homes.items():
            _, _, flat = self._padded(batch, group, n_kv, window, capacity, chunk, finer)
            if flat is None:
                return False
            dev.copy_(torch.from_numpy(flat).pin_memory(), non_blocking=True)
        return True


def _attention_plan(
    batch, group: int, n_kv: int, head_dim: int, window: Optional[int], device: torch.device, chunk: Optional[int] = None, halves: bool = False,
) -> _UploadedPlan:
    """The step's work list for this (group size, key/value heads and their size, window or block of keys), uploaded once per step.
    `halves`: whether blocks of 64 rows are built for what the layer has (`_half_blocks_built`)."""
    from .attention_plan import build_plan, cuts_finer, wide_item_tiles

    finer = cuts_finer(n_kv, head_dim)
    static = getattr(batch, "static", None)
    if static is not None:
        return static.plan(batch, group, n_kv, window, chunk, finer)
    # with such blocks the list depends on the head size, by which they are chosen; layers of other sizes have lists of their own
    key = ("attention_plan", group, n_kv, window, chunk, finer, head_dim if halves else None)
    cached = batch.scratch.get(key)
    if cached is None:
        # a sequence whose blocks of 128 rows, over all key/value heads, would not give every compute unit two
        wide_cut_below = -(-2 * _compute_units(device) // n_kv) if device.type == "cuda" else 0
        item_tiles = WIDE_TILES
        if device.type == "cuda" and halves:
            item_tiles = wide_item_tiles(batch.q_lens, batch.kv_lens, group, n_kv, head_dim, wide_cut_below, _compute_units(device))
        plan = build_plan(batch.q_lens, batch.kv_lens, group, window, wide_cut_below, chunk, finer, item_tiles)
        flat = np.concatenate([plan.work.reshape(-1), plan.work_wide.reshape(-1), plan.merge.reshape(-1)]).astype(np.int32)
        host = torch.from_numpy(flat)
        if device.type == "cuda":
            host = host.pin_memory()
        dev = host.to(device, non_blocking=True)
        n_work, n_wide, n_merge = plan.work.shape[0], plan.work_wide.shape[0], plan.merge.shape[0]
        a, b = n_work * 6, (n_work + n_wide) * 6
        wide_tiles = (plan.work_wide[:, 3] - (plan.work_wide[:, 2] & ~31) + 31) // 32 if n_wide else None  # key tiles of each wide item
        cached = _UploadedPlan(
            work=dev[:a], wide=dev[a:b], merge=dev[b:], n_work=n_work, n_wide=n_wide, n_merge=n_merge,
            n_merge_mid=plan.n_merge_mid, n_merge_wide=plan.n_merge_wide, n_partials=plan.n_partials,
            work_keys=int((plan.work[:, 3] - plan.work[:, 2]).mean()) if n_work else 0,
            wide_shape=(int(wide_tiles.max()), float(wide_tiles.mean())) if n_wide else (0, 0.0), item_tiles=item_tiles,
        )
        batch.scratch[key] = cached
    return cached


# a block's time for one tile of keys when three blocks share a compute unit, over that with two
_THREE_BLOCKS_TILE_TIME = 1.38


def _three_blocks_a_unit(n_blocks: int, shape: Tuple[int, float], device: torch.device) -> int:
    """Whether the blocks that share keys and values through LDS finish sooner three to a
    compute unit (the build with three buffers) than two (four buffers): `shape` is the
    longest block and the mean, in key tiles.  Two finish a launch of few, uneven blocks
    sooner (the longest block sets the time, and runs faster with one neighbour); three hide
    more latency when there are rounds of blocks.  Estimate of either: the longer of the
    longest block and the mean times the number of rounds, times a tile's time."""
    if n_blocks == 0:
        return 0
    units = _compute_units(device)
    longest, mean = shape
    two = max(longest, mean * -(-n_blocks // (2 * units)))
    three = _THREE_BLOCKS_TILE_TIME * max(longest, mean * -(-n_blocks // (3 * units)))
    return int(three < two)


def _half_blocks_built(n_kv: int, head_dim: int, page_size: int, keep_first: int = 0) -> bool:
    """Whether the matrix-core attention kernel has blocks of 64 rows for these sizes: the head sizes and pages whose keys and
    values the loads write to LDS themselves.  Not with kept first keys: a block takes those before its rows' windows ahead
    of them, so a tile that holds both is one pass or two by where the block's first row stands, and a row's bits would
    depend on the block's height, that is on what else is in the step."""
    return head_dim in _work_lists.WIDE_HALF_BLOCKS and page_size % 32 == 0 and n_kv * page_size * head_dim * 2 < 2 ** 31 and keep_first == 0


def mfma_attention_takes(dtype: torch.dtype, head_dim: int, page_size: int) -> bool:
    """Sizes the matrix-core attention kernel covers; everything else runs on the
    plain kernel."""
    return dtype == torch.bfloat16 and head_dim % 16 == 0 and 16 <= head_dim <= 256 and page_size % 8 == 0


def paged_attention_mfma(
    q: torch.Tensor,
    cache: torch.Tensor,
    block_table: torch.Tensor,
    batch,
    window: Optional[int],
    scale: float,
    sink: Optional[torch.Tensor] = None,
    softcap: Optional[float] = None,
    chunk: Optional[int] = None,
    distance_bias: Optional[Tuple[torch.Tensor, torch.Tensor]] = None,
    keep_first: int = 0,
    out_scale: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """Matrix-core attention (bfloat16): prompt portions and decoded tokens in one
    launch, long key ranges of short sequences split and merged.  `sink`, `softcap`, `chunk`, `distance_bias`, `keep_first`,
    `out_scale`: as in `paged_attention_simple`; the bias and the kept keys are builds of their own, so that the other
    models' kernel does without their instructions."""
    _check_kept(q, window, chunk, keep_first, out_scale)
    bias_slope, bias_rate = _check_bias(distance_bias, q.shape[1] if q.dim() == 3 else 0)
    _need_gpu(q, cache, block_table, sink, out_scale)
    _check_mask(window, chunk, softcap)
    _check_sink(sink, q.shape[1] if q.dim() == 3 else 0)
    if q.dtype != torch.bfloat16 or cache.dtype != torch.bfloat16:
        raise KernelError("the matrix-core attention kernel takes bfloat16 only")
    if q.dim() != 3 or q.stride(2) != 1 or q.stride(1) != q.shape[2]:
        raise KernelError("q must be [T, Hq, hd] with contiguous heads")
    n_tokens, n_q, hd = q.shape
    if cache.dim() != 4 or cache.shape[1] != 2 or cache.shape[3] % hd != 0 or not cache.is_contiguous():
        raise KernelError(f"cache {tuple(cache.shape)} does not fit heads of size {hd}")
    n_kv = cache.shape[2]
    page_size = cache.shape[3] // hd
    if not mfma_attention_takes(q.dtype, hd, page_size):
        raise KernelError(f"the matrix-core attention kernel does not take head_dim {hd} with pages of {page_size}")
    if n_q % n_kv != 0:
        raise KernelError(f"{n_q} query heads do not divide into {n_kv} key/value heads")
    if q.stride(0) % 8 != 0 or q.data_ptr() % 16 != 0:
        raise KernelError("q rows must be 16-byte aligned")
    _i32(block_table, "block_table")
    if block_table.dim() != 2 or block_table.shape[0] != batch.n_seqs or n_tokens != batch.n_tokens:
        raise KernelError("block_table must be [B, W] for the batch's sequences, q [T, ...] for its tokens")
    plan = _attention_plan(batch, n_q // n_kv, n_kv, hd, window, q.device, chunk, _half_blocks_built(n_kv, hd, page_size, keep_first))
    out = torch.empty((n_tokens, n_q * hd), dtype=q.dtype, device=q.device)
    partial = None
    if plan.n_partials:
        partial = torch.empty(plan.n_partials * n_kv * 16 * (hd + 4), dtype=torch.float32, device=q.device)
    defines = {"HEAD_DIM": hd}
    if distance_bias is not None:
        defines["DISTANCE_BIAS"] = 1
    if keep_first > 0:
        defines["KEPT_KEYS"] = 1
    lib = _build.load("attention_mfma", defines)
    _check(
        lib,
        lib.cwm_attention_mfma(
            _ptr(q), ctypes.c_long(q.stride(0)), _ptr(out), ctypes.c_long(n_q * hd), _ptr(cache),
            _ptr(block_table), ctypes.c_int(block_table.shape[1]), _ptr(batch.cu_q), _ptr(batch.kv_len),
            _ptr(plan.work), ctypes.c_int(plan.n_work), ctypes.c_int(plan.work_keys),
            _ptr(plan.wide), ctypes.c_int(plan.n_wide), ctypes.c_int(plan.item_tiles),
            ctypes.c_int(_three_blocks_a_unit(plan.n_wide * n_kv, plan.wide_shape, q.device)),
            _ptr(plan.merge), ctypes.c_int(plan.n_merge), ctypes.c_int(plan.n_merge_mid), ctypes.c_int(plan.n_merge_wide), _ptr(partial),
            ctypes.c_int(n_q), ctypes.c_int(n_kv), ctypes.c_int(hd), ctypes.c_int(page_size),
            ctypes.c_int(cache.shape[0]), ctypes.c_int(-1 if window is None else window - 1), ctypes.c_int(chunk or 0),
            ctypes.c_float(scale), ctypes.c_float(softcap or 0.0), _ptr(sink), _ptr(bias_slope), _ptr(bias_rate), _ptr(out_scale),
            ctypes.c_int(keep_first), _stream(),
        ),
    )
    return out


def paged_attention(
    q: torch.Tensor,
    cache: torch.Tensor,
    block_table: torch.Tensor,
    batch,
    window: Optional[int],
    scale: float,
    sink: Optional[torch.Tensor] = None,
    softcap: Optional[float] = None,
    chunk: Optional[int] = None,
    distance_bias: Optional[Tuple[torch.Tensor, torch.Tensor]] = None,
    keep_first: int = 0,
    out_scale: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """Attention of the step's tokens over the cache.  `batch` is the step's
    `StepBatch` (positions, sequence of each token and the per-sequence lengths).
    bfloat16 with head sizes in steps of 16 and pages in steps of 8 runs on the
    matrix cores; float32, and other sizes, on the plain kernel."""
    hd = q.shape[2]
    if q.is_cuda and mfma_attention_takes(q.dtype, hd, cache.shape[3] // hd):
        return paged_attention_mfma(q, cache, block_table, batch, window, scale, sink, softcap, chunk, distance_bias, keep_first, out_scale)
    static = getattr(batch, "static", None)
    max_keys = batch.max_kv_len if static is None else static.max_keys
    return paged_attention_simple(
        q, cache, block_table, batch.positions, batch.seq_of_token, window, scale, max_keys=max_keys, sink=sink, softcap=softcap, chunk=chunk,
        distance_bias=distance_bias, keep_first=keep_first, out_scale=out_scale,
    )


# --------------------------------------------------------------------------- #
def sample_packed(
    logits: torch.Tensor,
    temperature: torch.Tensor,
    top_p: torch.Tensor,
    uniform: torch.Tensor,
) -> torch.Tensor:
    """Per row of float32 `logits` [R, V]: greedy where temperature <= 0, else a draw
    from softmax(logits / T) cut to the nucleus `top_p`, using the row's uniform
    number.  Returns one int32 tensor [3, R], so that everything reaches the host in one
    copy: the tokens, then the bits of the float32 log-probabilities log softmax(logits)
    at the token and of the token under the sampling distribution (`unpack_sampled`)."""
    _need_gpu(logits, temperature, top_p, uniform)
    if logits.dtype != torch.float32 or logits.dim() != 2 or logits.stride(1) != 1:
        raise KernelError("logits must be float32 [R, V] with contiguous rows")
    n_rows, vocab = logits.shape
    for name, t in (("temperature", temperature), ("top_p", top_p), ("uniform", uniform)):
        if t.dtype != torch.float32 or t.numel() != n_rows or not t.is_contiguous():
            raise KernelError(f"{name} must be float32 [{n_rows}]")
    dev = logits.device
    out = torch.empty((3, n_rows), dtype=torch.int32, device=dev)
    workspace = torch.empty((max(n_rows, 1), vocab), dtype=torch.float32, device=dev)
    lib = _build.load("sampling")
    _check(
        lib,
        lib.cwm_sample(
            _ptr(logits), ctypes.c_long(logits.stride(0) if n_rows > 1 else vocab), ctypes.c_int(n_rows),
            ctypes.c_int(vocab), _ptr(temperature), _ptr(top_p), _ptr(uniform), _ptr(workspace),
            _ptr(out[0]), _ptr(out[1]), _ptr(out[2]), _stream(),
        ),
    )
    return out


def unpack_sampled(packed: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """(tokens int32, logprobs float32, sample_logprobs float32) as views of what `sample_packed` returned
    ([3, R], on any device)."""
    return packed[0], packed[1].view(torch.float32), packed[2].view(torch.float32)


def sample(
    logits: torch.Tensor,
    temperature: torch.Tensor,
    top_p: torch.Tensor,
    uniform: torch.Tensor,
) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """`sample_packed` as three tensors: (tokens int32, logprobs, sample_logprobs)."""
    return unpack_sampled(sample_packed(logits, temperature, top_p, uniform))


def token_logprobs(logits: torch.Tensor, rows: torch.Tensor, targets: torch.Tensor) -> torch.Tensor:
    """log softmax(logits[rows[i]])[targets[i]] (float32 [n]) for int32 `rows`, `targets`."""
    _need_gpu(logits, rows, targets)
    if logits.dtype != torch.float32 or logits.dim() != 2 or logits.stride(1) != 1:
        raise KernelError("logits must be float32 [R, V] with contiguous rows")
    _i32(rows, "rows")
    _i32(targets, "targets")
    if rows.numel() != targets.numel():
        raise KernelError("one target per row is needed")
    out = torch.empty(rows.numel(), dtype=torch.float32, device=logits.device)
    lib = _build.load("sampling")
    _check(
        lib,
        lib.cwm_token_logprob(
            _ptr(logits), ctypes.c_long(logits.stride(0) if logits.shape[0] > 1 else logits.shape[1]),
            ctypes.c_int(logits.shape[0]), ctypes.c_int(logits.shape[1]), _ptr(rows), _ptr(targets),
            ctypes.c_int(rows.numel()), _ptr(out), _stream(),
        ),
    )
    return out


__all__ = [
    "KernelError",
    "KernelBuildError",
    "embedding",
    "add_rmsnorm",
    "silu_mul",
    "gemm_f32",
    "gemm_f32_stream",
    "gemm_bf16",
    "gemm_bf16_stream",
    "linear_inputs",
    "linear_inputs_takes",
    "sum_partials",
    "linear",
    "rope_kv_write",
    "qkv_rope_write",
    "paged_attention_simple",
    "paged_attention_mfma",
    "mfma_attention_takes",
    "paged_attention",
    "sample",
    "sample_packed",
    "unpack_sampled",
    "token_logprobs",
]


# --------------------------------------------------------------------------- #
# what the GPU at hand reaches (for the measurement program; nothing on the model's path)
def measure_read_rate(buffer: torch.Tensor, window_bytes: int, launches: int, blocks: int) -> float:
    """GB/s at which a kernel that only reads gets through `window_bytes` of `buffer` (uint8, on the device):
    `launches` launches back to back, each on the next window of the buffer (so that, with a buffer several times
    the last-level cache, no launch finds its bytes cached), timed by events around all of them."""
    _need_gpu(buffer)
    if buffer.dtype != torch.uint8 or not buffer.is_contiguous() or window_bytes % 16 != 0 or not 0 < window_bytes <= buffer.numel():
        raise KernelError("measure_read_rate takes a contiguous uint8 buffer and a window that is a multiple of 16 bytes within it")
    lib = _build.load("ceilings")
    windows = max(1, buffer.numel() // window_bytes)
    base = buffer.data_ptr()
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    stream = _stream()
    for timed in (False, True):
        if timed:
            start.record()
        for i in range(launches if timed else 2):
            offset = (i % windows) * window_bytes
            _check(lib, lib.cwm_ceiling_read(ctypes.c_void_p(base + offset), ctypes.c_long(window_bytes), ctypes.c_int(blocks), ctypes.c_void_p(0), stream))
        if timed:
            end.record()
        torch.cuda.synchronize(buffer.device)
    return window_bytes * launches / (start.elapsed_time(end) * 1e-3) / 1e9


def measure_mfma_rate(device: torch.device, blocks: int, rounds: int, launches: int = 3, shape: int = 16, seed: float = 1.0) -> float:
    """PFLOP/s of the bfloat16 matrix instruction (`shape` 16: 16x16x32, 32: 32x32x16; float32 sums) issued from
    registers by `blocks` blocks of four wavefronts, `rounds` rounds of eight independent instructions each, on
    operands of `seed` times small varied numbers (0: all zeros, which costs the least power)."""
    lib = _build.load("ceilings")
    lib.cwm_ceiling_mfma_flops.restype = ctypes.c_double
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    with torch.cuda.device(device):
        stream = _stream()
        for timed in (False, True):
            if timed:
                start.record()
            for _ in range(launches if timed else 1):
                _check(lib, lib.cwm_ceiling_mfma(ctypes.c_int(blocks), ctypes.c_int(rounds), ctypes.c_int(shape), ctypes.c_float(seed), ctypes.c_void_p(0), stream))
            if timed:
                end.record()
            torch.cuda.synchronize(device)
    flops = lib.cwm_ceiling_mfma_flops(ctypes.c_int(blocks), ctypes.c_int(rounds)) * launches
    return flops / (start.elapsed_time(end) * 1e-3) / 1e15


# --------------------------------------------------------------------------- #
# entry points that live in modules of their own; parts reach them as `ops.<name>` like the ones above
from .sequence import (  # noqa: E402
    MAX_CONV_TAPS, MAX_MEMORY_DIM, MAX_SSM_STATE, ScaledSum, add_layernorm, add_rows, cast_rows, causal_conv_silu, group_rmsnorm,
    layernorm_limits, matrix_memory, matrix_memory_state_elems, matrix_memory_state_unpack, scan_state_elems, scan_state_pack,
    scan_state_unpack, selective_scan, sigmoid_mul, step_segments, token_shift,
)
from .routed import (  # noqa: E402
    MAX_EXPERTS, MAX_ROUTE_TOP, ExpertGroups, GatedActivation, absorb_queries, combine_routed, expand_values, expert_tiles, group_by_expert,
    grouped_gate_up, grouped_linear, route_and_group, route_group_limits, route_group_pays, route_rows, route_rows_pays, route_top,
)
from .streams import (  # noqa: E402
    ACTIVATIONS, MAX_STREAMS, RoutedSum, act_rows, embedding_streams, head_norm_rope_write, qk_norm_rope_write, stream_mix_norm,
)
from .mixing import (  # noqa: E402
    MAX_GLA_DIM, MAX_SHORT_CONV_TAPS, MAX_SIDE_ADDENDS, MAX_SIDE_DIM, MAX_TALK_HEADS, gated_act_rows, gated_linear_attention, gla_state_elems,
    gla_state_unpack, short_conv, side_tiles_take, talking_attention, token_side, wkv, wkv_token,
)
from .recurrence import (  # noqa: E402
    MAX_NORMED_ADDENDS, MAX_TOKEN_MIXES, NormedSum, add_normed_rmsnorm, embedding_sinusoid, min_gru, token_mixes,
)
from .projected import (  # noqa: E402
    MAX_CONV_QK_CHANNELS, MAX_CONV_QK_TAPS, conv_qk_rope_write, latent_rows,
)
