"""The minimal engine's own ops on a ROCm device: fused elementwise work (`li_add_rms_norm`,
`li_silu_mul`), the decode step's projections (`li_skinny_gemm`) and its inputs (`li_rotary_tables`,
`li_stage_decode`).

Same results as the model's torch ops (liteinfer/models/llama.py:34-48,
:101-116) up to the order of the fp32 sum of squares and the exponential's
last bit; one launch each instead of a chain of torch kernels. The kernels
read raw pointers, so every operand is checked here first: the projections
leave what they do not serve to `F.linear`, which serves or refuses it, the
others raise ValueError. The model keeps its torch ops for CPU tensors.
"""

from __future__ import annotations

import ctypes
import functools
from typing import NamedTuple

import torch
import torch.nn.functional as F

from liteinfer_amd import _native


def _rows(t: torch.Tensor, name: str) -> tuple[int, int]:
    if t.dim() < 1 or t.stride(-1) != 1:
        raise ValueError(f"{name} must have a contiguous last axis")
    flat = t.reshape(-1, t.shape[-1])
    if flat.data_ptr() != t.data_ptr() or (flat.shape[0] > 1 and t.dim() > 2 and not t.is_contiguous()):
        raise ValueError(f"{name} rows must be evenly strided")
    return flat.shape[0], (flat.stride(0) if flat.shape[0] > 1 else t.shape[-1])


def _same_device(what: str, *tensors: torch.Tensor) -> torch.device:
    device = tensors[0].device
    for t in tensors:
        if not t.is_cuda or t.device != device:
            raise ValueError(f"{what} takes tensors on one ROCm device, got {[str(t.device) for t in tensors]}")
    return device


class Partials(NamedTuple):
    """A projection as fp32 sums over runs of its K, ``[splits, rows, n]``: what an op that follows adds and rounds."""

    sums: torch.Tensor
    shape: torch.Size
    """The projection's shape, ``[..., n]``."""


# Rows of x up to which the projections may run as this library's kernels
# (LI_SKINNY_MAX_ROWS; li_skinny_gemm_plan says which); torch's GEMMs serve
# the others.
SKINNY_MAX_ROWS = 256


@functools.lru_cache(maxsize=4096)
def _splits(rows: int, n: int, k: int) -> int:
    """Runs of K one projection is cut into (0: torch's GEMM serves it)."""
    if rows > SKINNY_MAX_ROWS or n % 8 or k % 128 or not n or not k:
        return 0
    splits = ctypes.c_int()
    status = _native.load().li_skinny_gemm_plan(rows, n, k, ctypes.byref(splits))
    if status == _native.LI_EUNSUPPORTED:
        return 0
    _native.check(status, "skinny_gemm")
    return splits.value


def _skinny(x: torch.Tensor, w: torch.Tensor) -> tuple[torch.Tensor, int]:
    """x as ``[rows, k]`` and the splits of ``x @ w.T`` (0: not this kernel's, and x as it came)."""
    if (not x.is_cuda or w.device != x.device or x.dim() < 1 or w.dim() != 2 or x.shape[-1] != w.shape[1]
            or (torch.is_grad_enabled() and (x.requires_grad or w.requires_grad))):
        return x, 0
    flat = x.reshape(-1, x.shape[-1])
    if (x.dtype not in (torch.bfloat16, torch.float16) or w.dtype != x.dtype or not w.is_contiguous()
            or flat.stride(-1) != 1 or flat.stride(0) % 8 or flat.data_ptr() % 16 or w.data_ptr() % 16):
        return flat, 0
    return flat, _splits(flat.shape[0], *w.shape)


def _gemm(x: torch.Tensor, w: torch.Tensor, out: torch.Tensor | None, sums: torch.Tensor | None, splits: int,
          gate_up: bool) -> None:
    status = _native.load().li_skinny_gemm(
        x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), out.data_ptr() if out is not None else None,
        out.stride(0) if out is not None else 0, sums.data_ptr() if sums is not None else None,
        x.shape[0], w.shape[0], w.shape[1], splits, int(gate_up), _native.dtype_code(x.dtype),
        _native.stream_handle(x.device))
    _native.check(status, "skinny_gemm")


def linear_sums(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor | Partials:
    """``x @ w.T`` for an op that takes `Partials`: those where the kernel cut K, the rounded rows elsewhere."""
    flat, splits = _skinny(x, w)
    if splits == 0:
        return F.linear(x, w)
    shape = torch.Size((*x.shape[:-1], w.shape[0]))
    if splits > 1:
        sums = torch.empty(splits, flat.shape[0], w.shape[0], dtype=torch.float32, device=x.device)
        _gemm(flat, w, None, sums, splits, False)
        return Partials(sums, shape)
    out = torch.empty(flat.shape[0], w.shape[0], dtype=x.dtype, device=x.device)
    _gemm(flat, w, out, None, 1, False)
    return out.view(shape)


def linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """``x @ w.T``, the model's projection."""
    got = linear_sums(x, w)
    if not isinstance(got, Partials):
        return got
    splits, rows, n = got.sums.shape
    out = torch.empty(got.shape, dtype=x.dtype, device=x.device)
    status = _native.load().li_skinny_reduce(got.sums.data_ptr(), out.data_ptr(), n, rows, n, splits,
                                             _native.dtype_code(x.dtype), _native.stream_handle(x.device))
    _native.check(status, "skinny_reduce")
    return out


def gate_up_silu(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """``silu(gate) * up`` of the fused projection ``x @ w.T = [gate | up]``."""
    flat, splits = _skinny(x, w)
    if splits == 0 or w.shape[0] % 16:
        return silu_mul(F.linear(x, w))
    rows, ffn = flat.shape[0], w.shape[0] // 2
    out = torch.empty(*x.shape[:-1], ffn, dtype=x.dtype, device=x.device)
    if splits == 1:
        _gemm(flat, w, out.view(rows, ffn), None, 1, True)
        return out
    sums = torch.empty(splits, rows, 2 * ffn, dtype=torch.float32, device=x.device)
    _gemm(flat, w, None, sums, splits, True)
    status = _native.load().li_silu_mul_partials(sums.data_ptr(), splits, out.data_ptr(), rows, ffn, ffn,
                                                 _native.dtype_code(x.dtype), _native.stream_handle(x.device))
    _native.check(status, "silu_mul")
    return out


def add_rms_norm(h: torch.Tensor, weight: torch.Tensor, eps: float,
                 delta: torch.Tensor | Partials | None = None) -> torch.Tensor:
    """``h += delta`` in place (when given), then RMSNorm of h times `weight`; returns the normalised rows."""
    if h.dtype not in (torch.bfloat16, torch.float16) or weight.dtype != h.dtype or weight.shape != h.shape[-1:]:
        raise ValueError("add_rms_norm takes bf16 / f16 rows and a weight of their width and dtype")
    if delta is not None and (delta.shape != h.shape or (not isinstance(delta, Partials) and delta.dtype != h.dtype)):
        raise ValueError("delta must match h")
    _same_device("add_rms_norm", h, weight, *(() if delta is None else (delta.sums if isinstance(delta, Partials) else delta,)))
    rows, h_s = _rows(h, "h")
    if isinstance(delta, Partials):
        if (delta.sums.dtype != torch.float32 or delta.sums.dim() != 3 or not delta.sums.is_contiguous()
                or delta.sums.shape[1:] != (rows, h.shape[-1])):
            raise ValueError(f"partial sums must be contiguous float32 [splits, {rows}, {h.shape[-1]}], "
                             f"got {delta.sums.dtype} {list(delta.sums.shape)}")
        out = torch.empty(h.shape, dtype=h.dtype, device=h.device)
        status = _native.load().li_add_rms_norm_partials(
            h.data_ptr(), delta.sums.data_ptr(), delta.sums.shape[0], weight.contiguous().data_ptr(), out.data_ptr(),
            rows, h.shape[-1], h_s, h.shape[-1], float(eps), _native.dtype_code(h.dtype),
            _native.stream_handle(h.device))
        _native.check(status, "add_rms_norm")
        return out
    d_s = _rows(delta, "delta")[1] if delta is not None else 0
    out = torch.empty(h.shape, dtype=h.dtype, device=h.device)
    status = _native.load().li_add_rms_norm(
        h.data_ptr(), delta.data_ptr() if delta is not None else None, weight.contiguous().data_ptr(),
        out.data_ptr(), rows, h.shape[-1], h_s, d_s, h.shape[-1], float(eps), _native.dtype_code(h.dtype),
        _native.stream_handle(h.device))
    _native.check(status, "add_rms_norm")
    return out


def silu_mul(gate_up: torch.Tensor) -> torch.Tensor:
    """``silu(gate) * up`` of the fused projection's halves ``gate_up = [gate | up]``."""
    if gate_up.dtype not in (torch.bfloat16, torch.float16) or gate_up.shape[-1] % 2:
        raise ValueError("silu_mul takes bf16 / f16 rows of an even width")
    _same_device("silu_mul", gate_up)
    ffn = gate_up.shape[-1] // 2
    rows, gu_s = _rows(gate_up, "gate_up")
    out = torch.empty(*gate_up.shape[:-1], ffn, dtype=gate_up.dtype, device=gate_up.device)
    status = _native.load().li_silu_mul(gate_up.data_ptr(), out.data_ptr(), rows, ffn, gu_s, ffn,
                                        _native.dtype_code(gate_up.dtype), _native.stream_handle(gate_up.device))
    _native.check(status, "silu_mul")
    return out


def rotary_tables(positions: torch.Tensor, inv_freq: torch.Tensor, dtype: torch.dtype) -> tuple[torch.Tensor, torch.Tensor]:
    """cos / sin ``[..., D]`` of `positions` times `inv_freq` (``[D / 2]`` fp32, each twice), rounded to `dtype`."""
    _same_device("rotary_tables", positions, inv_freq)
    if positions.is_floating_point() or positions.is_complex():
        raise ValueError(f"rotary_tables takes whole positions, got {positions.dtype}")
    if inv_freq.dtype != torch.float32 or inv_freq.dim() != 1 or not inv_freq.is_contiguous():
        raise ValueError(f"inv_freq must be contiguous float32 [D / 2], got {inv_freq.dtype} {list(inv_freq.shape)}")
    positions = positions.to(torch.int64).contiguous()
    half = inv_freq.shape[0]
    cos, sin = (torch.empty(*positions.shape, 2 * half, dtype=dtype, device=positions.device) for _ in range(2))
    status = _native.load().li_rotary_tables(
        positions.data_ptr(), inv_freq.data_ptr(), cos.data_ptr(), sin.data_ptr(), positions.numel(), half,
        _native.dtype_code(dtype), _native.stream_handle(positions.device))
    _native.check(status, "rotary_tables")
    return cos, sin


def stage_decode(inputs: tuple[torch.Tensor, ...], static: tuple[torch.Tensor, ...], width: int, pad_slot: int) -> None:
    """A decode step's (ids, positions, write slots, slot table, context lengths) into a captured graph's buffers.

    `static` holds the buffers in the same order; rows past the step's, up to
    `width`, become a one-token context in `pad_slot`.
    """
    ids, positions, write_slots, slots, lens = inputs
    n, cols = slots.shape
    device = _same_device("stage_decode", *static)
    ids_out, positions_out, write_out, table_out, lens_out = static
    for t in (ids_out, positions_out, write_out, lens_out):
        if t.numel() < width or not t.is_contiguous() or t.dtype != (torch.int32 if t is lens_out else torch.int64):
            raise ValueError(f"the static columns must be contiguous int64 (lengths int32) of at least {width} rows, "
                             f"got {t.dtype} {list(t.shape)}")
    if (table_out.dtype != torch.int64 or table_out.dim() != 2 or table_out.stride(1) != 1 or n > width
            or width > table_out.shape[0] or max(cols, 1) > table_out.shape[1] or table_out.stride(0) < table_out.shape[1]):
        raise ValueError(f"a step of {n} x {cols} slots, padded to {width} rows, does not fit a "
                         f"{list(table_out.shape)} {table_out.dtype} slot table")

    def column(t: torch.Tensor, shape: tuple[int, ...], dtype: torch.dtype) -> torch.Tensor:
        if t.shape == shape and t.dtype == dtype and t.device == device and t.is_contiguous():
            return t  # (as the engine brings it: 0.6 us on the host, the conversions that change nothing 3)
        return torch.broadcast_to(t, shape).to(device=device, dtype=dtype).contiguous()

    ids, positions = column(ids, (n, 1), torch.int64), column(positions, (n, 1), torch.int64)
    write_slots, lens = column(write_slots, (1, n), torch.int64), column(lens, (n,), torch.int32)
    slots = slots.to(device=device, dtype=torch.int64)
    if slots.stride(-1) != 1:
        slots = slots.contiguous()
    status = _native.load().li_stage_decode(
        ids.data_ptr(), positions.data_ptr(), write_slots.data_ptr(), slots.data_ptr(), slots.stride(0), lens.data_ptr(),
        ids_out.data_ptr(), positions_out.data_ptr(), write_out.data_ptr(), table_out.data_ptr(), table_out.stride(0),
        lens_out.data_ptr(), n, cols, width, pad_slot, _native.stream_handle(device))
    _native.check(status, "stage_decode")
