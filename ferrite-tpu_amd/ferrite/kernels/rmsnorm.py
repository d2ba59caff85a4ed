"""Fused residual-add + RMSNorm on an MI355X HIP kernel, with a custom VJP.

Reference: src/ferrite/kernels/rmsnorm.py. Same public API and ValueErrors.
The forward is one HIP kernel (csrc/rmsnorm.hip: ferrite_hip_add_rmsnorm /
ferrite_hip_rmsnorm) that reads x and residual once, writes h and y once and
keeps the statistics in f32. The backward (rmsnorm.py:159-166, an XLA fusion in
the reference) is a HIP kernel too (ferrite_hip_rmsnorm_bwd): one pass over h,
dy and the fused add's direct gradient that writes dh, plus a fixed-order
reduction of dweight. Both are launched by csrc/native.cpp, the custom VJP's host side.
"""

from __future__ import annotations

import torch

from ferrite import _hip, platform
from ferrite.kernels._compat import round_up

_TARGET_BLOCK_BYTES = 4 << 20


def _rows_block(n_rows: int, dim: int, block_rows: int | None) -> int:
    """Row block of the reference (rmsnorm.py:67-74): validated identically, used only as a hint."""
    if block_rows is None:
        fit = max(platform.SUBLANES, _TARGET_BLOCK_BYTES // (dim * 20))
        fit = 1 << (fit.bit_length() - 1)
        block_rows = min(256, fit, round_up(n_rows, platform.SUBLANES))
    if block_rows % platform.SUBLANES:
        raise ValueError(f"block_rows must be a multiple of {platform.SUBLANES}")
    return block_rows


def rmsnorm(x, weight, *, residual=None, eps: float = 1e-6, block_rows: int | None = None):
    """RMSNorm over the last axis of ``x`` (rmsnorm.py:174-190).

    With ``residual`` given, returns ``(h, y)`` where ``h = x + residual`` is the
    new residual stream and ``y = rmsnorm(h) * weight``; otherwise returns ``y``.
    """
    dim = x.shape[-1]
    if tuple(weight.shape) != (dim,):
        raise ValueError(f"weight must have shape ({dim},), got {tuple(weight.shape)}")
    if residual is not None and residual.shape != x.shape:
        raise ValueError("residual must match x")
    if dim == 0:
        raise RuntimeError("rmsnorm needs a non-empty last dimension")
    _rows_block(x.numel() // dim, round_up(dim, platform.LANES), block_rows)
    if residual is None:
        _hip.require_gpu(x, weight)
    else:
        _hip.require_gpu(x, residual, weight)
    if residual is None:
        return _hip.autograd().rmsnorm(x, weight, float(eps))
    return _hip.autograd().add_rmsnorm(x, residual, weight, float(eps))


def rmsnorm_reference(x, weight, *, residual=None, eps: float = 1e-6):
    """Plain torch math with identical f32 numerics (the reference's XLA route, rmsnorm.py:193-199)."""
    h = x.float() + (0 if residual is None else residual.float())
    y = h * torch.rsqrt(torch.mean(h * h, dim=-1, keepdim=True) + eps) * weight.float()
    if residual is None:
        return y.to(x.dtype)
    return h.to(x.dtype), y.to(x.dtype)
