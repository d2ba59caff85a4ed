"""Blocked matmul with f32 accumulation on an MI355X MFMA kernel.

Reference: src/ferrite/kernels/matmul.py. Same public API, block-size
validation and custom VJP (dX = G Y^T, dY = X^T G through the same kernel,
matmul.py:89-107). The HIP kernel (csrc/matmul.hip: ferrite_hip_matmul) owns a
256x256 (bf16) or 128x128 (f32) output macro-tile per workgroup; ragged shapes
are zero-filled on load inside the kernel, which computes what the reference's
zero padding computes (matmul.py:59-63, :84-85). csrc/native.cpp launches them and holds the
custom VJPs.
"""

from __future__ import annotations

import torch

from ferrite import _hip, platform
from ferrite.kernels._compat import round_up, to_torch_dtype


def _pick_blocks(m: int, n: int, k: int, bm, bn, bk):
    """Block choice and ValueError of the reference (matmul.py:41-49); hints for the HIP kernel."""
    tile = platform.default_tile()
    big = 4 * tile
    bm = bm or (big if m >= big else round_up(m, platform.SUBLANES))
    bn = bn or (big if n >= big else round_up(n, platform.LANES))
    bk = bk or (big if k >= big else round_up(k, platform.LANES))
    if bm % platform.SUBLANES or bn % platform.LANES or bk % platform.LANES:
        raise ValueError(f"blocks must be multiples of ({platform.SUBLANES}, {platform.LANES}); got bm={bm} bn={bn} bk={bk}")
    return bm, bn, bk


def _mm(xs, ys, m: int, n: int, k: int, x_t: bool, y_t: bool, out_dtype):
    """out[m, n] = op(xs) @ op(ys) on the HIP kernels. xs holds x [m, k], or its transpose [k, m]
    when x_t; ys holds y [k, n], or [n, k] when y_t."""
    return _hip.native().mm(xs, ys, m, n, k, x_t, y_t, out_dtype)


def matmul(x, y, *, block_m: int | None = None, block_n: int | None = None, block_k: int | None = None, out_dtype=None):
    """``x @ y`` for 2-D ``x: [M, K]`` and ``y: [K, N]`` with f32 accumulation (matmul.py:110-126).

    Any shape is accepted; ragged edges behave as zero padding. Differentiable.
    """
    if x.ndim != 2 or y.ndim != 2 or x.shape[1] != y.shape[0]:
        raise ValueError(f"expected [M,K] @ [K,N], got {tuple(x.shape)} @ {tuple(y.shape)}")
    out_dtype = to_torch_dtype(out_dtype) if out_dtype is not None else x.dtype
    _pick_blocks(x.shape[0], y.shape[1], x.shape[1], block_m, block_n, block_k)
    _hip.require_gpu(x, y)
    return _hip.autograd().matmul(x, y, out_dtype)


def linear(x, w):
    """``x @ w`` for ``x: [..., in]`` and ``w: [in, out]`` rounded to x's dtype, as
    ``matmul(x, w.to(x.dtype))`` computes it (model/gpt.py:95-104). Differentiable; a float
    weight's gradient is not rounded."""
    if x.ndim < 1 or w.ndim != 2 or x.shape[-1] != w.shape[0]:
        raise ValueError(f"expected [..., in] @ [in, out], got {tuple(x.shape)} @ {tuple(w.shape)}")
    _hip.require_gpu(x, w)
    return _hip.autograd().linear(x, w)


def mlp_gelu(x, w1, w2):
    """``gelu(x @ w1) @ w2`` (the tanh GELU, jax.nn.gelu(approximate=True)) for bf16
    ``x: [..., d]``, ``w1: [d, f]``, ``w2: [f, e]``, differentiable. The transformer MLP of
    model/gpt.py:141, with the GELU and its derivative applied inside the matmul kernels."""
    if x.dtype != torch.bfloat16 or w1.dtype != torch.bfloat16 or w2.dtype != torch.bfloat16:
        raise ValueError("mlp_gelu takes bf16 x, w1, w2")
    return mlp_gelu_rounded(x, w1, w2)


def mlp_gelu_rounded(x, w1, w2):
    """:func:`mlp_gelu` with float32 or bf16 weights, rounded as :func:`linear` rounds its own."""
    if x.dtype != torch.bfloat16:
        raise ValueError(f"mlp_gelu takes bf16 x; got {x.dtype}")
    if w1.ndim != 2 or w2.ndim != 2 or x.shape[-1] != w1.shape[0] or w1.shape[1] != w2.shape[0]:
        raise ValueError(f"expected [..., d] @ [d, f] @ [f, e]; got {tuple(x.shape)}, {tuple(w1.shape)}, {tuple(w2.shape)}")
    _hip.require_gpu(x, w1, w2)
    if x.numel() == 0 and x.shape[-1] > 0:
        return x.new_zeros((*x.shape[:-1], w2.shape[1]))
    return _hip.autograd().mlp(x, w1, w2)


def matmul_reference(x, y, *, out_dtype=None):
    """Torch baseline with the same numerics contract (f32 accumulation), matmul.py:129-131."""
    out = torch.matmul(x.float(), y.float())
    return out.to(to_torch_dtype(out_dtype) if out_dtype is not None else x.dtype)


def matmul_flops(m: int, n: int, k: int) -> int:
    return 2 * m * n * k
