"""Softmax cross-entropy over f32 logits on MI355X HIP kernels.

Reference: src/ferrite/model/gpt.py:147-152 (loss_fn: f32 log_softmax, target
log-likelihood, mean) and its autodiff backward. The forward kernel
(csrc/loss.hip: ferrite_hip_cross_entropy_fwd) reads the logits once and
returns per-row loss and logsumexp; the backward kernel writes
(softmax - onehot) * dloss / N straight into the dtype the caller needs.
"""

from __future__ import annotations

import torch

from ferrite import _hip


def _check(logits, targets) -> None:
    if logits.ndim != 2 or targets.shape != logits.shape[:1]:
        raise ValueError(f"expected logits [N, V] and targets [N]; got {tuple(logits.shape)} and {tuple(targets.shape)}")
    if logits.dtype != torch.float32:
        raise ValueError("logits must be float32")
    _hip.require_gpu(logits, targets)


def cross_entropy_rows(logits: torch.Tensor, targets: torch.Tensor):
    """(loss, lse), both f32 [N], for f32 logits [N, V] and integer targets [N]."""
    _check(logits, targets)
    return _hip.native().cross_entropy_rows(logits, targets)


def cross_entropy_grad(logits, targets, lse, dloss, scale: float, dtype=torch.float32):
    """d(scale * sum(loss)) / d logits times the 0-d device tensor ``dloss``, in ``dtype``."""
    if logits.ndim != 2:
        raise ValueError(f"expected logits [N, V]; got {tuple(logits.shape)}")
    _hip.require_gpu(logits, targets, lse, dloss)
    return _hip.native().cross_entropy_grad(logits, targets, lse, dloss, scale, dtype)


def cross_entropy(logits: torch.Tensor, targets: torch.Tensor) -> torch.Tensor:
    """Mean softmax cross-entropy of f32 logits [N, V] against targets [N] (differentiable)."""
    _check(logits, targets)
    return _hip.autograd().cross_entropy(logits, targets)
