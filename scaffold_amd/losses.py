"""Fused loss head of the U-Net train step: fp32 log-softmax, cross entropy and soft Dice in one pass.

Mirrors the loss block of the reference's trainer (``ScaFFold/utils/trainer.py:634-663``): the logits are
upcast to fp32 once, ``CE = sum_v w[y_v] * -log p_v[y_v] / normaliser`` (``ScaFFold/utils/losses.py:119-214``;
the normaliser is the voxel count, or ``sum_v w[y_v]`` with class weights), the Dice score of every (sample, class)
is ``(2 I + eps) / (P + T + eps)`` over the softmax probabilities (``ScaFFold/utils/dice_score.py:101-136``), and the
loss is ``CE + 1 - mean foreground Dice`` (``trainer.py:331-333,660-663``).  One HIP kernel pass produces all
sums (fixed-order reductions, no atomics), a second one the gradient; nothing of size ``N*C*D*H*W`` is
materialised in fp32.
"""

from __future__ import annotations

from typing import Optional

import torch

from . import _lib

__all__ = ["ce_dice_loss", "is_supported_loss"]


def is_supported_loss(logits, labels, class_weight=None) -> bool:
    """Total gate: never raises."""
    try:
        if not isinstance(logits, torch.Tensor) or not isinstance(labels, torch.Tensor):
            return False
        if logits.dim() != 5 or labels.dim() != 4 or not logits.is_cuda or labels.device != logits.device:
            return False
        if logits.dtype not in _lib.SUPPORTED_DTYPES or labels.dtype is not torch.int64:
            return False
        n, c, d, h, w = logits.shape
        if tuple(labels.shape) != (n, d, h, w) or not 2 <= c <= 32 or n < 1 or d * h * w < 1:
            return False
        if class_weight is not None:
            if not isinstance(class_weight, torch.Tensor) or class_weight.device != logits.device \
                    or tuple(class_weight.shape) != (c,) or not class_weight.dtype.is_floating_point:
                return False
        return True
    except Exception:
        return False


def ce_dice_loss(logits: torch.Tensor, labels: torch.Tensor, class_weight: Optional[torch.Tensor] = None,
                 eps: float = 1e-6) -> torch.Tensor:
    """``CE(logits, labels[, class_weight]) + 1 - mean foreground soft Dice`` as a 0-dim fp32 tensor.

    ``logits``: ``(N, C, D, H, W)`` bf16 / fp16 / fp32 on the GPU (any memory format; channels-last is read in
    place); ``labels``: ``(N, D, H, W)`` int64 class ids, ids outside ``[0, C)`` contribute nothing."""
    loss = None
    if isinstance(logits, torch.Tensor) and isinstance(labels, torch.Tensor) and (class_weight is None or isinstance(class_weight, torch.Tensor)):
        if _lib.under_transform() and is_supported_loss(logits, labels, class_weight):
            return _lib.one_node(lambda *ts: _lib.native().ce_dice_loss(*ts, float(eps)), logits, labels,
                                 None if class_weight is None else class_weight.detach())
        loss = _lib.native().ce_dice_loss(logits, labels, class_weight, float(eps))
    if loss is None:
        raise NotImplementedError(
            f"unsupported: logits={tuple(getattr(logits, 'shape', ()))}/{getattr(logits, 'dtype', None)} "
            f"labels={tuple(getattr(labels, 'shape', ()))}/{getattr(labels, 'dtype', None)}")
    return loss
