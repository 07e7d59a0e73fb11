"""``MaxPool3d(2)`` on channels-last volumes: the down-sampling step of the U-Net's ``Down`` block.

The reference calls the stock module there (``ScaFFold/unet/unet_parts.py:165``).  This op keeps its
semantics (floor mode, ties to the first voxel of the cell, NaN wins) and its result bit for bit, but reads the
NDHWC tensor where it lies, keeps one byte per output element for the backward instead of an int64 index, and
writes the input gradient in one pass.
"""

from __future__ import annotations

import torch
import torch.nn as nn

from . import _lib

__all__ = ["max_pool3d_2x_with_skip", "max_pool3d_2x", "is_supported_pool", "FastMaxPool3d"]

_CL3D = torch.channels_last_3d


def is_supported_pool(x) -> bool:
    """Total gate: never raises."""
    try:
        return (isinstance(x, torch.Tensor) and x.dim() == 5 and x.is_cuda and x.dtype in _lib.SUPPORTED_DTYPES
                and x.shape[1] >= 1 and min(x.shape[2:]) >= 1)
    except Exception:
        return False


def _refuse(x):
    raise NotImplementedError(f"unsupported: x={tuple(getattr(x, 'shape', ()))}/{getattr(x, 'dtype', None)}")


def _pool(x, out_halo, with_skip):
    """The launch and its autograd node: ``(pooled, ...)``; the pooled tensor carries the slab it lies in, if any."""
    done = None
    if isinstance(x, torch.Tensor):
        # What a producer left on its result is never taken from there: by now the result may have been written past its version
        # counter, and the pooled tensor belongs to the stream and the capture it was made in.
        x.__dict__.pop("_sfh_pooled", None)
        done = _lib.native().max_pool(x, int(out_halo), with_skip)
    if done is None:
        _refuse(x)
    if done[1] is not None:
        done[0]._sfh_slab = (done[1], int(out_halo))
    return done


def max_pool3d_2x_with_skip(x: torch.Tensor, out_halo: int = 0, _given=None):
    """``(F.max_pool3d(x, 2), x)``: use the returned ``x`` for the skip connection and the gradients of both uses are
    combined in one kernel (same values as autograd's own addition: one fp32 sum, one rounding).  ``_given``: what the launch that
    made ``x`` has pooled, ``(pooled, slab, halo)``, a result of the same node: both gradients meet there."""
    if not is_supported_pool(x):
        _refuse(x)
    if not x.is_contiguous(memory_format=_CL3D) or _lib.under_transform():
        return max_pool3d_2x(x, out_halo), x
    if _given is not None and _given[2] == int(out_halo):
        pooled, slab, halo = _given
        if slab is not None:
            pooled._sfh_slab = (slab, halo)
        return pooled, x
    pooled, _, skip = _pool(x, out_halo, True)
    slab = getattr(x, "_sfh_slab", None)
    if slab is not None:  # the alias is the same memory: still the interior of the slab its producer wrote it into
        skip._sfh_slab = slab
    return pooled, skip


def max_pool3d_2x(x: torch.Tensor, out_halo: int = 0) -> torch.Tensor:
    """``F.max_pool3d(x, 2)`` for a 5-D GPU tensor; the result is channels-last.  ``out_halo=h`` (one sample): the result is
    the interior view of a slab with ``h`` zero depth planes on each face (``result._sfh_slab``), for ``FastConv3d.shard_halo``."""
    if _lib.under_transform() and is_supported_pool(x):
        return _lib.one_node(lambda t: _pool(t, 0, False)[0], x)
    return _pool(x, out_halo, False)[0]


def _all_equal(v, want) -> bool:
    if isinstance(v, (tuple, list)):
        return len(v) == 3 and all(int(e) == want for e in v)
    return int(v) == want


class FastMaxPool3d(nn.MaxPool3d):
    """``nn.MaxPool3d`` whose forward runs the HIP kernel. Only the configuration the U-Net uses exists:
    ``kernel_size == stride == 2``, no padding, no dilation, floor mode, no returned indices; anything else
    raises ``NotImplementedError`` at call time."""

    #: depth planes of zero halo to leave around the output for a following ``FastConv3d.shard_halo`` (0: none)
    out_halo = 0

    def _is_pool2(self) -> bool:
        stride = self.kernel_size if self.stride is None else self.stride
        return (_all_equal(self.kernel_size, 2) and _all_equal(stride, 2) and _all_equal(self.padding, 0)
                and _all_equal(self.dilation, 1) and not self.ceil_mode and not self.return_indices)

    def serves(self, input) -> bool:
        """Whether :meth:`with_skip` applies to this module and tensor."""
        return self._is_pool2() and is_supported_pool(input) and input.is_contiguous(memory_format=_CL3D)

    def with_skip(self, input, given=None):
        """``(self(input), input)`` for an input that is also used elsewhere (the U-Net's skip connection): use the
        returned pair and the two gradients of ``input`` are summed inside the pooling-gradient kernel.  ``given``: the
        ``_sfh_pooled`` of an input that nothing but the caller has seen since ``modules.conv_then_norm`` made it on this stream."""
        if not self._is_pool2():
            raise NotImplementedError("FastMaxPool3d.with_skip supports MaxPool3d(2) only")
        return max_pool3d_2x_with_skip(input, self.out_halo, given)

    def forward(self, input):
        if not self._is_pool2():
            raise NotImplementedError(
                f"FastMaxPool3d supports MaxPool3d(2) only, got kernel_size={self.kernel_size} stride={self.stride} "
                f"padding={self.padding} dilation={self.dilation} ceil_mode={self.ceil_mode} "
                f"return_indices={self.return_indices}")
        return max_pool3d_2x(input, self.out_halo)
