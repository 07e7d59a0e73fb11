"""Drop-in ``nn.Module``s over the HIP ops: ``FastConv3d``, ``FastConvTranspose3d``, ``FastGroupNorm``.

They stand where the reference's adapters stand (``ScaFFold/unet/conv3d.py:1235-1479,1790-1904``,
``ScaFFold/unet/group_norm.py:556-808``) and keep their contract:

* same parameters under the same names and no buffers, so ``state_dict`` keys and shapes are
  those of ``nn.Conv3d`` / ``nn.ConvTranspose3d`` / ``nn.GroupNorm`` in both directions;
* under ``torch.autocast`` only exactly-fp32 operands are cast, and the cast is an ordinary
  autograd node *outside* the kernel's node, so an fp32 parameter receives an fp32 gradient
  (``conv3d.py:446-480``);
* the autograd nodes save ``(x, weight)`` after the launch, compute the bias gradient as
  ``grad_output.sum((0, 2, 3, 4))`` (``conv3d.py:1231``) and are once-differentiable: a second
  differentiation raises instead of returning zeros;
* ``FastGroupNorm`` returns its input's dtype (not fp32) inside autocast and applies the ReLU
  when ``activation="relu"``.

What is deliberately absent: the reference's fallback ladder (Triton -> MIOpen, compiled ->
eager), its latches, the hardware allowlist and the mesh-wide vote.  There is one backend here;
a call it does not serve raises ``NotImplementedError``.

``FastConv3d.shard_halo`` reproduces the compute shape of one DistConv depth shard on a single
GPU: the input is extended by one voxel of (zero) halo on each depth face and the convolution
runs with depth padding 0, which is what the reference's own halo exchange hands its kernel
(``conv3d.py:648-677,748-792``); with no neighbour the halo is zero and the result equals the
ordinary padded convolution.
"""

from __future__ import annotations

import math
import threading
from typing import Optional

import torch
import torch.nn as nn

from . import _lib
from . import conv3d as _c3
from . import groupnorm as _gn
from . import halo as _halo

__all__ = ["FastConv3d", "FastConvTranspose3d", "FastGroupNorm", "autocast_dtype", "cast_operand", "compute_copy",
           "flush_weight_gradients"]

_CL3D = torch.channels_last_3d

#: pack each convolution weight once per step for forward and data gradient also outside graph capture
PACK_WEIGHTS_ONCE = False


def autocast_dtype(tensor: torch.Tensor) -> Optional[torch.dtype]:
    """The dtype autocast would cast a convolution's operands to on this device, or ``None``."""
    try:
        if not torch.is_autocast_enabled(tensor.device.type):
            return None
        return torch.get_autocast_dtype(tensor.device.type)
    except (RuntimeError, TypeError):
        return None


def cast_operand(tensor: Optional[torch.Tensor], dtype: Optional[torch.dtype]):
    """ATen's ``cached_cast`` rule: only an exactly-fp32 tensor is narrowed."""
    if tensor is None or dtype is None or tensor.dtype is not torch.float32:
        return tensor
    return tensor.to(dtype)


def compute_copy(param: Optional[torch.Tensor], dtype: Optional[torch.dtype]):
    """A current half-precision copy of an fp32 parameter kept by the optimizer (``FusedClipAdam(shadow_dtype=...)``
    refreshes it inside its update kernel), or ``None``.  It is used only while the parameter has not been written
    by anything else since the copy was made (torch's version counter), so a stale copy is never read."""
    if param is None or dtype is None or param.dtype is not torch.float32:
        return None
    copy = getattr(param, "_sfh_shadow", None)
    if copy is None or copy.dtype is not dtype or getattr(param, "_sfh_shadow_version", None) != param._version:
        return None
    return copy


def _current_packs(owner: torch.Tensor, source: torch.Tensor, in_shape, stride, padding, dilation):
    """The packed forms of a parameter's weight for this problem, or ``None`` when the problem reads no packed weight (or the
    weight is not on a GPU: the caller's gate comes after this and refuses).

    They are kept on the parameter (``owner._sfh_packs``) and trusted without a launch only under the rule that also
    guards the optimizer's half-precision copies: the optimizer that writes the parameter refreshes them inside its
    step (``maintained``) and nothing else has written the parameter since (torch's version counter).  Otherwise they
    are packed again here, in one launch for both directions."""
    if source.dtype is torch.float32 or not source.is_cuda:
        return None
    table = owner.__dict__.get("_sfh_packs")
    if table is None:
        table = owner._sfh_packs = {}
    key = (in_shape, padding)
    e = table.get(key)
    if e is None:
        if len(table) >= 8:  # a parameter meets few problems; shapes that keep changing are not worth the buffers
            table.clear()
        e = table[key] = _c3.PackedWeights(source, in_shape, stride, padding, dilation)
        e.version = owner._version
        return e if e else None
    if not e:
        return None
    if not (e.maintained and e.version == owner._version and e.source is source):
        e.repack(source)
        e.version = owner._version
    return e


# ---- weight gradients of a backward pass in one launch -----------------------------------------------------------------
# Nothing reads a weight gradient before the optimizer (``ScaFFold/utils/trainer.py:678-694``), and a launch of the
# weight-gradient kernel costs 15-20 us whatever the problem.  A convolution whose module has ``defer_weight_grad`` set
# therefore does not compute its weight gradient in its own backward node: the node leaves (parameter, operands) in the
# pass's queue (``csrc/host/native.cpp``) and returns no gradient for the weight, and a callback the autograd engine runs
# when the backward pass has finished -- still inside ``backward()`` -- computes all queued gradients in one batched call and
# adds them to the parameters' ``.grad``.  After ``backward()`` returns the gradients are where they always are.  What
# differs: hooks on the parameter's gradient accumulation do not see these gradients, and the operands stay alive until
# the end of the pass.  A pass that raises drops what it has queued.
_BATCHABLE: dict = {}

#: A weight gradient of more operations than this is computed in its own node although the module defers.  What a place
#: in the batch saves is a launch and a slice sum (20 us), a tenth of such a problem's time; what it costs is that the
#: operands have left the caches when the pass ends, and in early mode that half of the device works on it while the other
#: half runs out of work.  Measured on captured steps (ms; everything deferred early / this rule): base width 64 on 128^3
#: (problems of 464 and 928 GFLOP) 16.02 / 14.62, on 64 x 128 x 128 8.76 / 8.39, two samples of 64 x 70 x 75 6.52 / 6.29;
#: base width 32 on 128^3 (its largest problem has 232 GFLOP) 4.96 deferred against 4.98 with a limit of 125 and 5.05 of 60.
_DEFER_MAX_FLOPS = 250e9


def _deferrable(param, in_shape, wshape, stride, padding, dilation, dtype) -> int:
    """Whether a weight gradient can wait for the end of the pass: the parameter is a leaf that takes a ``.grad``, the
    library batches the problem and it is not too large to gain from that.  0, or the launch of the batch that takes it
    (``conv3d.weight_grad_batch_family``)."""
    if param is None or not param.is_leaf or not param.requires_grad:
        return 0
    key = (in_shape, wshape, stride, padding, dilation, dtype)
    ok = _BATCHABLE.get(key)
    if ok is None:
        ok = _c3.weight_grad_batch_family(in_shape, wshape, stride, padding, dilation, dtype)
        if ok:
            n, cout, *out = _c3.output_shape(in_shape, wshape, stride, padding, dilation)
            if 2.0 * n * math.prod(out) * cout * math.prod(wshape[1:]) > _DEFER_MAX_FLOPS:
                ok = 0
        if len(_BATCHABLE) > 256:
            _BATCHABLE.clear()
        _BATCHABLE[key] = ok
    return ok


_EARLY_LOCK = threading.Lock()
_EARLY_STREAMS: dict = {}  # (device, a pass's stream) -> the side stream beside it
_EARLY_DONE: set = set()  # batches sent and not joined yet: what keeps their operands alive


def _early_stream(main):
    """The side stream of passes on ``main``.  Each has its own: a pass that is being captured takes its side stream into the
    capture, and what a pass on another stream sent there meanwhile would become part of that graph."""
    with _EARLY_LOCK:
        key = (main.device, main.cuda_stream)
        side = _EARLY_STREAMS.get(key)
        if side is None:
            if len(_EARLY_STREAMS) >= 16:  # half of the streams torch hands out in turn
                _EARLY_STREAMS.clear()
            taken = [main, *_EARLY_STREAMS.values()]
            while side is None or side in taken:
                side = torch.cuda.Stream(device=main.device)
            _EARLY_STREAMS[key] = side
        return side


def _send_early(batch) -> None:
    # Operands and gradients are memory of the pass's stream: the side stream starts behind that stream, and they stay
    # referenced until that stream has been made to wait for the batch (in _join_early, or here if a launch is refused), so
    # the caching allocator hands none of it out while the batch runs.
    main = torch.cuda.current_stream(_lib.native().batch_device(batch))
    side = _early_stream(main)
    _lib.native().launch_beside(batch, side.stream_id, side.device_index)
    _EARLY_DONE.add(batch)


def _join_early(batch) -> None:
    _EARLY_DONE.remove(batch)
    _lib.native().join_beside(batch)


def flush_weight_gradients() -> None:
    """Compute the weight gradients that the backward pass this is called from (by a hook, say) has queued so far and add them
    to their parameters' ``.grad``.  A pass that ends does this by itself, and one that raises drops what it has queued:
    outside of a pass nothing waits."""
    _lib.native().finish_current_pass()


_early_callbacks_set = False


def _set_early_callbacks() -> None:
    global _early_callbacks_set
    if not _early_callbacks_set:
        # (looked up in the module at the time of the call)
        _lib.native().set_early_callbacks(lambda batch: _send_early(batch), lambda batch: _join_early(batch))
        _early_callbacks_set = True


def _narrowed(weight, bias, dt, x_dtype) -> bool:
    """Whether autocast narrows these parameters to the 16-bit dtype of the activations."""
    return dt in (torch.bfloat16, torch.float16) and x_dtype is dt and weight.dtype is torch.float32 and weight.is_cuda \
        and not _lib.under_transform() and (bias is None or bias.dtype is torch.float32 or bias.dtype is dt)


def _master_operands(weight, bias, dt, in_shape, stride, padding, dilation, want_dgrad):
    """What the kernels read of fp32 parameters under 16-bit autocast when nobody keeps half-precision copies:
    ``(w, b, (packed_fwd, packed_dgrad), complete)``.  The packed forms come from the master in one launch, rounded on the
    way; only a direction that reads the weight where it lies (the stem, the 1x1x1 head) needs a cast of it.  The parameters'
    gradients are then produced in fp32 directly: no cast nodes either way."""
    pf, pd, complete = _lib.native().pack_master(weight, dt, in_shape, stride, padding, dilation, want_dgrad)
    w = weight if complete else weight.detach().to(dt)
    b = None if bias is None else (bias if bias.dtype is dt else bias.detach().to(dt))
    return w, b, (pf, pd), complete


def _run_conv(x, second, x_read, second_read, weight, bias, w, b, packs, halo, stride, padding, dilation, master, gn_groups, defer):
    """The forward launch of a convolution and its autograd node.  ``x`` / ``second`` are the tensors that receive gradients,
    ``x_read`` / ``second_read`` what the kernels read (slabs of which x and second are the depth interiors when ``halo`` > 0,
    else the same tensors).  ``weight`` / ``bias`` receive gradients, ``w`` / ``b`` are what the kernels read: when half-precision
    copies of fp32 masters are given (``master``) the gradients are produced in the masters' dtype directly.  The caller has
    passed the gate (for all three directions when the call will be differentiated)."""
    if _lib.under_transform():
        # (the packed forms and half-precision copies belong to the parameters, not to what a replay is given)
        return _lib.one_node(
            lambda x_, w_, b_, x2_, r_, r2_: _run_conv_here(x_, x2_, x_ if x_read is x else r_, x2_ if second_read is second else r2_, w_, b_,
                                                            w_ if w is weight else w, b_ if b is bias else b, None, halo, stride, padding,
                                                            dilation, master, 0, False),
            x, weight, bias, second, None if x_read is x else x_read.detach(), None if second_read is second else second_read.detach())
    return _run_conv_here(x, second, x_read, second_read, weight, bias, w, b, packs, halo, stride, padding, dilation, master, gn_groups, defer)


def _run_conv_here(x, second, x_read, second_read, weight, bias, w, b, packs, halo, stride, padding, dilation, master, gn_groups, defer):
    pf = pd = None
    in_shape = x_read.shape if second is None else torch.Size((x_read.shape[0], x_read.shape[1] + second_read.shape[1], *x_read.shape[2:]))
    if packs is not None:
        pf, pd = packs
    elif torch.is_grad_enabled() and x.requires_grad and (PACK_WEIGHTS_ONCE or torch.cuda.is_current_stream_capturing()):
        # When the data gradient will be wanted too, the weight can be packed for both directions in one launch.
        # That saves a launch per convolution on the GPU and costs a little more host time, so it is done where
        # host time is free (under graph capture) or when asked for (PACK_WEIGHTS_ONCE).
        pf, pd = _c3.pack_weights(w, in_shape, stride, padding, dilation)
    # gn_groups: a GroupNorm of that many groups follows; the launch leaves its statistics on y where it can
    if x_read.shape[0] > 1 and in_shape[1] == 32:
        gn_groups = 0  # (module_groups in native.cpp: a batch's statistics stay with the pass that reads it)
    if second is None:
        y = _c3.conv3d_forward(x_read, w, b, stride, padding, dilation, 1, packed_weight=pf, gn_groups=gn_groups, _checked=True)
    else:
        y = _c3.conv3d_forward_pair(x_read, second_read, w, b, stride, padding, dilation, packed_weight=pf, gn_groups=gn_groups,
                                    _checked=True)
    if _wants_grad(x, second, weight, bias):
        family = 0
        if defer:
            _set_early_callbacks()
            family = _deferrable(weight, in_shape, w.shape, stride, padding, dilation, x_read.dtype)
        _lib.native().record_conv(y, x, weight, bias, second, x_read, second_read, w, pd, halo, stride, padding, dilation, master, family,
                           defer == 2)
    return y


def _wants_grad(*tensors) -> bool:
    return torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in tensors)


class FastConv3d(nn.Conv3d):
    """``nn.Conv3d`` served by the HIP kernels.  ``__init__`` is inherited unchanged."""

    #: emulate one depth shard: zero halo on both depth faces + depth padding 0
    shard_halo = False
    #: groups of a GroupNorm that reads this module's output next (0: none): the forward launch then also leaves that
    #: GroupNorm's statistics on its result, where the kernel offers it, and the normalisation skips its statistics pass
    gn_groups = 0
    #: leave this module's weight gradient to the end of the backward pass, where all such gradients come from one launch
    #: (see flush_weight_gradients); taken up only where the weight is the parameter itself and the library batches the shape.
    #: 2 instead of True: besides, the large-row gradients queued when the pass reaches its first small volume are computed
    #: there and then on a stream of their own, on half of the device, beside the rest of the pass
    defer_weight_grad = False

    def _pair_operands(self, x, second):
        """The tensors the kernels would read for ``forward(x, second)`` and the padding they would run with, or ``None``
        when the pair is not served as it stands: ``(x_read, second_read, padding, slab, slab2)``.  In the depth-shard
        form both tensors must already lie in slabs with zero faces (their producers wrote them there)."""
        if self.padding_mode != "zeros" or isinstance(self.padding, str) or self.groups != 1:
            return None
        if not isinstance(x, torch.Tensor) or not isinstance(second, torch.Tensor) or x.dtype is not second.dtype:
            return None
        dt = autocast_dtype(x)
        if dt is not None and x.dtype is torch.float32:
            return None  # the casts would make new tensors (outside the slabs); the caller concatenates instead
        if (dt if (dt is not None and self.weight.dtype is torch.float32) else self.weight.dtype) is not x.dtype:
            return None  # the weight the kernel would read (autocast narrows an fp32 parameter) is of another dtype
        padding = tuple(self.padding)
        slab = slab2 = None
        if self.shard_halo and padding[0] > 0:
            slab, slab2 = getattr(x, "_sfh_slab", None), getattr(second, "_sfh_slab", None)
            if slab is None or slab2 is None or slab[1] != padding[0] or slab2[1] != padding[0]:
                return None
            if slab[0].dtype is not x.dtype or slab2[0].dtype is not x.dtype:
                return None
            x_read, second_read = slab[0], slab2[0]
            padding = (0, padding[1], padding[2])
        else:
            x_read, second_read = x, second
        if not (x_read.is_contiguous(memory_format=_CL3D) and second_read.is_contiguous(memory_format=_CL3D)):
            return None
        return x_read, second_read, padding, slab, slab2

    def takes_pair(self, x, second) -> bool:
        """Whether ``forward(x, second)`` is served: the convolution of ``torch.cat([x, second], 1)`` read from the two
        tensors themselves, all three directions.  Total: never raises."""
        try:
            ops = self._pair_operands(x, second)
            return ops is not None and self._pair_gate(ops[0], ops[1], ops[2])
        except (TypeError, ValueError, AttributeError, RuntimeError):
            return False

    def _pair_gate(self, x_read, second_read, padding) -> bool:
        """The library's answer for the tensors the kernels would read, remembered per shape (the parameters' shapes and
        the module's geometry do not change; their dtypes under autocast are the activations')."""
        key = (x_read.shape, second_read.shape, x_read.dtype, x_read.device, padding, self.bias is None)
        table = self.__dict__.get("_pair_ok")
        if table is None:
            table = self.__dict__["_pair_ok"] = {}
        ok = table.get(key)
        if ok is None:
            # stand-ins with the dtype the kernel's operands will have (metadata only)
            w = self.weight if self.weight.dtype is x_read.dtype else self.weight.new_empty((1, 1, 1, 1, 1), dtype=x_read.dtype).expand(
                self.weight.shape)
            b = None
            if self.bias is not None:
                b = self.bias if self.bias.dtype is x_read.dtype else torch.empty(self.bias.shape, dtype=x_read.dtype, device=x_read.device)
            ok = _c3.is_supported_pair(x_read, second_read, w, b, tuple(self.stride), padding, tuple(self.dilation))
            if len(table) > 64:
                table.clear()
            table[key] = ok
        return ok

    def _kernel_operands(self, weight, bias, dt, x_dtype, in_shape, stride, padding, dilation, want_dgrad):
        """``(w, b, packs, master, complete)``: what the kernels read of the parameters (``packs``: the packed forms that are
        current, or None), whether the parameters are fp32 masters whose gradients are produced in fp32 directly, and whether
        the packed forms are all that is read (``w`` is then the master itself).  The caller has not passed its gate yet: a
        weight that does not belong to an input of this shape is not packed (packing walks the input's channels)."""
        if len(in_shape) != 5 or in_shape[1] != weight.shape[1] or self.groups != 1:
            return cast_operand(weight, dt), cast_operand(bias, dt), None, False, False
        # under autocast, up-to-date half-precision copies kept by the optimizer, with their packed forms
        wc = compute_copy(weight, dt)
        if wc is not None:
            bc = compute_copy(bias, dt)
            if bias is None or bc is not None:
                packs = _current_packs(weight, wc, in_shape, stride, padding, dilation)
                return wc, bc, None if packs is None else (packs.fwd, packs.dgrad), True, False
        if _narrowed(weight, bias, dt, x_dtype):
            w, b, packs, complete = _master_operands(weight, bias, dt, in_shape, stride, padding, dilation, want_dgrad)
            return w, b, packs, True, complete
        w, b = cast_operand(weight, dt), cast_operand(bias, dt)
        packs = _current_packs(w, w, in_shape, stride, padding, dilation) if w is weight else None
        return w, b, None if packs is None else (packs.fwd, packs.dgrad), False, False

    def _forward_pair(self, x, second):
        ops = self._pair_operands(x, second)
        if ops is None:
            raise NotImplementedError(f"FastConv3d: the pair x={tuple(x.shape)}/{x.dtype}, second={tuple(second.shape)}/{second.dtype} "
                                      "is not served as it stands (see takes_pair); concatenate instead")
        x_read, second_read, padding, slab, slab2 = ops
        dt = autocast_dtype(x)
        weight, bias = self.weight, self.bias  # (each lookup of a parameter is a call into Module.__getattr__)
        stride, dilation = tuple(self.stride), tuple(self.dilation)
        in_shape = torch.Size((x_read.shape[0], x_read.shape[1] + second_read.shape[1], *x_read.shape[2:]))
        want_dgrad = torch.is_grad_enabled() and (x.requires_grad or second.requires_grad)
        w, b, packs, master, complete = self._kernel_operands(weight, bias, dt, x_read.dtype, in_shape, stride, padding, dilation, want_dgrad)
        if not (complete or w.dtype is x_read.dtype) or not self._pair_gate(x_read, second_read, padding):
            raise NotImplementedError(
                f"FastConv3d: pair not served: x={tuple(x_read.shape)}/{x_read.dtype} second={tuple(second_read.shape)} on {x.device}, "
                f"weight={tuple(w.shape)}/{w.dtype}, stride={stride} padding={padding} dilation={dilation}")
        halo = 0 if slab is None else slab[1]
        return _run_conv(x, second, x_read, second_read, weight if master else w, bias if master else b, w, b, packs, halo, stride, padding,
                         dilation, master, self.gn_groups, self.defer_weight_grad if master or w is weight else False)

    def forward(self, x: torch.Tensor, second: Optional[torch.Tensor] = None) -> torch.Tensor:
        """``second``: the input is ``torch.cat([x, second], 1)``, read from the two tensors themselves (the decoder's skip
        connection and upsampled tensor, ``ScaFFold/unet/unet_parts.py:107-120``); ask :meth:`takes_pair` first."""
        if second is not None:
            return self._forward_pair(x, second)
        if self.padding_mode != "zeros" or isinstance(self.padding, str):
            raise NotImplementedError(f"FastConv3d: padding_mode={self.padding_mode!r} padding={self.padding!r}")
        dt = autocast_dtype(x)
        x = cast_operand(x, dt)
        weight, bias = self.weight, self.bias  # (each lookup of a parameter is a call into Module.__getattr__)
        padding = tuple(self.padding)
        inner, slab = x, None
        if self.shard_halo and padding[0] > 0:
            # (N, C, D, H, W): extend D by the halo the neighbours would have sent (none here: zeros). A producer that
            # already wrote x into the interior of such a slab (zero faces) has left it on the tensor.
            slab = getattr(x, "_sfh_slab", None)
            if slab is not None and slab[1] == padding[0] and slab[0].dtype is x.dtype:
                x = slab[0]
            else:
                slab = None
                x = inner = _halo.halo_assemble(x, None, None, int(padding[0]))
            padding = (0, padding[1], padding[2])
        x = x.contiguous(memory_format=_CL3D)
        # the node below skips its own gates on the strength of this one (a call that will be differentiated is
        # gated for all three directions here)
        wants = _wants_grad(inner, weight, bias)
        stride, dilation = tuple(self.stride), tuple(self.dilation)
        w, b, packs, master, complete = self._kernel_operands(weight, bias, dt, x.dtype, x.shape, stride, padding, dilation,
                                                              wants and inner.requires_grad)
        if self.groups != 1 or not (_lib.native().conv_supported(x, w, b, stride, padding, dilation, wants, complete) or
                                    (_c3.is_supported_all if wants else _c3.is_supported)(x, w, b, stride, padding, dilation, 1)):
            raise NotImplementedError(
                f"FastConv3d: not served: x={tuple(x.shape)}/{x.dtype} on {x.device}, weight={tuple(w.shape)}/{w.dtype}, "
                f"stride={self.stride} padding={padding} dilation={self.dilation} groups={self.groups}"
            )
        if slab is None:
            inner = x
        halo = 0 if slab is None else slab[1]
        return _run_conv(inner, None, x, None, weight if master else w, bias if master else b, w, b, packs, halo, stride, padding, dilation,
                         master, self.gn_groups, self.defer_weight_grad if master or w is weight else False)


def _plain_call(module) -> bool:
    """Whether calling the module is its class's ``forward`` and nothing else: no hooks, no ``forward`` or compiled call of its own."""
    return not (module._forward_hooks or module._forward_pre_hooks or module._backward_hooks or module._backward_pre_hooks
                or "forward" in module.__dict__ or module._compiled_call_impl is not None)


def conv_then_norm(conv, norm, x, pools=True):
    """``norm(conv(x))`` as one call into the host path and one autograd node, or ``None`` where the two modules have to run
    by themselves (a bias, hooks on either or a ``forward`` of its own, a subclass, an input that is not channels-last, ...).

    ``pools``: where ``norm.pool_next`` announces a pooling, the result also carries what that pooling would compute, as
    ``result._sfh_pooled``, for a caller that hands it to ``FastMaxPool3d.with_skip`` before anything else sees the result."""
    if type(conv) is not FastConv3d or type(norm) is not FastGroupNorm or conv.groups != 1 or torch.compiler.is_compiling() \
            or conv.padding_mode != "zeros" or isinstance(conv.padding, str) or not _plain_call(conv) or not _plain_call(norm) \
            or torch.nn.modules.module._has_any_global_hook() or _lib.under_transform() or not isinstance(x, torch.Tensor) or x.dim() != 5:
        return None
    weight, gamma, beta = conv.weight, norm.weight, norm.bias
    if conv.bias is not None or gamma is None or beta is None:
        return None
    dt = autocast_dtype(x)
    x = cast_operand(x, dt)
    padding, stride, dilation = tuple(conv.padding), tuple(conv.stride), tuple(conv.dilation)
    x_read, halo = x, 0
    if conv.shard_halo and padding[0] > 0:
        slab = getattr(x, "_sfh_slab", None)
        if slab is None or slab[1] != padding[0] or slab[0].dtype is not x.dtype:
            return None
        x_read, halo = slab
        padding = (0, padding[1], padding[2])
    if not x_read.is_contiguous(memory_format=_CL3D):
        return None
    in_shape = x_read.shape
    grad = torch.is_grad_enabled()
    w, _, packs, master, _ = conv._kernel_operands(weight, None, dt, x.dtype, in_shape, stride, padding, dilation, grad and x.requires_grad)
    if packs is None and torch.cuda.is_current_stream_capturing():
        return None  # the module packs for both directions at once under capture
    receives = weight if master else w
    family, defer = 0, conv.defer_weight_grad
    if defer and grad and receives is weight:
        family = _deferrable(weight, in_shape, weight.shape, stride, padding, dilation, x_read.dtype)
        _set_early_callbacks()
    pf, pd = (None, None) if packs is None else packs
    pool_halo = norm.pool_next if pools and norm.pool_next is not None and not torch.is_inference_mode_enabled() else -1
    done = _lib.native().conv_norm(x, x_read, receives, w, pf, pd, halo, stride, padding, dilation, master, family, defer == 2, norm.num_groups,
                                   gamma, beta, norm.eps, norm.activation == "relu", norm.out_halo, pool_halo)
    if done is None:
        return None
    y, slab, pooled = done
    if slab is not None:
        y._sfh_slab = (slab, norm.out_halo)
    if pooled is not None:
        y._sfh_pooled = (*pooled, pool_halo)
    return y


class FastConvTranspose3d(nn.ConvTranspose3d):
    """``nn.ConvTranspose3d`` at ``kernel == stride`` served by the HIP kernels."""

    #: depth planes of zero halo to leave around the output for a following ``FastConv3d.shard_halo`` (0: none)
    out_halo = 0

    def _served(self, done, x, w):
        if done is None:
            raise NotImplementedError(
                f"FastConvTranspose3d: not served: x={tuple(x.shape)}/{x.dtype} on {x.device}, weight={tuple(w.shape)}, "
                f"stride={self.stride} padding={self.padding} output_padding={self.output_padding} "
                f"dilation={self.dilation} groups={self.groups}"
            )
        return done

    def forward(self, x: torch.Tensor, output_size=None) -> torch.Tensor:
        if output_size is not None:
            raise NotImplementedError("FastConvTranspose3d: output_size is not supported")
        return self._upsample(x, None)

    def padded_to(self, x: torch.Tensor, extents):
        """``F.pad(self(x), ...)`` with zeros at the end of the axes that are a voxel short of ``extents``, written by the same launch
        (and left out of the gradients by theirs), or ``None`` where that is not what ``extents`` asks for or the module has to
        run by itself (hooks or a ``forward`` of its own, a subclass, a transform, a problem off the matrix cores)."""
        if type(self) is not FastConvTranspose3d or torch.compiler.is_compiling() or not _plain_call(self) \
                or torch.nn.modules.module._has_any_global_hook() or _lib.under_transform() or not isinstance(x, torch.Tensor) or x.dim() != 5 \
                or self.groups != 1 or tuple(self.stride) != (2, 2, 2) or tuple(self.padding) != (0, 0, 0) \
                or tuple(self.output_padding) != (0, 0, 0) or tuple(self.dilation) != (1, 1, 1):
            return None
        if (autocast_dtype(x) or x.dtype) not in (torch.bfloat16, torch.float16) or self.in_channels % 64 or self.out_channels % 32 or x.shape[0] == 0:
            return None  # (said before anything is packed for the call)
        extents = [int(e) for e in extents]
        short = [e - 2 * x.shape[2 + i] for i, e in enumerate(extents)]
        if min(short) < 0 or max(short) != 1:
            return None
        return self._upsample(x, extents)

    def _upsample(self, x, extents):
        dt = autocast_dtype(x)
        x = cast_operand(x, dt)
        weight, bias = self.weight, self.bias
        wc = compute_copy(weight, dt)
        bc = compute_copy(bias, dt) if wc is not None else None
        master = wc is not None and (bias is None or bc is not None)
        stride, done, w, b = tuple(self.stride), None, weight, bias
        if self.groups == 1 and tuple(self.padding) == tuple(self.output_padding) == (0, 0, 0) and tuple(self.dilation) == (1, 1, 1) \
                and x.dim() == 5:
            # the problem the packed forms belong to: the stride-k convolution over this op's output
            n, _, d, h, wd = x.shape
            big = torch.Size((n, weight.shape[1], d * stride[0], h * stride[1], wd * stride[2]))
            pf = pd = None
            if not master and _narrowed(weight, bias, dt, x.dtype):
                w, b, (pf, pd), _ = _master_operands(weight, bias, dt, big, stride, (0, 0, 0), (1, 1, 1), True)
                master = True
            else:
                w, b = (wc, bc) if master else (cast_operand(weight, dt), cast_operand(bias, dt))
                packs = _current_packs(weight, w, big, stride, (0, 0, 0), (1, 1, 1)) if master or w is weight else None
                if packs is not None:
                    pf, pd = packs.fwd, packs.dgrad
            if pf is None or pd is None:
                pf = pd = None
            takes_w, takes_b = weight if master else w, bias if master else b
            if _lib.under_transform():
                return _lib.one_node(
                    lambda x_, w_, b_: self._served(_lib.native().conv_transpose(x_, w_, b_, w_ if takes_w is w else w, b_ if takes_b is b else b,
                                                                                 stride, None, None, 0, master, None), x, w)[0], x, takes_w, takes_b)
            done = _lib.native().conv_transpose(x, takes_w, takes_b, w, b, stride, pf, pd, self.out_halo, master, extents)
        if extents is not None:
            return None if done is None else done[0]
        y, slab = self._served(done, x, w)
        if slab is not None:
            y._sfh_slab = (slab, self.out_halo)
        return y


class FastGroupNorm(nn.GroupNorm):
    """``nn.GroupNorm`` (+ optional fused ReLU) served by the HIP kernels; output dtype = input dtype."""

    activation = None  # class-level default: not a parameter, buffer or state-dict key
    #: the halo of a ``FastMaxPool3d`` that reads this module's output next (None: none does): where the convolution in front runs
    #: with this module in one call, that call can make the pooled tensor too (:func:`conv_then_norm`)
    pool_next = None
    #: depth planes of zero halo to leave around the output for a following ``FastConv3d.shard_halo`` (0: none)
    out_halo = 0

    def __init__(self, num_groups, num_channels, eps=1e-5, affine=True, device=None, dtype=None, activation=None):
        super().__init__(num_groups, num_channels, eps=eps, affine=affine, device=device, dtype=dtype)
        if activation not in _gn.SUPPORTED_ACTIVATIONS:
            raise ValueError(f"activation must be one of {_gn.SUPPORTED_ACTIVATIONS}, got {activation!r}")
        self.activation = activation

    def extra_repr(self) -> str:
        base = super().extra_repr()
        return base if self.activation is None else f"{base}, activation={self.activation!r}"

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        if x.dim() == 5 and not x.is_contiguous(memory_format=_CL3D):
            x = x.contiguous(memory_format=_CL3D)
        return _gn.group_norm(x, self.num_groups, self.weight, self.bias, self.eps, self.activation, out_dtype=None,
                              out_halo=self.out_halo)
