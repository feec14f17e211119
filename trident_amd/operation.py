"""Attention autograd Function behind the reference's operator API.

Mirrors trident/operation/attention.py:23-202: the same eight positional arguments, the same
validation errors, the same saved state and the same 8-tuple returned by backward. The three
Triton launches of the reference (attention.py:109, 161, 170) become calls into
libtrident_attn.so (include/tri_attn.h).
"""
import ctypes
from typing import Any

import torch

from . import _lib, config, util


def _strides4(t: torch.Tensor):
    s = list(t.stride())
    if t.shape[-1] == 1:
        s[-1] = 1
    return s


def _dense_rows(t: torch.Tensor) -> torch.Tensor:
    """The kernels need unit stride along the last dimension and non-negative strides."""
    if t.shape[-1] != 1 and t.stride(-1) != 1:
        return t.contiguous()
    return t


def _require_same_gpu(device, **tensors):
    """Every tensor handed to the library must live on the one GPU the call runs on: the kernels
    dereference the raw pointers, so a host or other-device tensor must stop here, as an exception."""
    if device.type != "cuda":
        raise RuntimeError("trident_amd attention runs on the GPU only; got a tensor on " + str(device))
    for name, t in tensors.items():
        if t is not None and t.device != device:
            raise RuntimeError(f"trident_amd attention: {name} is on {t.device}, expected {device} "
                               "(all tensors of a call must be on the same GPU)")


def _next_seed():
    fixed = config.dropout_seed
    if fixed is None:
        return int(torch.randint(0, 2**63 - 1, (1,), dtype=torch.int64).item()), 0
    if isinstance(fixed, int):
        fixed = (fixed, 0)
    seed, offset = int(fixed[0]), int(fixed[1])
    config.dropout_seed = (seed, offset + 1)
    return seed, offset


_NO_STRIDES = (0, 0, 0, 0)


def _strides_or_zero(t):
    if t is None:
        return _NO_STRIDES
    return t.stride() if t.shape[-1] != 1 else tuple(_strides4(t))


def _make_args(query, key, value, output, log2sum, mask, dropout_p, is_causal, softmax_scale, seed, offset,
               grad_output=None, grad_query=None, grad_key=None, grad_value=None, grad_mask=None, delta=None):
    """TriAttnArgs (include/tri_attn.h) for one call, on torch's current stream of the query's device."""
    args = _lib.TriAttnArgs()
    num_batches, num_heads, y_size, x_size = query.shape
    _lib.ARGS_PACKER.pack_into(
        args, 0,
        _lib.ARGS_PACKER.size, util.dtype(query.dtype), num_batches, num_heads, y_size, x_size,
        1 if is_causal else 0, 0 if mask is None else util.dtype(mask.dtype), softmax_scale, dropout_p, seed, offset,
        query.data_ptr(), key.data_ptr(), value.data_ptr(), output.data_ptr(), log2sum.data_ptr(),
        0 if mask is None else mask.data_ptr(),
        0 if grad_output is None else grad_output.data_ptr(),
        0 if grad_query is None else grad_query.data_ptr(),
        0 if grad_key is None else grad_key.data_ptr(),
        0 if grad_value is None else grad_value.data_ptr(),
        0 if grad_mask is None else grad_mask.data_ptr(),
        0 if delta is None else delta.data_ptr(),
        *query.stride(), *key.stride(), *value.stride(), *output.stride(),
        *_strides_or_zero(grad_output), *_strides_or_zero(grad_query), *_strides_or_zero(grad_key),
        *_strides_or_zero(grad_value), *_strides_or_zero(mask), *_strides_or_zero(grad_mask),
        torch._C._cuda_getCurrentRawStream(query.device.index), 0,
    )
    return args


def _take_workspace(args, which, device):
    """Gives the call (0: forward, 3: backward, 4: mask gradient) the scratch memory with which it runs split along the sequence, where it does and
    the GPU has that much left; returns the tensor to keep alive until the call is enqueued."""
    size = _lib.lib().tri_attn_workspace_size(ctypes.byref(args), which)
    if size <= 0:
        return None
    try:
        workspace = torch.empty(size, dtype=torch.uint8, device=device)
    except torch.OutOfMemoryError:
        return None
    args.workspace, args.workspace_size = workspace.data_ptr(), size
    return workspace


# Classes of a mask's 64 x 64 blocks (tri_attn_classify_mask), kept per mask tensor (csrc_torch/torch_ops.cpp): the forward
# call computes them, the backward call and later calls with the same, unmodified tensor (other layers, other steps) find
# them there. An entry ends with its tensor (weak reference) and is recomputed when the tensor was written to through torch
# (its version counter moved), when another stream asks for it (no event orders the two), and it is neither made nor used
# while a stream is being captured (the classification would be recorded, not run). A write that torch does not see (through
# ``.data``, a raw pointer, a graph replay into the mask's memory) leaves stale classes behind, and the kernels skip
# tiles on their word: such callers set ``config.cache_mask_classes = False`` (every call classifies the mask again)
# or call ``forget_mask_classes()`` after the write.
def forget_mask_classes():
    """Drops every cached block classification (after a write to a mask's memory that torch's version counter did not see)."""
    _lib.torch_ops().forget_mask_classes()


def _mask_classes(mask: torch.Tensor, args):
    """Sets args.mask_classes for the mask already described in ``args``; returns the tensor to keep alive, or None
    where the library has no use for classes (nothing is launched then; padded masks bring theirs along, the kernels use no others at
    lengths that are no multiple of 64, and those of fp32 calls use none)."""
    return _lib.torch_ops().mask_classes(mask, ctypes.addressof(args), bool(config.cache_mask_classes))


class _BooleanMask:
    """A boolean attn_mask (True = the key takes part) on its way through forward and backward: the additive mask the
    kernels read is made by the forward call and kept for the backward."""

    __slots__ = ("source", "device", "prepared")
    requires_grad = False

    def __init__(self, source):
        self.source = source
        self.device = source.device
        self.prepared = None


class _PreparedMask:
    """Additive mask for ``query``'s kernels, its rows padded to whole pieces of 64 keys (tri_attn_prepare_mask), broadcast
    like ``source`` (additive or boolean), and the classes of its blocks for the kernels that look at them. (Plain numbers
    and two allocations: views of the buffer would cost a small call as much as its kernels.)"""

    __slots__ = ("padded", "classes", "strides", "dtype")

    def __init__(self, source, query):
        num_batches, num_heads, y_size, _ = query.shape
        full = (num_batches, num_heads, y_size, y_size)
        missing = 4 - source.dim()
        if missing < 0 or any(n != 1 and n != m for n, m in zip(source.shape, full[missing:])):
            source.expand(full)  # (raises)
        # (a dimension the source broadcasts is kept once)
        shape = (1,) * missing + tuple(source.shape)
        given = (0,) * missing + source.stride()
        from_strides = [0 if n == 1 else t for n, t in zip(shape, given)]
        batches, heads, rows = [1 if t == 0 else n for n, t in zip(shape[:3], from_strides)]
        pitch = (y_size + 63) // 64 * 64
        boolean = source.dtype == torch.bool
        dtype = query.dtype if boolean else source.dtype
        self.padded = torch.empty(batches * heads * rows * pitch, device=query.device, dtype=dtype)
        self.strides = (heads * rows * pitch if batches > 1 else 0, rows * pitch if heads > 1 else 0, pitch if rows > 1 else 0, 1)
        self.dtype = util.dtype(dtype) | _lib.MASK_PADDED | (_lib.MASK_BINARY if boolean else 0)
        self.classes = None
        args = _lib.TriAttnArgs()
        args.struct_size = _lib.ARGS_PACKER.size
        args.B, args.H, args.S = num_batches, num_heads, y_size
        args.stream = torch._C._cuda_getCurrentRawStream(query.device.index)
        if query.dtype != torch.float32:
            blocks = pitch // 64
            self.classes = torch.empty(batches * heads * (blocks if rows > 1 else 1) * blocks, dtype=torch.uint8, device=query.device)
        self.describe(args)
        _lib.check(_lib.lib().tri_attn_prepare_mask(ctypes.byref(args), source.data_ptr(), _lib.BOOL if boolean else util.dtype(dtype),
                                                    (ctypes.c_int64 * 4)(*from_strides)))

    def describe(self, args):
        """The mask's fields of a call's arguments."""
        args.mask = self.padded.data_ptr()
        args.mask_dtype = self.dtype
        args.mask_stride[:] = self.strides
        if self.classes is not None:
            args.mask_classes = self.classes.data_ptr()


# Scores times head size from which an additive mask at a ragged length is copied into padded rows (_prepared_mask), and what
# lengths beyond 128 count as at least.
_PADS_FROM = 1 << 28
_PADS_LONG = 1 << 28


def _worth_padding(query):
    num_batches, num_heads, y_size, x_size = query.shape
    work = num_batches * num_heads * y_size * y_size * max(x_size, 32)
    return max(work, _PADS_LONG if y_size > 128 else 0) >= _PADS_FROM


def _sums_mask_gradient(mask, query):
    """Whether the gradient of ``mask`` is made by a kernel of its own (tri_attn_bwd_dmask) behind the backward: 16-bit problems, a
    mask with rows and keys of its own that batches or heads share, or any such mask at a length that is no multiple of 128,
    where the dQ pass of the 16-bit kernels does not write it (and the call is large enough for them)."""
    shape4 = (1,) * (4 - mask.dim()) + tuple(mask.shape)
    num_batches, num_heads, y_size, _ = query.shape
    return query.dtype != torch.float32 and shape4[2:] == (y_size, y_size) and (
        shape4[:2] != (num_batches, num_heads) or (y_size % 128 != 0 and (y_size % 64 == 0 or _worth_padding(query))))


def _prepared_mask(mask, query):
    """The _PreparedMask of a call, or None where the mask is handed over as it is. Boolean masks always have one. Additive
    ones are copied into padded rows for 16-bit problems at lengths that are no multiple of 64, whose kernels fetch mask rows
    in 16-byte pieces up to the end of a 64-key tile: one more pass over the mask (at the copy rate) in each direction against
    kernels that read masks element by element (bf16, dense fp32 mask, forward + backward: B=16 H=12 S=777 D=64 2.22 -> 0.39 ms,
    S=500 D=16 0.38 -> 0.21, S=333 D=128 0.93 -> 0.22). Those kernels take their time per row whatever the number of heads (B=1
    H=4 D=64: S=400 57 -> 20 us forward, 190 -> 80 with the backward; S=200 32 -> 15 forward), so that only at lengths up to 128, below
    _PADS_FROM scores times head size, the launches and their arguments cost a call more than the kernels save (S=100, 64 heads,
    with the backward: 70 -> 81 us). A mask whose gradient the dQ pass writes stays as it is: the gradient is laid out like it.
    So does one that the GPU has no memory left to copy."""
    if isinstance(mask, _BooleanMask):
        if mask.prepared is None:
            mask.prepared = _PreparedMask(mask.source, query)
            mask.source = None
        return mask.prepared
    if query.shape[2] % 64 == 0 or not _worth_padding(query):
        return None
    if query.dtype == torch.float32 or mask.dtype not in (torch.float32, query.dtype):
        return None
    if mask.requires_grad and not _sums_mask_gradient(mask, query):
        return None
    try:
        return _PreparedMask(mask.detach(), query)
    except torch.OutOfMemoryError:
        return None


def _expand_mask(mask: torch.Tensor, shape):
    """View of the additive mask broadcast to [B,H,S,S] (stride 0 on broadcast dims)."""
    view = mask
    while view.dim() < 4:
        view = view.unsqueeze(0)
    view = view.expand(*shape)
    if view.shape[-1] != 1 and view.stride(-1) != 1:
        view = view.contiguous()
    return view


class _NoGraph:
    """Stands in for the autograd context when no gradient is asked for."""

    def save_for_backward(self, *tensors):
        pass


class Attention(torch.autograd.Function):
    @staticmethod
    def call(query, key, value, mask, dropout_p, is_causal, softmax_scale, use_accelerator):
        """``apply`` with the same arguments, checks and result. Plain calls run in C++ (csrc_torch/torch_ops.cpp), which
        returns None for all others; when no input asks for a gradient (or gradients are switched off) the forward runs
        without autograd's bookkeeping, which a small problem would feel."""
        output = _lib.torch_ops().attention(query, key, value, mask, dropout_p, is_causal, softmax_scale)
        if output is not None:
            return output
        if torch.is_grad_enabled() and (
            query.requires_grad or key.requires_grad or value.requires_grad or (mask is not None and mask.requires_grad)
        ):
            return Attention.apply(query, key, value, mask, dropout_p, is_causal, softmax_scale, use_accelerator)
        return Attention.forward(_NoGraph(), query, key, value, mask, dropout_p, is_causal, softmax_scale, use_accelerator)

    @staticmethod
    def forward(ctx: Any, *args: Any, **kwargs: Any):
        query, key, value, mask, dropout_p, is_causal, softmax_scale, use_accelerator = args

        if query.dim() != 4 or key.dim() != 4 or value.dim() != 4:
            raise ValueError("The dimension of query, key and value should be 4.")

        if (
            not util.is_pow2(query.shape[-1])
            or not util.is_pow2(key.shape[-1])
            or not util.is_pow2(value.shape[-1])
            or (
                config.reference_limits
                and (
                    not util.is_pow2(query.shape[-2])
                    or not util.is_pow2(key.shape[-2])
                    or not util.is_pow2(value.shape[-2])
                )
            )
        ):
            raise ValueError("Attention supports only for power of 2 size tensors.")

        if mask is not None:
            if is_causal:
                raise ValueError("Error because both attn_mask and is_causal are set.")
            if mask.dtype == torch.bool:
                if config.reference_limits:
                    raise ValueError("Boolean mask is not supported yet.")
                # torch's meaning of a boolean attn_mask: True = the key takes part in the attention (the additive
                # mask is made in the operand type: half the bytes of an fp32 one for the 16-bit kernels to stream)
                mask = _BooleanMask(mask)

        seed, offset = _next_seed() if dropout_p > 0.0 else (0, 0)

        util.push_trace("Attention.__forward")
        output, log_sum_exp = Attention._forward(
            query, key, value, mask, dropout_p, is_causal, softmax_scale, seed, offset
        )
        util.pop_trace()

        ctx.save_for_backward(query, key, value, output, log_sum_exp)
        ctx.mask = mask
        ctx.dropout_p = dropout_p
        ctx.is_causal = is_causal
        ctx.softmax_scale = softmax_scale
        ctx.use_accelerator = use_accelerator
        ctx.seed = seed
        ctx.offset = offset

        return output

    @staticmethod
    def backward(ctx: Any, *grad_outputs: Any):
        (grad_output,) = grad_outputs
        query, key, value, output, log_sum_exp = ctx.saved_tensors

        util.push_trace("Attention.__backward")
        grad_query, grad_key, grad_value, grad_mask = Attention._backward(
            grad_output,
            query,
            key,
            value,
            output,
            log_sum_exp,
            ctx.mask,
            ctx.softmax_scale,
            ctx.dropout_p,
            ctx.is_causal,
            ctx.seed,
            ctx.offset,
            ctx.mask is not None and ctx.needs_input_grad[3],
        )
        util.pop_trace()

        return grad_query, grad_key, grad_value, grad_mask, None, None, None, None

    @staticmethod
    def _forward(query, key, value, mask, dropout_p, is_causal, softmax_scale, seed, offset):
        assert query.shape[-1] == key.shape[-1] and key.shape[-1] == value.shape[-1]
        assert key.shape[-1] in {16, 32, 64, 128}
        _require_same_gpu(query.device, key=key, value=value, mask=mask)
        if key.shape != query.shape or value.shape != query.shape:
            raise ValueError("query, key and value must have the same shape.")
        if key.dtype != query.dtype or value.dtype != query.dtype:
            raise ValueError("query, key and value must have the same dtype.")

        lib = _lib.lib()
        query, key, value = _dense_rows(query), _dense_rows(key), _dense_rows(value)
        num_batches, num_heads, y_size, x_size = query.shape
        output = torch.empty(query.shape, device=query.device, dtype=query.dtype)
        log2sum = torch.empty(num_batches, num_heads, y_size, device=query.device, dtype=torch.float32)
        # (a mask handed over as it is goes into the arguments with everything else: setting its fields one by one afterwards
        # cost a small call 2 us of its 17)
        prepared = _prepared_mask(mask, query) if mask is not None else None
        mask_view = None
        if mask is not None and prepared is None:
            mask_view = _expand_mask(mask.detach(), (num_batches, num_heads, y_size, y_size))
        args = _make_args(query, key, value, output, log2sum, mask_view, dropout_p, is_causal, softmax_scale, seed, offset)
        if prepared is not None:
            prepared.describe(args)
        classes = _mask_classes(mask, args) if mask_view is not None else None  # (kept alive until the call is enqueued)

        workspace = _take_workspace(args, 0, query.device)  # noqa: F841  (kept alive until the call is enqueued)

        util.push_trace("kernel.Attention.forward")
        _lib.check(lib.tri_attn_fwd(ctypes.byref(args)))
        util.pop_trace()

        return output, log2sum

    @staticmethod
    def _backward(grad_output, query, key, value, output, log2sum, mask, softmax_scale, dropout_p, is_causal,
                  seed, offset, want_grad_mask, delta_out=None):
        """``delta_out``: optional fp32 [B,H,S] tensor that receives delta (the backward's intermediate,
        trident/operation/attention.py:155); allocated here when not given."""
        _require_same_gpu(query.device, key=key, value=value, mask=mask, grad_output=grad_output, output=output,
                          log_sum_exp=log2sum)
        lib = _lib.lib()
        query, key, value = _dense_rows(query), _dense_rows(key), _dense_rows(value)
        grad_output = _dense_rows(grad_output)
        log2sum = log2sum.contiguous()  # (a saved-tensor hook may have laid it out anew)
        num_batches, num_heads, y_size, x_size = output.shape
        grad_query = torch.empty(query.shape, device=query.device, dtype=query.dtype)
        grad_key = torch.empty(key.shape, device=key.device, dtype=key.dtype)
        grad_value = torch.empty(value.shape, device=value.device, dtype=value.dtype)
        delta = torch.empty_like(log2sum) if delta_out is None else delta_out
        full = (num_batches, num_heads, y_size, y_size)
        # The mask gradient (trident/kernel/attention.py:332-335) in the mask's own shape: a full [B,H,S,S] mask gets
        # dS written in place; one shared by batches or heads gets dS summed over them by a kernel of its own
        # (tri_attn_bwd_dmask); what that does not take (fp32, a mask that is also shared by the rows) gets a zero-filled
        # fp32 buffer of its shape that the kernels add to through strides of 0.
        grad_mask_buf = grad_mask_view = mask_view = None
        summed = want_grad_mask and _sums_mask_gradient(mask, query)
        prepared = _prepared_mask(mask, query) if mask is not None and not want_grad_mask else None
        if mask is not None and prepared is None:
            mask_view = _expand_mask(mask.detach(), full)
        if want_grad_mask:
            shape4 = (1,) * (4 - mask.dim()) + tuple(mask.shape)
            if shape4 == full or summed:
                grad_mask_buf = torch.empty(shape4, device=mask.device, dtype=mask.dtype)
                grad_mask_view = grad_mask_buf if shape4 == full else grad_mask_buf.expand(*full)

        args = _make_args(query, key, value, output, log2sum, mask_view, dropout_p, is_causal, softmax_scale, seed, offset,
                          grad_output, grad_query, grad_key, grad_value, grad_mask_view, delta)
        classes = None  # (kept alive until the call is enqueued, as ``prepared``)
        if summed:
            summed = lib.tri_attn_uses_matrix_cores(ctypes.byref(args), 3) == 1
            if summed:  # (else the dQ pass writes it: in place, or below, into what broadcast dimensions are added up in)
                args.dmask = None
                prepared = _prepared_mask(mask, query)
        if prepared is not None:
            prepared.describe(args)
        elif mask is not None and (summed or not want_grad_mask):
            # (a learned mask finds the classes of its forward call; under capture nothing is kept, and in the 16-bit types, where the
            # mask matrix is small beside the scores' work, one more pass over it costs more than it saves: B=2 H=4 S=128 D=128,
            # replayed backward 49 us with it, 39 without)
            if not summed or mask.dtype == torch.float32 or not torch.cuda.is_current_stream_capturing():
                classes = _mask_classes(mask, args)
        elif want_grad_mask:
            if shape4 != full:
                grad_mask_buf = torch.zeros(shape4, device=mask.device, dtype=torch.float32)
                grad_mask_view = grad_mask_buf.expand(*full)
                args.dmask = grad_mask_view.data_ptr()
                args.dmask_stride[:] = _strides_or_zero(grad_mask_view)
                if mask_view.dtype != torch.float32:  # (mask and dmask share one dtype field)
                    mask_view = _expand_mask(mask.detach().float(), full)
                    args.mask = mask_view.data_ptr()
                    args.mask_dtype = util.dtype(torch.float32)
                    args.mask_stride[:] = _strides_or_zero(mask_view)
            # (the classes describe the mask tensor as the kernels see it: not when it was converted to fp32 above)
            if mask_view.dtype == mask.dtype:
                classes = _mask_classes(mask, args)

        # one call for the three backward launches (trident/operation/attention.py:161-199 launches the
        # delta pre-pass and the backward kernel): the library orders them, and where the dQ kernel can
        # compute delta on its way the pre-pass disappears into it
        workspace = _take_workspace(args, 3, query.device)  # noqa: F841  (kept alive until the call is enqueued)
        util.push_trace("kernel.Attention.backward")
        _lib.check(lib.tri_attn_bwd(ctypes.byref(args)))
        if summed:
            args.mask = mask_view.data_ptr()
            args.mask_dtype = util.dtype(mask_view.dtype)
            args.mask_stride[:] = _strides_or_zero(mask_view)
            args.dmask = grad_mask_buf.data_ptr()
            args.workspace, args.workspace_size = None, 0
            sums = _take_workspace(args, 4, query.device)  # noqa: F841  (kept alive until the call is enqueued)
            _lib.check(lib.tri_attn_bwd_dmask(ctypes.byref(args)))
        util.pop_trace()

        grad_mask = None
        if grad_mask_buf is not None:
            grad_mask = grad_mask_buf.to(mask.dtype).reshape(mask.shape)

        return grad_query, grad_key, grad_value, grad_mask


from .rowops import Dropout, MaskedSoftmax, Softmax  # noqa: E402,F401  (trident.operation.Softmax etc.)
