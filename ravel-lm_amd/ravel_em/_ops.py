"""torch.library custom ops over the C ABI.

The ops carry fake (meta) implementations and autograd formulas so that
``torch.compile(fullgraph=True)`` can trace through them, following the
custom_op + register_fake + register_autograd pattern of the reference's MPS arm
(ravel_lm/mps_memory.py:109-187).  Every op launches on torch's current stream
and allocates its workspace from torch's caching allocator.
"""
from __future__ import annotations

from typing import Optional, Tuple

import torch

from . import _native as nat

Tensor = torch.Tensor


def _call(fn, *args) -> None:
    nat.check(fn(*args))


def eager(*tensors: Optional[Tensor]) -> bool:
    """True when a call may run an op's implementation directly instead of
    through the dispatcher: nothing is tracing (no torch.compile) and every
    tensor is a plain tensor (no fake, meta-programming or other subclass).
    The callers also require that no autograd graph is recorded.  The
    dispatcher costs several microseconds a call, which short tapes notice."""
    if torch.compiler.is_compiling():
        return False
    return all(t is None or type(t) is torch.Tensor for t in tensors)


# No functorch transform and no dispatch mode may watch a call that takes the
# autograd functions at the end of this file instead of the custom ops.
_transforms = getattr(torch._C, "_are_functorch_transforms_active", None)
_modes = getattr(torch._C, "_len_torch_dispatch_stack", None)


def eager_graph(*tensors: Optional[Tensor]) -> bool:
    """eager() for a call that records an autograd graph."""
    return (_transforms is not None and _modes is not None and eager(*tensors)
            and not _transforms() and _modes() == 0)


# ------------------------------------------------------------- latest-k --


def latest_k_impl(
    write_addresses: Tensor,
    payloads: Tensor,
    read_addresses: Optional[Tensor],
    write_mask: Optional[Tensor],
    address_space: int,
    k: int,
    want_src: bool,
) -> Tuple[Tensor, Tensor, Tensor]:
    """The body of ravel_em::latest_k (also called directly, see eager)."""
    lib = nat.library()
    B, T, C = write_addresses.shape
    D = payloads.shape[-1]
    dev = payloads.device
    values = payloads.new_empty(B, T, C, k, D)
    mask = torch.empty(B, T, C, k, dtype=torch.bool, device=dev)
    src = torch.empty((B, T, C, k) if want_src else (0,), dtype=torch.int32, device=dev)
    has_read = read_addresses is not None
    has_mask = write_mask is not None
    nbytes = lib.ravel_em_latest_k_workspace(B, T, C, address_space, k, int(has_read), int(has_mask), int(want_src))
    ws = nat.workspace(nbytes, dev)
    _call(
        lib.ravel_em_latest_k_fwd,
        nat.ptr(write_addresses), nat.ptr(read_addresses), nat.addr_code(write_addresses.dtype),
        nat.ptr(write_mask), nat.ptr(payloads), nat.payload_code(payloads.dtype),
        B, T, C, D, address_space, k,
        nat.ptr(values), nat.ptr(mask), nat.ptr(src) if want_src else None,
        nat.ptr(ws), ws.numel(), nat.stream_of(payloads),
    )
    nat.after_call(ws)
    return values, mask, src


@torch.library.custom_op("ravel_em::latest_k", mutates_args=())
def latest_k(
    write_addresses: Tensor,
    payloads: Tensor,
    read_addresses: Optional[Tensor],
    write_mask: Optional[Tensor],
    address_space: int,
    k: int,
    want_src: bool,
) -> Tuple[Tensor, Tensor, Tensor]:
    return latest_k_impl(write_addresses, payloads, read_addresses, write_mask, address_space, k,
                         want_src)


@latest_k.register_fake
def _latest_k_fake(write_addresses, payloads, read_addresses, write_mask, address_space, k, want_src):
    B, T, C = write_addresses.shape
    D = payloads.shape[-1]
    dev = payloads.device
    return (
        payloads.new_empty(B, T, C, k, D),
        torch.empty(B, T, C, k, dtype=torch.bool, device=dev),
        torch.empty((B, T, C, k) if want_src else (0,), dtype=torch.int32, device=dev),
    )


def latest_k_backward_impl(src: Tensor, grad_values: Tensor, chain: bool) -> Tensor:
    lib = nat.library()
    B, T, C, k, D = grad_values.shape
    grad_values = grad_values.contiguous()
    grad_payload = grad_values.new_empty(B, T, C, D)
    code = nat.payload_code(grad_values.dtype)
    nbytes = lib.ravel_em_latest_k_bwd_workspace(B, T, C, D, k, code, int(chain))
    ws = nat.workspace(nbytes, grad_values.device)
    _call(
        lib.ravel_em_latest_k_bwd,
        nat.ptr(src), nat.ptr(grad_values), code, B, T, C, D, k, int(chain),
        nat.ptr(grad_payload), nat.ptr(ws), ws.numel(), nat.stream_of(grad_values),
    )
    if not chain:  # the sorted form's workspace carries a status word
        nat.after_call(ws)
    return grad_payload


@torch.library.custom_op("ravel_em::latest_k_backward", mutates_args=())
def latest_k_backward(src: Tensor, grad_values: Tensor, chain: bool) -> Tensor:
    return latest_k_backward_impl(src, grad_values, chain)


@latest_k_backward.register_fake
def _latest_k_backward_fake(src, grad_values, chain):
    B, T, C, k, D = grad_values.shape
    return grad_values.new_empty(B, T, C, D)


def _latest_k_setup(ctx, inputs, output):
    write_addresses, payloads, read_addresses, write_mask, address_space, k, want_src = inputs
    _, mask, src = output
    ctx.save_for_backward(src)
    ctx.chain = read_addresses is None and write_mask is None
    ctx.want_src = want_src
    ctx.mark_non_differentiable(mask, src)
    ctx.set_materialize_grads(False)  # no zero gradients of the mask and the sources


def _latest_k_grad(ctx, grad_values, _grad_mask, _grad_src):
    (src,) = ctx.saved_tensors
    if not ctx.want_src:
        raise RuntimeError("ravel_em.latest_k was called without sources; cannot differentiate")
    if grad_values is None:
        return (None,) * 7
    grad_payload = latest_k_backward(src, grad_values, ctx.chain)
    return None, grad_payload, None, None, None, None, None


latest_k.register_autograd(_latest_k_grad, setup_context=_latest_k_setup)


# -------------------------------------------------------------- seg-sum --


def seg_sum_impl(
    write_addresses: Tensor,
    payloads: Tensor,
    read_addresses: Optional[Tensor],
    write_mask: Optional[Tensor],
    address_space: int,
    keys: Optional[Tensor] = None,
) -> Tuple[Tensor, Tensor]:
    """The body of ravel_em::seg_sum (also called directly, see eager); the
    sorted keys of the tape go to `keys` when given (kept_keys)."""
    lib = nat.library()
    B, T, C = write_addresses.shape
    D = payloads.shape[-1]
    dev = payloads.device
    out = payloads.new_empty(B, T, C, D)
    mask = torch.empty(B, T, C, dtype=torch.bool, device=dev)
    code = nat.payload_code(payloads.dtype)
    nbytes = lib.ravel_em_seg_sum_workspace(
        B, T, C, D, address_space, int(read_addresses is not None), int(write_mask is not None), code
    )
    ws = nat.workspace(nbytes, dev)
    keep = () if keys is None else (nat.ptr(keys), keys.numel())
    _call(
        lib.ravel_em_seg_sum_fwd if keys is None else lib.ravel_em_seg_sum_fwd_keep,
        nat.ptr(write_addresses), nat.ptr(read_addresses), nat.addr_code(write_addresses.dtype),
        nat.ptr(write_mask), nat.ptr(payloads), code, B, T, C, D, address_space,
        nat.ptr(out), nat.ptr(mask), *keep, nat.ptr(ws), ws.numel(), nat.stream_of(payloads),
    )
    nat.after_call(ws)
    return out, mask


@torch.library.custom_op("ravel_em::seg_sum", mutates_args=())
def seg_sum(
    write_addresses: Tensor,
    payloads: Tensor,
    read_addresses: Optional[Tensor],
    write_mask: Optional[Tensor],
    address_space: int,
) -> Tuple[Tensor, Tensor]:
    return seg_sum_impl(write_addresses, payloads, read_addresses, write_mask, address_space)


@seg_sum.register_fake
def _seg_sum_fake(write_addresses, payloads, read_addresses, write_mask, address_space):
    B, T, C = write_addresses.shape
    D = payloads.shape[-1]
    return payloads.new_empty(B, T, C, D), torch.empty(B, T, C, dtype=torch.bool, device=payloads.device)


def seg_sum_backward_impl(
    write_addresses: Tensor,
    read_addresses: Optional[Tensor],
    write_mask: Optional[Tensor],
    grad_sum: Tensor,
    address_space: int,
) -> Tensor:
    lib = nat.library()
    B, T, C, D = grad_sum.shape
    grad_sum = grad_sum.contiguous()
    grad_payload = grad_sum.new_empty(B, T, C, D)
    code = nat.payload_code(grad_sum.dtype)
    nbytes = lib.ravel_em_seg_sum_bwd_workspace(
        B, T, C, D, address_space, int(read_addresses is not None), int(write_mask is not None), code
    )
    ws = nat.workspace(nbytes, grad_sum.device)
    _call(
        lib.ravel_em_seg_sum_bwd,
        nat.ptr(write_addresses), nat.ptr(read_addresses), nat.addr_code(write_addresses.dtype),
        nat.ptr(write_mask), nat.ptr(grad_sum), code, B, T, C, D, address_space,
        nat.ptr(grad_payload), nat.ptr(ws), ws.numel(), nat.stream_of(grad_sum),
    )
    nat.after_call(ws)
    return grad_payload


@torch.library.custom_op("ravel_em::seg_sum_backward", mutates_args=())
def seg_sum_backward(
    write_addresses: Tensor,
    read_addresses: Optional[Tensor],
    write_mask: Optional[Tensor],
    grad_sum: Tensor,
    address_space: int,
) -> Tensor:
    return seg_sum_backward_impl(write_addresses, read_addresses, write_mask, grad_sum,
                                 address_space)


@seg_sum_backward.register_fake
def _seg_sum_backward_fake(write_addresses, read_addresses, write_mask, grad_sum, address_space):
    return grad_sum.new_empty(grad_sum.shape)


def _seg_sum_setup(ctx, inputs, output):
    write_addresses, payloads, read_addresses, write_mask, address_space = inputs
    ctx.save_for_backward(write_addresses, read_addresses, write_mask)
    ctx.address_space = address_space
    ctx.mark_non_differentiable(output[1])
    ctx.set_materialize_grads(False)


def _seg_sum_grad(ctx, grad_sum, _grad_mask):
    write_addresses, read_addresses, write_mask = ctx.saved_tensors
    if grad_sum is None:
        return (None,) * 5
    grad_payload = seg_sum_backward(write_addresses, read_addresses, write_mask, grad_sum, ctx.address_space)
    return None, grad_payload, None, None, None


seg_sum.register_autograd(_seg_sum_grad, setup_context=_seg_sum_setup)


# ------------------------------------------------------ latest-k + sum --


def latest_k_sum_impl(
    write_addresses: Tensor,
    payloads: Tensor,
    read_addresses: Optional[Tensor],
    write_mask: Optional[Tensor],
    address_space: int,
    k: int,
    want_src: bool,
    keys: Optional[Tensor] = None,
) -> Tuple[Tensor, Tensor, Tensor, Tensor, Tensor]:
    """The body of ravel_em::latest_k_sum (also called directly, see eager):
    (values, mask, src, sum, sum_mask) of one tape in one C call; the sorted keys
    of the tape go to `keys` when given (kept_keys; then no sources)."""
    lib = nat.library()
    B, T, C = write_addresses.shape
    D = payloads.shape[-1]
    dev = payloads.device
    values = payloads.new_empty(B, T, C, k, D)
    mask = torch.empty(B, T, C, k, dtype=torch.bool, device=dev)
    src = torch.empty((B, T, C, k) if want_src else (0,), dtype=torch.int32, device=dev)
    out = payloads.new_empty(B, T, C, D)
    smask = torch.empty(B, T, C, dtype=torch.bool, device=dev)
    code = nat.payload_code(payloads.dtype)
    nbytes = lib.ravel_em_latest_k_sum_workspace(
        B, T, C, D, address_space, k, int(read_addresses is not None), int(write_mask is not None),
        int(want_src), code)
    ws = nat.workspace(nbytes, dev)
    tape = (nat.ptr(write_addresses), nat.ptr(read_addresses), nat.addr_code(write_addresses.dtype),
            nat.ptr(write_mask), nat.ptr(payloads), code, B, T, C, D, address_space, k,
            nat.ptr(values), nat.ptr(mask))
    work = (nat.ptr(ws), ws.numel(), nat.stream_of(payloads))
    if keys is None:
        _call(lib.ravel_em_latest_k_sum_fwd, *tape, nat.ptr(src) if want_src else None,
              nat.ptr(out), nat.ptr(smask), *work)
    else:
        _call(lib.ravel_em_latest_k_sum_fwd_keep, *tape, nat.ptr(out), nat.ptr(smask),
              nat.ptr(keys), keys.numel(), *work)
    nat.after_call(ws)
    return values, mask, src, out, smask


@torch.library.custom_op("ravel_em::latest_k_sum", mutates_args=())
def latest_k_sum(
    write_addresses: Tensor,
    payloads: Tensor,
    read_addresses: Optional[Tensor],
    write_mask: Optional[Tensor],
    address_space: int,
    k: int,
    want_src: bool,
) -> Tuple[Tensor, Tensor, Tensor, Tensor, Tensor]:
    return latest_k_sum_impl(write_addresses, payloads, read_addresses, write_mask, address_space,
                             k, want_src)


@latest_k_sum.register_fake
def _latest_k_sum_fake(write_addresses, payloads, read_addresses, write_mask, address_space, k,
                       want_src):
    B, T, C = write_addresses.shape
    D = payloads.shape[-1]
    dev = payloads.device
    return (
        payloads.new_empty(B, T, C, k, D),
        torch.empty(B, T, C, k, dtype=torch.bool, device=dev),
        torch.empty((B, T, C, k) if want_src else (0,), dtype=torch.int32, device=dev),
        payloads.new_empty(B, T, C, D),
        torch.empty(B, T, C, dtype=torch.bool, device=dev),
    )


def joint_backward_applies(T: int, C: int, D: int, k: int, element_size: int) -> bool:
    """Whether latest_k_sum_backward (one walk, no sources) takes the shape: the
    library's own rule (its workspace query is not 0), in plain arithmetic that
    torch.compile can trace."""
    step = C * D * element_size * k  # gradient bytes of one time step
    return (1 <= k <= 8 and 1 <= T <= 1 << 24 and C * k < 1 << 24 and step < 1 << 24
            and T * step < 1 << 31)


def latest_k_sum_backward_impl(
    write_addresses: Tensor,
    read_addresses: Optional[Tensor],
    write_mask: Optional[Tensor],
    grad_values: Optional[Tensor],
    grad_sum: Optional[Tensor],
    address_space: int,
    k: int,
    taped: bool,
    keys: int = 0,
) -> Tensor:
    """Payload gradient of latest_k (grad_values [B,T,C,k,D]), of seg_sum
    (grad_sum [B,T,C,D]) or of both of one tape; with ``taped`` the first
    argument is the tape that latest_k_taped returned, with `keys` (nat.KEYS or
    nat.KEYS_SAME) the sorted keys that the forward kept."""
    lib = nat.library()
    gv = None if grad_values is None else grad_values.contiguous()
    gs = None if grad_sum is None else grad_sum.contiguous()
    g = gs if gv is None else gv
    B, T, C, D = g.shape[0], g.shape[1], g.shape[2], g.shape[-1]
    grad_payload = g.new_empty(B, T, C, D)
    code = nat.payload_code(g.dtype)
    nbytes = lib.ravel_em_latest_k_sum_bwd_workspace(
        B, T, C, D, address_space, k,
        int(taped or keys == nat.KEYS or read_addresses is not None),
        int(write_mask is not None), code)
    ws = nat.workspace(nbytes, g.device)
    _call(
        lib.ravel_em_latest_k_sum_bwd,
        nat.ptr(write_addresses), nat.ptr(read_addresses),
        keys or (nat.TAPE if taped else nat.addr_code(write_addresses.dtype)), nat.ptr(write_mask),
        nat.ptr(gv), nat.ptr(gs), code, B, T, C, D, address_space, k, nat.ptr(grad_payload),
        nat.ptr(ws), ws.numel(), nat.stream_of(g),
    )
    nat.after_call(ws)
    return grad_payload


@torch.library.custom_op("ravel_em::latest_k_sum_backward", mutates_args=())
def latest_k_sum_backward(
    write_addresses: Tensor,
    read_addresses: Optional[Tensor],
    write_mask: Optional[Tensor],
    grad_values: Optional[Tensor],
    grad_sum: Optional[Tensor],
    address_space: int,
    k: int,
    taped: bool,
) -> Tensor:
    return latest_k_sum_backward_impl(write_addresses, read_addresses, write_mask, grad_values,
                                      grad_sum, address_space, k, taped)


@latest_k_sum_backward.register_fake
def _latest_k_sum_backward_fake(write_addresses, read_addresses, write_mask, grad_values, grad_sum,
                                address_space, k, taped):
    g = grad_sum if grad_values is None else grad_values
    return g.new_empty(*g.shape[:3], g.shape[-1])


def _latest_k_sum_setup(ctx, inputs, output):
    write_addresses, payloads, read_addresses, write_mask, address_space, k, want_src = inputs
    _, mask, src, _, smask = output
    ctx.save_for_backward(src, write_addresses, read_addresses, write_mask)
    ctx.chain = read_addresses is None and write_mask is None
    ctx.want_src = want_src
    ctx.address_space = address_space
    ctx.k = k
    ctx.mark_non_differentiable(mask, src, smask)
    ctx.set_materialize_grads(False)


def _latest_k_sum_grad(ctx, grad_values, _grad_mask, _grad_src, grad_sum, _grad_smask):
    src, write_addresses, read_addresses, write_mask = ctx.saved_tensors
    if grad_values is None and grad_sum is None:
        return (None,) * 7
    g = grad_sum if grad_values is None else grad_values
    B, T, C, D = g.shape[0], g.shape[1], g.shape[2], g.shape[-1]
    if joint_backward_applies(T, C, D, ctx.k, g.element_size()):
        grad_payload = latest_k_sum_backward(write_addresses, read_addresses, write_mask,
                                             grad_values, grad_sum, ctx.address_space, ctx.k, False)
        return None, grad_payload, None, None, None, None, None
    grad_payload = None
    if grad_values is not None:
        if not ctx.want_src:
            raise RuntimeError("ravel_em.latest_k_sum was called without sources; "
                               "cannot differentiate")
        grad_payload = latest_k_backward(src, grad_values, ctx.chain)
    if grad_sum is not None:
        gs = seg_sum_backward(write_addresses, read_addresses, write_mask, grad_sum,
                              ctx.address_space)
        grad_payload = gs if grad_payload is None else grad_payload + gs
    return None, grad_payload, None, None, None, None, None


latest_k_sum.register_autograd(_latest_k_sum_grad, setup_context=_latest_k_sum_setup)


# ------------------------------------------- latest-k with its own tape --


def _tape_dtype(address_space: int) -> torch.dtype:
    """Storage type of a merged tape (the kernels' unsigned kind of that size)."""
    if address_space < 1 << 16:
        return torch.int16
    return torch.int32 if address_space < 1 << 32 else torch.int64


def latest_k_taped_impl(
    write_addresses: Tensor,
    payloads: Tensor,
    read_addresses: Optional[Tensor],
    write_mask: Optional[Tensor],
    address_space: int,
    k: int,
) -> Tuple[Tensor, Tensor, Tensor]:
    """latest_k for a training step with separate reads or a write mask: values,
    mask and the compact tape of its reads and writes ([B, 2T, C]), from which
    the backward sorts again.  The tape is a copy, so the addresses may change
    between the passes, and smaller than k sources a record."""
    lib = nat.library()
    B, T, C = write_addresses.shape
    values, mask, _ = latest_k_impl(write_addresses, payloads, read_addresses, write_mask,
                                    address_space, k, False)
    tape = torch.empty(B, 2 * T, C, dtype=_tape_dtype(address_space), device=payloads.device)
    _call(
        lib.ravel_em_tape, nat.ptr(write_addresses), nat.ptr(read_addresses),
        nat.addr_code(write_addresses.dtype), nat.ptr(write_mask), B, T, C, address_space,
        nat.ptr(tape), nat.stream_of(payloads),
    )
    return values, mask, tape


@torch.library.custom_op("ravel_em::latest_k_taped", mutates_args=())
def latest_k_taped(
    write_addresses: Tensor,
    payloads: Tensor,
    read_addresses: Optional[Tensor],
    write_mask: Optional[Tensor],
    address_space: int,
    k: int,
) -> Tuple[Tensor, Tensor, Tensor]:
    return latest_k_taped_impl(write_addresses, payloads, read_addresses, write_mask,
                               address_space, k)


@latest_k_taped.register_fake
def _latest_k_taped_fake(write_addresses, payloads, read_addresses, write_mask, address_space, k):
    B, T, C = write_addresses.shape
    return (
        payloads.new_empty(B, T, C, k, payloads.shape[-1]),
        torch.empty(B, T, C, k, dtype=torch.bool, device=payloads.device),
        torch.empty(B, 2 * T, C, dtype=_tape_dtype(address_space), device=payloads.device),
    )


def _latest_k_taped_setup(ctx, inputs, output):
    _, mask, tape = output
    ctx.save_for_backward(tape)
    ctx.address_space, ctx.k = inputs[4], inputs[5]
    ctx.mark_non_differentiable(mask, tape)
    ctx.set_materialize_grads(False)


def _latest_k_taped_grad(ctx, grad_values, _grad_mask, _grad_tape):
    (tape,) = ctx.saved_tensors
    if grad_values is None:
        return (None,) * 6
    grad_payload = latest_k_sum_backward(tape, None, None, grad_values, None, ctx.address_space,
                                         ctx.k, True)
    return None, grad_payload, None, None, None, None


latest_k_taped.register_autograd(_latest_k_taped_grad, setup_context=_latest_k_taped_setup)


# ------------------------------------------------- eager training calls --
#
# The same forwards and backwards as torch.autograd.Functions, for plain eager
# calls (eager_graph()): the dispatcher and the custom ops' autograd wrapper cost
# some 90 us of host time a training step (bf16 latest-4 of 262k records, whose
# kernels take 46 us: 151 us a step through the ops).  Their backwards go through
# the custom ops where a graph of the gradient itself is recorded (no op has a
# second derivative: it raises then, as before) or the gradient is no plain tensor.


def direct(op, impl, *grads: Optional[Tensor]):
    """impl where a backward may call it directly, else the custom op."""
    return impl if not torch.is_grad_enabled() and eager_graph(*grads) else op


class LatestKFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, payloads, write_addresses, read_addresses, write_mask, address_space, k):
        ctx.chain = read_addresses is None and write_mask is None
        B, T, C, D = payloads.shape
        ctx.taped = not ctx.chain and joint_backward_applies(T, C, D, k, payloads.element_size())
        if ctx.taped:
            values, mask, saved = latest_k_taped_impl(write_addresses, payloads, read_addresses,
                                                      write_mask, address_space, k)
        else:
            values, mask, saved = latest_k_impl(write_addresses, payloads, read_addresses,
                                                write_mask, address_space, k, True)
        ctx.save_for_backward(saved)
        ctx.args = (address_space, k)
        ctx.mark_non_differentiable(mask)
        ctx.set_materialize_grads(False)
        return values, mask

    @staticmethod
    def backward(ctx, grad_values, _grad_mask):
        (saved,) = ctx.saved_tensors
        if grad_values is None:
            return (None,) * 6
        if ctx.taped:
            g = direct(latest_k_sum_backward, latest_k_sum_backward_impl, grad_values)(
                saved, None, None, grad_values, None, *ctx.args, True)
        else:
            g = direct(latest_k_backward, latest_k_backward_impl, grad_values)(
                saved, grad_values, ctx.chain)
        return g, None, None, None, None, None


def kept_keys(payloads, read_addresses, write_mask, address_space, k) -> Optional[Tensor]:
    """Room for the sorted keys that a training forward keeps for its backward
    (None where the forward of the shape sorts nothing that the backward uses):
    4 or 8 bytes a record, twice that with separate reads or a mask."""
    B, T, C, D = payloads.shape
    n = nat.library().ravel_em_tape_keys_bytes(
        B, T, C, D, address_space, k, int(read_addresses is not None), int(write_mask is not None),
        nat.payload_code(payloads.dtype))
    return torch.empty(n, dtype=torch.uint8, device=payloads.device) if n else None


class SegSumFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, payloads, write_addresses, read_addresses, write_mask, address_space):
        keys = kept_keys(payloads, read_addresses, write_mask, address_space, 1)
        out, mask = seg_sum_impl(write_addresses, payloads, read_addresses, write_mask,
                                 address_space, keys)
        ctx.save_for_backward(write_addresses, read_addresses, write_mask, keys)
        ctx.address_space = address_space
        ctx.mark_non_differentiable(mask)
        ctx.set_materialize_grads(False)
        return out, mask

    @staticmethod
    def backward(ctx, grad_sum, _grad_mask):
        *tape, keys = ctx.saved_tensors
        if grad_sum is None:
            return (None,) * 5
        fn = direct(seg_sum_backward, seg_sum_backward_impl, grad_sum)
        if keys is not None and fn is seg_sum_backward_impl:
            g = latest_k_sum_backward_impl(keys, None, None, None, grad_sum, ctx.address_space, 1,
                                           False, _keys_code(tape))
        else:
            g = fn(*tape, grad_sum, ctx.address_space)
        return g, None, None, None, None


def _keys_code(tape) -> int:
    return nat.KEYS_SAME if tape[1] is None and tape[2] is None else nat.KEYS


class LatestKSumFn(torch.autograd.Function):
    """For the shapes of joint_backward_applies()."""

    @staticmethod
    def forward(ctx, payloads, write_addresses, read_addresses, write_mask, address_space, k):
        keys = kept_keys(payloads, read_addresses, write_mask, address_space, k)
        values, mask, _, out, smask = latest_k_sum_impl(write_addresses, payloads, read_addresses,
                                                        write_mask, address_space, k, False, keys)
        ctx.save_for_backward(write_addresses, read_addresses, write_mask, keys)
        ctx.args = (address_space, k)
        ctx.mark_non_differentiable(mask, smask)
        ctx.set_materialize_grads(False)
        return values, mask, out, smask

    @staticmethod
    def backward(ctx, grad_values, _grad_mask, grad_sum, _grad_smask):
        *tape, keys = ctx.saved_tensors
        if grad_values is None and grad_sum is None:
            return (None,) * 6
        fn = direct(latest_k_sum_backward, latest_k_sum_backward_impl, grad_values, grad_sum)
        if keys is not None and fn is latest_k_sum_backward_impl:
            g = fn(keys, None, None, grad_values, grad_sum, *ctx.args, False, _keys_code(tape))
        else:
            g = fn(*tape, grad_values, grad_sum, *ctx.args, False)
        return g, None, None, None, None, None


# ------------------------------------------------------- direct C calls --


def sort_order(write_addresses: Tensor, write_mask: Optional[Tensor], address_space: int,
               key_dtype: torch.dtype) -> Tuple[Tensor, Tensor]:
    """(sorted_keys, order) exactly as torch.sort of the reference's flat keys."""
    lib = nat.library()
    B, T, C = write_addresses.shape
    dev = write_addresses.device
    n_valid = B * T * C if write_mask is None else C * int(write_mask.sum().item())
    keys = torch.empty(n_valid, dtype=key_dtype, device=dev)
    order = torch.empty(n_valid, dtype=torch.int64, device=dev)
    if n_valid == 0:
        return keys, order
    nbytes = lib.ravel_em_sort_order_workspace(B, T, C, address_space, int(write_mask is not None))
    ws = nat.workspace(nbytes, dev)
    _call(
        lib.ravel_em_sort_order,
        nat.ptr(write_addresses), nat.addr_code(write_addresses.dtype), nat.ptr(write_mask),
        B, T, C, address_space, nat.ptr(keys), nat.ptr(order), nat.ptr(ws), ws.numel(),
        nat.stream_of(write_addresses),
    )
    nat.after_call(ws)
    return keys, order


def cache_read(values: Tensor, filled: Tensor, addresses: Tensor, k: int) -> Tuple[Tensor, Tensor]:
    lib = nat.library()
    B, C, A = filled.shape[:3]
    D = values.shape[-1]
    out = values.new_empty(B, C, k, D)
    mask = torch.empty(B, C, k, dtype=torch.bool, device=values.device)
    _call(
        lib.ravel_em_cache_read,
        nat.ptr(values), nat.ptr(filled), nat.ptr(addresses), nat.addr_code(addresses.dtype),
        nat.payload_code(values.dtype), B, C, A, k, D, nat.ptr(out), nat.ptr(mask),
        nat.stream_of(values),
    )
    return out, mask


def cache_write(values: Tensor, filled: Tensor, addresses: Tensor, payloads: Tensor, k: int) -> None:
    lib = nat.library()
    B, C, A = filled.shape[:3]
    D = values.shape[-1]
    _call(
        lib.ravel_em_cache_write,
        nat.ptr(values), nat.ptr(filled), nat.ptr(addresses), nat.addr_code(addresses.dtype),
        nat.ptr(payloads), nat.payload_code(values.dtype), B, C, A, k, D, nat.stream_of(values),
    )


def cache_step(values: Tensor, filled: Tensor, read_addresses: Tensor, write_addresses: Tensor,
               payloads: Tensor, k: int) -> Tuple[Tensor, Tensor]:
    lib = nat.library()
    B, C, A = filled.shape[:3]
    D = values.shape[-1]
    out = values.new_empty(B, C, k, D)
    mask = torch.empty(B, C, k, dtype=torch.bool, device=values.device)
    _call(
        lib.ravel_em_cache_step,
        nat.ptr(values), nat.ptr(filled), nat.ptr(read_addresses), nat.ptr(write_addresses),
        nat.addr_code(read_addresses.dtype), nat.ptr(payloads), nat.payload_code(values.dtype),
        B, C, A, k, D, nat.ptr(out), nat.ptr(mask), nat.stream_of(values),
    )
    return out, mask


def cache_prefill(write_addresses: Tensor, payloads: Tensor, write_mask: Optional[Tensor],
                  address_space: int, k: int, values: Tensor, filled: Tensor) -> None:
    lib = nat.library()
    B, T, C = write_addresses.shape
    D = payloads.shape[-1]
    dev = payloads.device
    nbytes = lib.ravel_em_cache_prefill_workspace(B, T, C, address_space, int(write_mask is not None))
    ws = nat.workspace(nbytes, dev)
    _call(
        lib.ravel_em_cache_prefill,
        nat.ptr(write_addresses), nat.addr_code(write_addresses.dtype), nat.ptr(write_mask),
        nat.ptr(payloads), nat.payload_code(payloads.dtype), B, T, C, D, address_space, k,
        nat.ptr(values), nat.ptr(filled), nat.ptr(ws), ws.numel(), nat.stream_of(payloads),
    )
    nat.after_call(ws)
