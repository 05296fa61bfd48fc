"""What of autograd a native kernel cannot serve.  The kernels read tensors by address and record
nothing, so a call whose tensors carry a forward-mode tangent, or stand for other tensors inside
a functorch transform, belongs to stock, and so does a backward that is to be differentiated
again or runs over batched or dual gradients.  Both questions are asked on every call: the
answer no costs about 0.1 us."""
from __future__ import annotations

import torch
import torch.autograd.forward_ad as _forward_ad

_transforming = torch._C._are_functorch_transforms_active
_wrapped = torch._C._functorch.is_functorch_wrapped_tensor
_grad_enabled = torch.is_grad_enabled


def _dual(tensors) -> bool:
    return any(isinstance(t, torch.Tensor) and _forward_ad.unpack_dual(t).tangent is not None for t in tensors)


def transformed(*tensors) -> bool:
    """True when one of `tensors` (None and other values pass) carries a forward-mode tangent or is
    a functorch wrapper (vmap, jvp, grad)."""
    if _forward_ad._current_level < 0 and not _transforming():
        return False
    if any(isinstance(t, torch.Tensor) and _wrapped(t) for t in tensors):
        return True
    return _forward_ad._current_level >= 0 and _dual(tensors)


def graph_wanted(grad_output, *saved) -> bool:
    """In a backward: True when the gradients must come from differentiable ops -- they are to be
    differentiated again (create_graph=True), or the incoming gradient is batched
    (is_grads_batched=True, vmap) or carries a tangent."""
    if _grad_enabled() and any(t is not None and t.requires_grad for t in (grad_output, *saved)):
        return True
    try:
        grad_output.data_ptr()
    except RuntimeError:  # a batched tensor has no storage of its own
        return True
    return _forward_ad._current_level >= 0 and _dual((grad_output, *saved))
