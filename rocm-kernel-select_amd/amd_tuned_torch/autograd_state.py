"""What of autograd a native kernel cannot serve.  The kernels read tensors by address and record
nothing, so a call whose tensors carry a forward-mode tangent, or stand for other tensors inside
a functorch transform, belongs to stock, and so does a backward that is to be differentiated
again or runs over batched or dual gradients."""
from __future__ import annotations

import torch
import torch.autograd.forward_ad as _forward_ad

_functorch = torch._C._functorch


def transformed(*tensors) -> bool:
    """True when one of `tensors` (None and other values pass) carries a forward-mode tangent or is
    a functorch wrapper (vmap, jvp, grad).  Outside a forward-mode level and a transform this is
    two reads, about 0.15 us."""
    if _forward_ad._current_level < 0 and _functorch.peek_interpreter_stack() is None:
        return False
    for t in tensors:
        if isinstance(t, torch.Tensor) and (
                _functorch.is_functorch_wrapped_tensor(t)
                or (_forward_ad._current_level >= 0 and _forward_ad.unpack_dual(t).tangent is not None)):
            return True
    return False


def graph_wanted(grad_output, *saved) -> bool:
    """In a backward: True when the gradients must come from differentiable ops -- they are to be
    differentiated again (create_graph=True), or the incoming gradient is batched
    (is_grads_batched=True) or carries a tangent."""
    if torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in (grad_output, *saved)):
        return True
    return _functorch.is_legacy_batchedtensor(grad_output) or transformed(grad_output, *saved)
