"""When the quantizer's tensor expressions run as one device kernel (csrc/quantize.hip) instead."""
from __future__ import annotations

import torch


def takes_kernel(t: torch.Tensor) -> bool:
    """True for an ordinary tensor on the GPU that nothing observes: no subclass, no gradient or tangent to carry, no
    negation still to be done (torch's negative views), no vmap / tracing / dispatch mode that has to see the tensor
    operations. Everything else takes the expressions."""
    return (t.is_cuda and t.numel() > 0 and type(t) in (torch.Tensor, torch.nn.Parameter) and not t.is_neg()
            and not (t.requires_grad and torch.is_grad_enabled())
            and torch.autograd.forward_ad._current_level < 0
            and not torch._C._functorch.is_functorch_wrapped_tensor(t)
            and torch._C._len_torch_dispatch_stack() == 0 and torch._C._len_torch_function_stack() == 0
            and not torch.compiler.is_compiling() and not torch.jit.is_tracing())
