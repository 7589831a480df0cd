"""``nn.Linear`` drop-in on the HIP GEMM (reference: qwen_triton/modules/linear.py:11-34)."""
from __future__ import annotations

import math

import torch
from torch import nn

from qwen_triton.kernels.matmul import triton_matmul


def plain_linears(*modules: nn.Module) -> bool:
    """True when calling each module does nothing but its product: no subclass, replaced ``forward``
    or forward hook that a launch from the weights alone would leave out."""
    hooks = nn.modules.module
    if hooks._global_forward_hooks or hooks._global_forward_pre_hooks or TritonLinear.forward is not _FORWARD:
        return False
    return all(
        type(m) is TritonLinear and "forward" not in m.__dict__ and not m._forward_hooks and not m._forward_pre_hooks
        for m in modules)


class TritonLinear(nn.Module):
    def __init__(self, in_features: int, out_features: int, bias: bool = True) -> None:
        super().__init__()
        self.in_features = in_features
        self.out_features = out_features
        self.weight = nn.Parameter(torch.empty(out_features, in_features))
        if bias:
            self.bias = nn.Parameter(torch.empty(out_features))
        else:
            self.register_parameter("bias", None)
        self.reset_parameters()

    def reset_parameters(self) -> None:
        # Same distribution as nn.Linear: kaiming-uniform weight, U(+-1/sqrt(fan_in)) bias.
        nn.init.kaiming_uniform_(self.weight, a=math.sqrt(5))
        if self.bias is not None:
            bound = 1.0 / math.sqrt(self.in_features) if self.in_features > 0 else 0.0
            nn.init.uniform_(self.bias, -bound, bound)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return triton_matmul(x, self.weight, self.bias)

    def extra_repr(self) -> str:
        return f"in_features={self.in_features}, out_features={self.out_features}, bias={self.bias is not None}"


_FORWARD = TritonLinear.forward
