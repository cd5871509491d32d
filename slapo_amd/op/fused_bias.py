"""Bias epilogues fused with the following activation / dropout, on hand-written HIP kernels.

Same public names and call signatures as the reference's slapo/op/fused_bias.py
(`BiasGeLUFunction` :13-46, `new_gelu` :49-60, `bias_new_gelu` :63-64, `bias_dropout` :67-74); each runs as ONE
streaming kernel per direction instead of a TorchScript / functorch fusion.  Two modules,
`HipBiasGeLU` and `HipBiasDropoutResidual`, package them with the positional signatures
(`forward(x, bias)`, `forward(x, bias, residual)`) that `sch.replace(module, subgraph)` needs
for the fusion patterns of tests/test_fusion.py:118-204.
"""
from __future__ import annotations

import torch
from torch import nn

from .._lib import host
from ..random import draw_philox_state
from ._tracing import record, tracing_state


def bias_gelu(inp: torch.Tensor, bias: torch.Tensor) -> torch.Tensor:
    """gelu_tanh(inp + bias); backward is the closed form of fused_bias.py:26-34 and returns the
    bias gradient already reduced to the bias shape."""
    if tracing_state() is not None:
        return record(bias_gelu, inp, bias)
    return host().bias_gelu(inp, bias)


class BiasGeLUFunction(torch.autograd.Function):
    """The reference's name for `bias_gelu`: `BiasGeLUFunction.apply(inp, bias)`."""

    # pylint: disable=abstract-method
    apply = staticmethod(bias_gelu)


def new_gelu(inp: torch.Tensor) -> torch.Tensor:
    """HF `gelu_new` (fused_bias.py:49-60) as one kernel per direction."""
    if tracing_state() is not None:
        return record(new_gelu, inp)
    return host().bias_gelu(inp, None)


def bias_new_gelu(inp: torch.Tensor, bias: torch.Tensor) -> torch.Tensor:
    """HF `gelu_new` on inp + bias.  Its constant sqrt(2/pi) equals the 0.79788456 of
    `BiasGeLUFunction` to 8 digits, so both names share one kernel."""
    return bias_gelu(inp, bias)


def _draw(x, p):
    """(seed, offset, state) of the mask F.dropout(x, p) would draw; the generator moves exactly as
    it would there.  Nothing is drawn for p of 0 or 1, nor for an empty tensor."""
    n = x.numel()
    if not 0.0 < p < 1.0 or n == 0 or not x.is_cuda:
        return 0, 0, None
    return draw_philox_state(host().philox_increment(n, x.element_size(), x.device.index),
                             x.device)


def bias_dropout(x: torch.Tensor, bias: torch.Tensor, p: float = 0.5, training: bool = True,
                 inplace: bool = False) -> torch.Tensor:
    """dropout(x + bias).  `inplace` is accepted for signature compatibility; the reference's
    in-place target is the temporary x + bias, which this kernel never materialises."""
    del inplace
    if tracing_state() is not None:
        return record(bias_dropout, x, bias, p, training)
    _check_p(p)
    p = p if training else 0.0
    return host().bias_dropout_residual(x, bias, None, p, *_draw(x, p))


def bias_dropout_residual(x: torch.Tensor, bias: torch.Tensor, residual: torch.Tensor,
                          p: float = 0.5, training: bool = True) -> torch.Tensor:
    """dropout(x + bias) + residual, the pattern of tests/test_fusion.py:179-180."""
    if tracing_state() is not None:
        return record(bias_dropout_residual, x, bias, residual, p, training)
    _check_p(p)
    p = p if training else 0.0
    return host().bias_dropout_residual(x, bias, residual, p, *_draw(x, p))


def bias_dropout_residual_layer_norm(x: torch.Tensor, bias, residual, weight: torch.Tensor,
                                     ln_bias: torch.Tensor, p: float = 0.5, eps: float = 1e-5,
                                     training: bool = True) -> torch.Tensor:
    """layer_norm(dropout(x + bias) + residual) over the last dimension, the pattern of
    tests/test_fusion.py:184-185 (bias and residual may be None)."""
    if tracing_state() is not None:
        return record(bias_dropout_residual_layer_norm, x, bias, residual, weight, ln_bias, p, eps,
                      training)
    _check_p(p)
    p = p if training else 0.0
    return host().bias_dropout_residual_layer_norm(x, bias, residual, weight, ln_bias, eps, p,
                                                   *_draw(x, p))


def _check_p(p):
    if p < 0.0 or p > 1.0:
        raise ValueError(f"dropout probability has to be between 0 and 1, but got {p}")


class HipBiasGeLU(nn.Module):
    """Replacement payload for a matched `gelu(x + bias)` subgraph."""

    def forward(self, x, bias):
        return bias_gelu(x, bias)


class HipBiasDropoutResidual(nn.Module):
    """Replacement payload for a matched `dropout(x + bias) + residual` subgraph."""

    def __init__(self, p: float = 0.5):
        super().__init__()
        _check_p(p)
        self.p = p

    def forward(self, x, bias, residual):
        return bias_dropout_residual(x, bias, residual, self.p, self.training)

    def extra_repr(self):
        return f"p={self.p}"


class HipBiasDropoutResidualLayerNorm(nn.Module):
    """Replacement payload for a matched `layer_norm(dropout(x + bias) + residual)` subgraph;
    owns the LayerNorm parameters under the names of `nn.LayerNorm` (`weight`, `bias`)."""

    def __init__(self, normalized_shape: int, p: float = 0.5, eps: float = 1e-5, device=None,
                 dtype=None):
        super().__init__()
        _check_p(p)
        if not isinstance(normalized_shape, int):
            if len(normalized_shape) != 1:
                raise NotImplementedError("only the last dimension can be normalized")
            normalized_shape = int(normalized_shape[0])
        self.normalized_shape = (normalized_shape,)
        self.p, self.eps = p, eps
        self.weight = nn.Parameter(torch.ones(normalized_shape, device=device, dtype=dtype))
        self.bias = nn.Parameter(torch.zeros(normalized_shape, device=device, dtype=dtype))

    @classmethod
    def from_layer_norm(cls, ln: nn.LayerNorm, p: float):
        """Takes over the parameters of an existing nn.LayerNorm (shared, not copied)."""
        if not ln.elementwise_affine or ln.bias is None:
            raise NotImplementedError("LayerNorm without affine parameters")
        mod = cls(ln.normalized_shape, p, ln.eps, device=ln.weight.device, dtype=ln.weight.dtype)
        mod.weight, mod.bias = ln.weight, ln.bias
        return mod

    def forward(self, x, bias, residual):
        return bias_dropout_residual_layer_norm(x, bias, residual, self.weight, self.bias,
                                                self.p, self.eps, self.training)

    def extra_repr(self):
        return f"{self.normalized_shape}, p={self.p}, eps={self.eps}"
