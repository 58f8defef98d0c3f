"""The DiT block's elementwise glue around attention, fused, on MI355X.

`ln_modulate(x, weight, shift, scale)` = modulate(LN(x), shift, scale) of
DiTBlock.forward (model/modules.py:537-568; LayerNorm :243-288, modulate
:778-788) in one pass; `gate_residual(x, gate, y)` = x + gate * y
(:560-566). Both follow the reference's eager dtypes (bf16 ops rounded op by
op, fp32 otherwise); gate_residual is bit-exact, ln_modulate differs from the
eager path only by the fp32 summation order of the row statistics.
Shapes: x, y (batch, seq, d_model); shift, scale, gate (batch, d_model) or
(batch, 1, d_model) (the AdaLN chunks); weight (d_model).
"""
from __future__ import annotations

import torch
from torch import Tensor

from kernels._native import host

_F = {torch.float32: 1, torch.bfloat16: 0}


def _out_flag(out_dtype: torch.dtype | None) -> int:
    return -1 if out_dtype is None else _F[out_dtype]


def ln_modulate(x: Tensor, weight: Tensor, shift: Tensor, scale: Tensor, eps: float = 1e-5,
                out_dtype: torch.dtype | None = None) -> Tensor:
    """modulate(LN(x), shift, scale). The result's dtype is the eager one
    (bf16 when x and the vectors are bf16, else fp32); out_dtype=bf16 rounds
    an fp32 result for the next matmul."""
    assert x.dim() == 3 and x.is_cuda, "x must be (batch, seq, d_model) on CUDA"
    return host().ln_modulate(x, weight, shift, scale, eps, _out_flag(out_dtype))


def gate_residual(x: Tensor, gate: Tensor, y: Tensor, out: Tensor | None = None) -> Tensor:
    """x + gate * y in the eager dtypes; `out=x` updates the residual in place."""
    assert x.dim() == 3 and x.shape == y.shape and x.is_cuda
    return host().gate_residual(x, gate, y, out)


def gate_residual_ln_modulate(x: Tensor, gate: Tensor, y: Tensor, weight: Tensor, shift: Tensor,
                              scale: Tensor, eps: float = 1e-5, out_dtype: torch.dtype | None = None,
                              x_out: Tensor | None = None) -> tuple[Tensor, Tensor]:
    """(x + gate * y, modulate(LN(x + gate * y), shift, scale)) in one launch,
    bit-exact with gate_residual followed by ln_modulate; `x_out=x` updates
    the residual in place."""
    assert x.dim() == 3 and x.shape == y.shape and x.is_cuda
    return host().gate_residual_ln_modulate(x, gate, y, weight, shift, scale, eps, _out_flag(out_dtype), x_out)
