"""FP8 W8A8 linear op, same contract as the reference's ``Fp8LinearOp``
(vllm/model_executor/layers/quantization/utils/w8a8_utils.py:390-491) with a single backend: the gfx950 fused
scaled GEMM, which covers per-tensor and per-token activations x per-tensor and per-channel weights."""
from __future__ import annotations

from collections.abc import Callable

import torch

from vllm_amd import _custom_ops as ops
from ..input_quant_fp8 import GroupShape, QuantFP8


def cutlass_w8a8_scaled_mm(*, qinput: torch.Tensor, weight: torch.Tensor, out_dtype: torch.dtype,
                           scale_a: torch.Tensor, scale_b: torch.Tensor, bias: torch.Tensor | None,
                           output_shape: list, **kwargs) -> torch.Tensor:
    """w8a8_utils.py:146-161: fused GEMM + dequant."""
    output = ops.cutlass_scaled_mm(qinput, weight, out_dtype=out_dtype, scale_a=scale_a, scale_b=scale_b, bias=bias)
    return output.view(*output_shape)


def dispatch_w8a8_scaled_mm(preferred_backend: str, per_tensor_weights: bool,
                            per_tensor_activations: bool) -> Callable[..., torch.Tensor]:
    """w8a8_utils.py:360-385: every scale combination maps onto the one fused kernel."""
    return cutlass_w8a8_scaled_mm


class Fp8LinearOp:
    def __init__(self, act_quant_static: bool, act_quant_group_shape: GroupShape = GroupShape.PER_TENSOR,
                 pad_output: bool | None = None):
        self.preferred_backend = "hip"
        self.output_padding = None      # padding is only useful to the torch._scaled_mm fallback, which does not exist here
        self.act_quant_static = act_quant_static
        self.act_quant_group_shape = act_quant_group_shape
        self.act_quant_per_token = act_quant_group_shape == GroupShape.PER_TOKEN
        self.quant_fp8 = QuantFP8(static=act_quant_static, group_shape=act_quant_group_shape,
                                  num_token_padding=self.output_padding)

    def apply(self, input: torch.Tensor, weight: torch.Tensor, weight_scale: torch.Tensor,
              out_dtype: torch.dtype | None = None, input_scale: torch.Tensor | None = None,
              input_scale_ub: torch.Tensor | None = None, bias: torch.Tensor | None = None) -> torch.Tensor:
        static, quant = self.act_quant_static, self.quant_fp8
        if input.dtype != ops.FP8_DTYPE and (input_scale is not None) == static and \
                (input_scale_ub is None if static else self.act_quant_per_token) and \
                not torch.compiler.is_dynamo_compiling() and type(quant) is QuantFP8 and quant.runs_forward_only():
            output = ops.fp8_linear(input, weight, weight_scale, input_scale, input_scale_ub, out_dtype or input.dtype, bias)
            if output is not None:
                return output
        input_2d = input.view(-1, input.shape[-1])
        output_shape = [*input.shape[:-1], weight.shape[1]]
        if out_dtype is None:
            out_dtype = input.dtype
        if input.dtype != ops.FP8_DTYPE:
            qinput, x_scale = self.quant_fp8(input_2d, input_scale, input_scale_ub)
        else:
            qinput, x_scale = input_2d, input_scale
        # a one-token per-token scale is [[s]] (dim 2), a per-tensor scale is [s] or () -- dim() tells them apart
        per_tensor_weights = (weight_scale.numel() == 1) and weight_scale.dim() < 2
        per_tensor_activations = (x_scale.numel() == 1) and x_scale.dim() < 2
        w8a8_scaled_mm_func = dispatch_w8a8_scaled_mm(self.preferred_backend, per_tensor_weights,
                                                      per_tensor_activations)
        return w8a8_scaled_mm_func(qinput=qinput, weight=weight, out_dtype=out_dtype, scale_a=x_scale,
                                   scale_b=weight_scale, bias=bias, output_shape=output_shape)
