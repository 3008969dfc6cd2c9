"""Quantized-GEMM operators with the interface of flashnn/quant_gemm.py.

DynamicQuantize, GemmA8W8 and GemmWeightOnly keep the reference's constructor and forward
signatures, return types and error behaviour.  `_hip_impl` runs the gfx950 kernels;
`_torch_impl` is the plain torch formula, selected only by set_use_triton(False).
"""
import torch

from . import torch_formulas
from .kernel_backend import BackendKernel
from .launchers import (_check_dynamic_quantize, _check_weight_only, _dynamic_quantize, _weight_only, hip_a16w4_prepack,
                        hip_gemm_a8w8_forward, hip_gemm_a16w4_prepacked_forward)


def _weight_type(quant_w, scale_w):
    rows, channels = quant_w.size(0), scale_w.size(-1)
    if rows * 2 == channels:
        return torch.quint4x2
    if rows == channels:
        return torch.int8
    return None


class DynamicQuantize(BackendKernel):
    """Per-token dynamic quantization (flashnn/quant_gemm.py:39-66).
    input fp16/bf16 [M,K] -> (int8 [M,K], fp16 scale [M])."""

    def __init__(self):
        super().__init__()

    def _torch_impl(self, input):
        out, scale = torch_formulas.rows_to_int8(input)
        return out, scale.half().squeeze(-1)

    def _hip_impl(self, input):
        out = torch.empty(input.shape, dtype=torch.int8, device=input.device)
        scale = torch.empty(input.shape[0], dtype=torch.half, device=input.device)
        _check_dynamic_quantize(input)
        return _dynamic_quantize(out, input, scale)

    def forward(self, input):
        return BackendKernel.forward(self, input)


class GemmA8W8(BackendKernel):
    """out <- (int8 A[m,k] x int8 B[n,k]^T) * (scale_row[m,1] * scale_col[1,n])
    (flashnn/quant_gemm.py:69-107)."""

    def __init__(self, out_ty: torch.dtype = torch.float16):
        super().__init__()
        self.out_ty = out_ty

    def _hip_impl(self, a, b, alpha_row, alpha_col):
        out = torch.empty([a.shape[0], b.shape[0]], dtype=self.out_ty, device=a.device)
        hip_gemm_a8w8_forward(out, a, b, alpha_row, alpha_col)
        return out

    def _torch_impl(self, a, b, alpha_row, alpha_col):
        return torch_formulas.a8w8(a, b, alpha_row, alpha_col, self.out_ty)

    def forward(self, a, b, alpha_row, alpha_col):
        return BackendKernel.forward(self, a, b, alpha_row, alpha_col)


class GemmWeightOnly(BackendKernel):
    """Weight-only quantized GEMM, int8 or packed int4 weights (flashnn/quant_gemm.py:110-209)."""

    def __init__(self, out_ty: torch.dtype = torch.float16):
        super().__init__()
        self.out_ty = out_ty

    def _hip_impl(self, act, quant_w, scale_w, bias=None, zero_points=None):
        _check_weight_only(act, quant_w)
        weight_type = _weight_type(quant_w, scale_w)
        if weight_type == torch.int8:
            entry, channels = "fnn_gemm_a16w8", quant_w.shape[0]
        elif weight_type == torch.quint4x2:
            entry, channels = "fnn_gemm_a16w4", quant_w.shape[0] * 2
        else:
            raise AssertionError("Gemm WeightOnly only support int8 or int4x2")
        out = torch.empty((act.shape[0], channels), dtype=self.out_ty, device=act.device)
        return _weight_only(entry, out, act, quant_w, scale_w, bias, zero_points, channels)

    def _torch_impl(self, act, quant_w, scale_w, bias=None, zero_points=None):
        assert act.shape[1] == quant_w.shape[1], "Matrix B must be transposed"
        weight_type = _weight_type(quant_w, scale_w)
        if weight_type == torch.int8:
            w = quant_w.t()
        elif weight_type == torch.quint4x2:
            w = torch_formulas.unpack_int4_rows(quant_w)
        else:
            raise AssertionError("Gemm WeightOnly only support int8 or int4x2")
        return torch_formulas.weight_only(act, w, scale_w, bias, zero_points, self.out_ty,
                                          round_before_bias=weight_type == torch.int8)

    def forward(self, act, quant_w, scale_w, bias=None, zero_points=None):
        return BackendKernel.forward(self, act, quant_w, scale_w, bias, zero_points)

    @staticmethod
    def prepack(quant_w, scale_w, zero_points=None):
        """int4 weights with fp16 tables per group of 128, repacked once into the stream the decode
        kernels of forward_prepacked read (not in the reference: its launcher reads [N/2, K] as it is,
        flashnn/triton_kernels/gemm_a16w4.py:336-406).  Explicit: forward never repacks."""
        return hip_a16w4_prepack(quant_w, scale_w, zero_points)

    def forward_prepacked(self, act, packed, bias=None):
        """forward on weights from prepack(); HIP path only."""
        out = torch.empty([act.shape[0], packed.n], dtype=self.out_ty, device=act.device)
        return hip_gemm_a16w4_prepacked_forward(out, act, packed, bias=bias)
