"""int8_linear_forward / int8_linear_backward on top of the BlockQuantizeCUDA extension.

Data format everywhere: codes int8 [..., R, C] with one scale per 32x32 tile, scales [..., R/32, C/32]
(float16 as in the reference, float32 accepted).  The GEMM entry points take their scale operands as [K/32, rows/32];
the reference makes transposed copies for that (linear_fwd.py:17-18, linear_bwd.py:11), here the kernel reads the block
tensor's own scale array in place, and no bias is no operand (the reference allocates a zero bias on every call,
linear_fwd.py:20-21).  The weight-gradient GEMM reads the gradient
[tokens, C_out] in place as its [K, M] operand when no pre-transposed copy is supplied (G8T=None); the reference needs
the copy (linear_bwd.py:21, made by int8_transpose / int8_quantize_transpose).

Bias (sketched in the reference, JetfireGEMMKernel/BlockQuantize/QBlockLinear.py:38-39, 63-66; its recipe runs without):
`bias=` of the forward functions is added to the accumulator in the kernel's requantising epilogue with
biasmax = max|bias| added to the block absmax (…BiasRowCol.cu:313,357); `bias_grad=True` of the backward functions
also returns the bias gradient, the column sums of the (dequantised) output gradient.

Every function here is one call of the C++ extension (BlockQuantizeCUDA.jetfire), which reads the leading dimensions,
validates, allocates and enqueues: the views and reshapes this took in Python were most of a small call's time.
"""
import os
import sys

import torch

_PKG = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import BlockQuantizeCUDA as BQC  # noqa: E402

_jf = BQC.jetfire       # GEMMs with fused epilogues, column sums


def bias_operands(bias, n_out, device):
    """(bias as contiguous float32 [N], biasmax = max|bias| as float32 [1]) for the kernel; no pair for None."""
    if bias is None:
        return None, None
    if bias.numel() != n_out:
        raise RuntimeError(f"bias must have {n_out} elements, got {bias.numel()}")
    b = bias.detach().reshape(-1).to(torch.float32).contiguous()
    return b, b.abs().max().reshape(1)


def _bias_pair(bias, n_out, device):
    """bias may already be the (bias, biasmax) pair (a caller that caches it per parameter version)."""
    if isinstance(bias, tuple):
        return bias
    return bias_operands(bias, n_out, device)


def _check_block(B):
    if B != 32:
        raise RuntimeError(f"the INT8 GEMM kernels use 32x32 quantisation blocks, got B={B}")


def int8_linear_forward(X8_3D, SX16_3D, W8, SW16, output_quantized, B, bias=None):
    """Y = X W^T (+ bias).  X8 [BS,T,K] (or [M,K]), SX [BS,T/32,K/32]; W8 [N,K], SW [N/32,K/32]; bias [N] or None.
    Returns (O8 [BS,T,N], SO [BS,T/32,N/32]) or, with output_quantized=False, the dequantised
    output in the scale dtype (reference: linear_fwd.py:4-32; bias: QBlockLinear.py:38-39)."""
    _check_block(B)
    b, bmax = (None, None) if bias is None else _bias_pair(bias, W8.shape[0], W8.device)
    # unquantised: the quantising GEMM and the codes x scales product of the reference (linear_fwd.py:22-31) in one kernel
    o, so = _jf.linear_forward(X8_3D, SX16_3D, W8, SW16, bool(output_quantized), b, bmax)
    return (o, so) if output_quantized else o


def int8_linear_forward_gelu(X8_3D, SX16_3D, W8, SW16, B, approximate="none", bias=None):
    """int8_linear_forward(..., output_quantized=True) followed by int8_gelu_forward, in one kernel (no counterpart in
    the reference, whose MLP runs the two back to back, qmodel.py:210-214).  Returns (O8, SO, G8, SG): the linear
    output (kept for the backward pass) and its GELU (the next layer's input), bit-identical to the two separate calls."""
    _check_block(B)
    if approximate not in ("none", "tanh"):
        raise RuntimeError("approximate must be 'none' or 'tanh'")
    b, bmax = (None, None) if bias is None else _bias_pair(bias, W8.shape[0], W8.device)
    tanh = approximate == "tanh"
    # (the threshold as in Nonlinear.int8_gelu_forward)
    return _jf.linear_forward_gelu(X8_3D, SX16_3D, W8, SW16, _jf.GELU_TANH if tanh else _jf.GELU_ERF, 0.0 if tanh else 5e-5, b, bmax)


def int8_linear_backward(X8_3D, SX16_3D, G8_3D, SG16_3D, G8T, W8, SW16, B, stochastic=True, dgrad_quantize=True,
                         wgrad_splitk=1, wgrad_dtype=None, bias_grad=False):
    """dX = dY W (requantised with stochastic rounding) and dW = dY^T X (fp16).
    G8 [BS,T,N] with SG [BS,T/32,N/32]; G8T = G8 transposed to [N, BS*T], or None (then G8 itself is read, no copy);
    W8 [N,K], SW [N/32,K/32].
    Returns (GX8, GSX, GW) or (GX_fp, GW) when dgrad_quantize=False (reference: linear_bwd.py:4-29; like
    there, the activation gradient is always rounded stochastically).  wgrad_splitk (not in the reference): 1 = its
    arithmetic; 0 = let the library cut K into ordered partial sums when dW has too few tiles to fill the GPU.
    wgrad_dtype (not in the reference): None = float16 as there; float32 / bfloat16 = dW leaves the kernel in that type.
    bias_grad=True appends the bias gradient (float32 [N], the column sums of G8 x SG; QBlockLinear.py:63-66)."""
    _check_block(B)
    return tuple(_jf.linear_backward(X8_3D, SX16_3D, G8_3D, SG16_3D, G8T, W8, SW16, dgrad_quantize, wgrad_splitk, wgrad_dtype, bias_grad))


def int8_linear_backward_gelu(X8_3D, SX16_3D, G8_3D, SG16_3D, W8, SW16, PRE8_3D, SPRE16_3D, B, approximate="none",
                              stochastic=True, wgrad_splitk=1, wgrad_dtype=None, bias_grad=False):
    """int8_linear_backward(...) followed by int8_gelu_backward(PRE8, SPRE, <its activation gradient>, ...), with the
    GELU backward running in the epilogue of the activation-gradient GEMM (no counterpart in the reference, whose MLP
    backward runs the two back to back, qmodel.py:249-253).  X8 / SX: the linear layer's input (= the GELU's output),
    PRE8 / SPRE: the GELU's input; G8 [BS,T,N], W8 [N,K].  Returns (GPRE8, GSPRE, GW): the gradient with respect to the
    GELU's input, requantised (`stochastic` as in int8_gelu_backward), and the weight gradient; bit-identical to the
    two separate calls (which draw their rounding noise in the same order)."""
    _check_block(B)
    if approximate not in ("none", "tanh"):
        raise RuntimeError("approximate must be 'none' or 'tanh'")
    return tuple(_jf.linear_backward_gelu(X8_3D, SX16_3D, G8_3D, SG16_3D, W8, SW16, PRE8_3D, SPRE16_3D,
                                          _jf.GELU_TANH if approximate == "tanh" else _jf.GELU_ERF,
                                          _jf.ROUND_STOCHASTIC if stochastic else _jf.ROUND_NEAREST, wgrad_splitk, wgrad_dtype, bias_grad))
