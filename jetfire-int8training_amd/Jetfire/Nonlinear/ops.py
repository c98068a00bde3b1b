"""The Nonlinear operators: shape handling over the C++ extension (BlockQuantizeCUDA.jetfire, csrc/jf_ops_ext.cpp), which
validates the tensors, allocates the outputs and enqueues the gfx950 kernels through the C ABI with the GIL released.

All functions accept 2-D [M,N] or 3-D [BS,T,N] operands like the reference launchers and return tensors
of matching rank (the extension reads either, without views made here); scales are float16 [.., M/32, N/32] unless the inputs carry float32 scales.
Stochastic rounding draws its Philox (seed, offset) from the device's default torch generator, so it follows
torch.manual_seed (the reference materialises a uniform_(-0.5,0.5) noise tensor, quantize.py:143-146).
"""
import os
import sys

import torch

_PKG = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import BlockQuantizeCUDA as _BQC  # noqa: E402

_jf = _BQC.jetfire      # the operators below, as C++ functions on 2-D tensors

from .common import SCALE_MIN_THRES  # noqa: E402


def _check_qb(QB):
    if QB != 32:
        raise RuntimeError(f"quantisation block size must be 32, got {QB}")


class _Shape:
    """Remembers how to fold 2-D results back to the rank of the input."""

    def __init__(self, t):
        if t.dim() not in (2, 3):
            raise RuntimeError(f"expected a 2-D or 3-D tensor, got {t.dim()} dimensions")
        self.batched = t.dim() == 3
        self.bs = t.shape[0] if self.batched else None

    def fold(self, t):
        return t.reshape(self.bs, -1, t.shape[-1]) if self.batched else t


def _c(t):
    """The extension reads contiguous 2-D and 3-D operands as they are."""
    return t if t.is_contiguous() else t.contiguous()


def _f32(v):
    return v if v.dtype == torch.float32 and v.is_contiguous() else v.to(torch.float32).contiguous()


def int8_quantize(x, QB, stochastic=False, scale_dtype=torch.float16):
    """x fp32/fp16/bf16 -> (int8 codes, scales).  Reference: quantize.py:128-164."""
    _check_qb(QB)
    q, s, _ = _jf.quantize(_c(x), _jf.ROUND_STOCHASTIC if stochastic else _jf.ROUND_NEAREST, scale_dtype)
    return q, s


def int8_quantize_concat(xs, QB, stochastic=False, scale_dtype=torch.float16):
    """int8_quantize(torch.cat(xs, dim=-1), ...) without the concatenation (no counterpart in the reference, which
    quantises the concatenated gradient of the attention kernel's inputs, qmodel.py:112-120): every tensor of xs is
    quantised where it lies into its columns of the result.  Same codes, scales and noise as the two-step form."""
    _check_qb(QB)
    sh = _Shape(xs[0])
    flat = []
    for x in xs:
        if x.dim() != xs[0].dim() or x.shape[:-1] != xs[0].shape[:-1]:
            raise RuntimeError("tensors to concatenate must agree in all but the last dimension")
        f = x.reshape(-1, x.shape[-1])                             # a view whenever the leading dimensions can be merged
        in_place = (f.stride(1) == 1 and f.stride(0) >= f.shape[1]     # (an expanded gradient has row stride 0: copied)
                    and (f.stride(0) * f.element_size()) % 16 == 0 and f.data_ptr() % 16 == 0)
        flat.append(f if in_place else f.contiguous())
    q, s = _jf.quantize_slabs(flat, _jf.ROUND_STOCHASTIC if stochastic else _jf.ROUND_NEAREST, scale_dtype)
    return sh.fold(q), sh.fold(s)


def int8_quantize_transpose(x, QB, stochastic=False, transpose_output_2d=False, scale_dtype=torch.float16):
    """As int8_quantize, plus the transposed codes [N, M].  Reference: quantize_transpose.py:131-171."""
    _check_qb(QB)
    q, s, qt = _jf.quantize(_c(x), _jf.ROUND_STOCHASTIC if stochastic else _jf.ROUND_NEAREST, scale_dtype, True)
    if x.dim() == 3 and not transpose_output_2d:
        qt = qt.reshape(x.shape[0], -1, qt.shape[-1])
    return q, s, qt


def int8_transpose(x, transpose_output_2d=False):
    """int8 [M,N] -> [N,M] (3-D input is flattened over its leading dimensions first).  Reference: transpose.py:69-97."""
    y = _jf.transpose_s8(_c(x))
    if x.dim() == 3 and not transpose_output_2d:
        y = y.reshape(x.shape[0], -1, y.shape[-1])
    return y


def int8_dequantize(x, s_x, QB):
    """(codes, scales) -> float32.  Reference: dequantize.py:86-116."""
    _check_qb(QB)
    return _jf.dequantize(_c(x), _c(s_x), torch.float32)


def int8_rowstats(x, s_x, QB, eps=1e-5):
    """Per-row (mean, rstd) of a block tensor: the statistics int8_layernorm_forward consumes."""
    _check_qb(QB)
    return _jf.rowstats(_c(x), _c(s_x), eps)


def int8_layernorm_forward(x, sx, weight, mean, rstd, QB, eps=1e-6, bias=None):
    """dequant -> (x-mean)*rstd*weight (+bias) -> requant; returns (y, sy, (mean, rstd)).
    mean/rstd are per-row inputs as in the reference (layernorm.py:430-465, where `eps` is unused too);
    pass mean=None to have them computed from (x, sx) with this eps."""
    _check_qb(QB)
    x, sx = _c(x), _c(sx)
    if mean is None or rstd is None:
        mean, rstd = _jf.rowstats(x, sx, eps)
    qy, sy = _jf.layernorm_fwd(x, sx, _f32(weight), None if bias is None else _f32(bias), _f32(mean), _f32(rstd))
    return qy, sy, (mean, rstd)


def int8_layernorm_backward(x, sx, g, sg, w, QB, m, v, stochastic=False, eps=1e-6, return_dbias=False):
    """Returns (dx codes, dx scales, dweight[, dbias]).  m, v are the forward's (mean, rstd).
    Row reductions run over the full row (the reference reduces over its 128-column tile only,
    layernorm.py:331-332).  Reference launcher: layernorm.py:467-526."""
    _check_qb(QB)
    rounding = _jf.ROUND_STOCHASTIC if stochastic else _jf.ROUND_NEAREST
    qdx, sdx, dg, db = _jf.layernorm_bwd(_c(x), _c(sx), _c(g), _c(sg), _f32(w), _f32(m), _f32(v), rounding, return_dbias)
    out = (qdx, sdx, dg if w.dtype == torch.float32 else dg.to(w.dtype))
    return out + (db.to(w.dtype),) if return_dbias else out


def int8_layernorm_backward_add(x, sx, g, sg, w, QB, m, v, x1, stochastic=False, add_stochastic=False, add_rounding="trunc",
                                out_dtype=torch.float32, return_dbias=False):
    """int8_layernorm_backward followed by int8_add_Ifp_Ig16_Ofp_Og(x1, dx, s_dx, ...) (the pair the reference's recipe
    calls back to back, qmodel.py:125-128, 258-261) as one kernel for rows of up to 2048 columns, same bits.
    Returns (y1, y2, s_y2, dweight[, dbias])."""
    _check_qb(QB)
    rounding = _jf.ROUND_STOCHASTIC if stochastic else _jf.ROUND_NEAREST
    y1, q, s, dg, db = _jf.layernorm_bwd_add(_c(x), _c(sx), _c(g), _c(sg), _f32(w), _f32(m), _f32(v), _c(x1), rounding,
                                             _add_rounding(add_stochastic, add_rounding), return_dbias, out_dtype)
    out = (y1, q, s, dg if w.dtype == torch.float32 else dg.to(w.dtype))
    return out + (db.to(w.dtype),) if return_dbias else out


def int8_gelu_forward(x, s_x, QB, approximate="none"):
    """dequant -> GELU -> requant.  'none' = erf form with SCALE_MIN_THRES added to the block absmax
    (reference: gelu_fwd.py:81,90); 'tanh' = tanh approximation, no threshold."""
    _check_qb(QB)
    if approximate == "none":
        return _jf.gelu_fwd(_c(x), _c(s_x), _jf.GELU_ERF, SCALE_MIN_THRES)
    if approximate == "tanh":
        return _jf.gelu_fwd(_c(x), _c(s_x), _jf.GELU_TANH, 0.0)
    raise RuntimeError("approximate must be 'none' or 'tanh'")


def int8_gelu_backward(x, s_x, g, s_g, QB, stochastic=False, approximate="none"):
    """(x, g) -> gelu'(x) * g, requantised.  Reference: gelu_bwd.py:173-215."""
    _check_qb(QB)
    if approximate not in ("none", "tanh"):
        raise RuntimeError("approximate must be 'none' or 'tanh'")
    return _jf.gelu_bwd(_c(x), _c(s_x), _c(g), _c(s_g), _jf.GELU_ERF if approximate == "none" else _jf.GELU_TANH,
                        _jf.ROUND_STOCHASTIC if stochastic else _jf.ROUND_NEAREST)


def _add_rounding(stochastic, rounding):
    if rounding == "trunc":       # what the reference computes: .to(int8) without llrint (add.py:139)
        return _jf.ROUND_STOCHASTIC_TRUNC if stochastic else _jf.ROUND_TRUNC
    if rounding == "nearest":
        return _jf.ROUND_STOCHASTIC if stochastic else _jf.ROUND_NEAREST
    raise RuntimeError("rounding must be 'trunc' or 'nearest'")


def int8_add_Ifp_Ig16_Ofp_Og(x1, x2, s_x2, QB, stochastic=False, rounding="trunc", out_dtype=torch.float32):
    """y1 = x1 + dequant(x2) as float32, and its block quantisation (y2, s_y2).  Reference: add.py:164-211.
    out_dtype = float16 / bfloat16: y1 leaves the kernel already cast (what the reference's recipe does with a separate
    `.to()`, qmodel.py:228); y2, s_y2 are those of the fp32 sum either way."""
    _check_qb(QB)
    y1, q, s, _, _ = _jf.add(_c(x1), _c(x2), _c(s_x2), _add_rounding(stochastic, rounding), False, out_dtype)
    return y1, q, s


def int8_add_Ifp_Ig16_Ofp_Og_MeanVar(x1, x2, s_x2, QB, rounding="trunc", out_dtype=torch.float32):
    """As above plus per-row (mean, rstd) of the fp32 y1 for the next LayerNorm: var = E[y^2] - mean^2,
    rstd = 1/sqrt(var), no epsilon (reference: add_mean_var.py:179-230, finishing step :219-221)."""
    _check_qb(QB)
    # the statistics are finished by a second kernel inside the same call (the reference: eight torch operators)
    return _jf.add(_c(x1), _c(x2), _c(s_x2), _add_rounding(False, rounding), True, out_dtype)


def int8_column_sums(g, s_g, QB):
    """Column sums over all rows of the block tensor (g, s_g), float32 [N]: the bias gradient of a linear layer from its
    quantised output gradient (sketched in the reference as G8.sum(0), QBlockLinear.py:63-66).  3-D operands are summed
    over both leading dimensions."""
    _check_qb(QB)
    return _jf.block_colsum(_c(g), _c(s_g))
