// BlockQuantizeCUDA.jetfire -- the rest of the host side of the INT8 data-flow path as PyTorch C++ functions: the
// operators of Jetfire/Nonlinear (quantize, transpose, dequantize, LayerNorm, GELU, residual add; reference launchers:
// Jetfire/Nonlinear/*.py) and the GEMMs with fused epilogues that Jetfire/Linear uses besides the reference's eight
// (bindings.cpp:6-35 lives in bqc_ext.cpp).  The reference launches its Triton kernels from Python; here every operator
// is one C++ call that validates its tensors, allocates the outputs, reserves Philox counters under the generator's
// mutex, releases the GIL and enqueues the gfx950 kernel on the current stream through the C ABI.
//
// Operands are 2-D ([R, C] codes / values, [R/32, C/32] scales) or 3-D ([B, T, C] with [B, T/32, C/32] scales; results then
// have that rank too), vectors (per row, per column) of any shape with the right number of elements.
// seed / offset arguments: None = reserve from the device's default generator (what the operator API does); integers =
// use exactly these (tests, captured graphs).
#include "bqc_common.h"

#include <cmath>
#include <vector>

namespace jfext {
namespace {

using torch::Tensor;
using OptU64 = c10::optional<uint64_t>;
using OptTensor = c10::optional<Tensor>;
using OptDtype = c10::optional<torch::ScalarType>;

int fp_code(torch::ScalarType t, const char *name)
{
    if (t == torch::kFloat16) return JF_FP_F16;
    if (t == torch::kFloat32) return JF_FP_F32;
    if (t == torch::kBFloat16) return JF_FP_BF16;
    TORCH_CHECK(false, name, ": expected float16, float32 or bfloat16, got ", t);
    return -1;
}

int scale_code_of(torch::ScalarType t)
{
    TORCH_CHECK(t == torch::kFloat16 || t == torch::kFloat32, "scale_dtype must be float16 or float32, got ", t);
    return t == torch::kFloat16 ? JF_SCALE_F16 : JF_SCALE_F32;
}

void check_rounding(int64_t r, bool trunc_ok)
{
    TORCH_CHECK(r == JF_ROUND_NEAREST || r == JF_ROUND_STOCHASTIC ||
                    (trunc_ok && (r == JF_ROUND_TRUNC || r == JF_ROUND_STOCHASTIC_TRUNC)),
                "unknown rounding code ", r);
}

bool is_stochastic(int64_t r) { return r == JF_ROUND_STOCHASTIC || r == JF_ROUND_STOCHASTIC_TRUNC; }

void need(const Tensor &t, const char *name, int64_t dim)
{
    TORCH_CHECK(t.is_cuda(), name, ": expected a GPU tensor");
    TORCH_CHECK(t.dim() == dim, name, ": expected ", dim, " dimensions, got ", t.dim());
    TORCH_CHECK(t.is_contiguous(), name, ": expected a contiguous tensor");
}

// a contiguous tensor of 2 to max_dim dimensions, read as [R, C]
void rows_of(const Tensor &t, const char *name, int64_t &R, int64_t &C, int64_t max_dim = 3)
{
    TORCH_CHECK(t.is_cuda(), name, ": expected a GPU tensor");
    TORCH_CHECK(t.dim() >= 2 && t.dim() <= max_dim, name, ": expected a 2-D or 3-D tensor, got ", t.dim(), " dimensions");
    TORCH_CHECK(t.is_contiguous(), name, ": expected a contiguous tensor");
    C = t.size(-1);
    R = 1;
    for (int64_t d = 0; d + 1 < t.dim(); ++d) R *= t.size(d);
}

// the scales of a [R, C] or [B, T, C] tensor
std::vector<int64_t> scale_shape(const Tensor &x)
{
    std::vector<int64_t> n = x.sizes().vec();
    const int64_t T = n[n.size() - 2];
    TORCH_CHECK(T % QB == 0, "dimension ", T, " is not a positive multiple of 32");
    n[n.size() - 2] = T / QB;
    n[n.size() - 1] /= QB;
    return n;
}

// scales of a result laid out like the codes q (an operand's own scales may have another rank: [B, T, C] with [B T/32, C/32])
Tensor scales_for(const Tensor &q, const Tensor &s)
{
    return fresh(scale_shape(q), s.options());
}

// one value per row, [R] or [B, T]
std::vector<int64_t> row_shape(const Tensor &x)
{
    std::vector<int64_t> n = x.sizes().vec();
    n.pop_back();
    return n;
}

void mult32(int64_t d)
{
    TORCH_CHECK(d > 0 && d % QB == 0, "dimension ", d, " is not a positive multiple of 32");
}

// (codes [R,C] int8, scales [R/32,C/32]) -> scale code; R, C out
int block_tensor(const Tensor &q, const Tensor &s, const char *name, int64_t &R, int64_t &C, int64_t max_dim = 3)
{
    rows_of(q, name, R, C, max_dim);
    TORCH_CHECK(q.scalar_type() == torch::kInt8, name, ": codes must be int8, got ", q.scalar_type());
    mult32(R); mult32(C);
    int64_t SR, SC;
    rows_of(s, name, SR, SC, max_dim);
    TORCH_CHECK(SR == R / QB && SC == C / QB, name, ": scale shape ", s.sizes(), " does not match codes ", q.sizes());
    TORCH_CHECK(s.device() == q.device(), name, ": codes and scales are on different devices");
    return scale_code(s, name);
}

const float *vec(const Tensor &v, int64_t n, const Tensor &like, const char *name)
{
    TORCH_CHECK(v.is_cuda(), name, ": expected a GPU tensor");
    TORCH_CHECK(v.is_contiguous() && v.scalar_type() == torch::kFloat32 && v.numel() == n && v.device() == like.device(), name,
                ": expected a float32 vector of ", n, " elements on ", like.device());
    return v.data_ptr<float>();
}

// (seed, offset): the given pair, or counters reserved from the device's generator when the rounding draws noise
std::pair<uint64_t, uint64_t> rng(int64_t rounding, const Tensor &like, int64_t numel, const OptU64 &seed, const OptU64 &offset)
{
    if (is_stochastic(rounding) && !seed.has_value()) return next_philox(like, numel);
    return {seed.value_or(0), offset.value_or(0)};
}

Tensor scratch(const Tensor &like, size_t bytes)
{
    return fresh({(int64_t)(bytes ? bytes : 16)}, like.options().dtype(torch::kInt8));
}

// ---- quantize / dequantize / transpose -----------------------------------------------------------------------------

// quantize.py:128-164; with transpose: quantize_transpose.py:131-171
std::tuple<Tensor, Tensor, OptTensor> quantize(const Tensor &x, int64_t rounding, OptDtype scale_dtype_o, bool transpose,
                                               double amax_eps, OptU64 seed, OptU64 offset)
{
    int64_t R, C;
    rows_of(x, "x", R, C);
    const int xc = fp_code(x.scalar_type(), "x");
    mult32(R); mult32(C);
    check_rounding(rounding, true);
    const torch::ScalarType scale_dtype = scale_dtype_o.value_or(torch::kFloat16);
    const int sc = scale_code_of(scale_dtype);
    c10::DeviceGuard guard(x.device());
    Tensor q = fresh(x.sizes(), x.options().dtype(torch::kInt8));
    Tensor s = fresh(scale_shape(x), x.options().dtype(scale_dtype));
    OptTensor qT;
    if (transpose) qT = fresh({C, R}, x.options().dtype(torch::kInt8));
    const auto so = rng(rounding, x, R * C, seed, offset);
    {
        pybind11::gil_scoped_release nogil;
        check_rc(jf_quantize(x.data_ptr(), xc, (int)R, (int)C, (int8_t *)q.data_ptr(), s.data_ptr(),
                             transpose ? (int8_t *)qT->data_ptr() : nullptr, sc, (int)rounding, so.first, so.second,
                             (float)amax_eps, current_stream(x)),
                 "quantize");
    }
    return std::make_tuple(q, s, qT);
}

// several floating tensors (weights) in one launch, round to nearest: [(codes, scales), ...]
std::vector<std::tuple<Tensor, Tensor>> quantize_many(const std::vector<Tensor> &xs, OptDtype scale_dtype_o)
{
    TORCH_CHECK(!xs.empty() && xs.size() <= 8, "between 1 and 8 tensors");
    const torch::ScalarType scale_dtype = scale_dtype_o.value_or(torch::kFloat16);
    const int sc = scale_code_of(scale_dtype), xc = fp_code(xs[0].scalar_type(), "xs"), n = (int)xs.size();
    c10::DeviceGuard guard(xs[0].device());
    std::vector<std::tuple<Tensor, Tensor>> out;
    const void *xp[8];
    int Rs[8], Cs[8];
    int8_t *qp[8];
    void *sp[8];
    for (int k = 0; k < n; ++k) {
        const Tensor &x = xs[k];
        int64_t R, C;
        rows_of(x, "xs", R, C);
        mult32(R); mult32(C);
        TORCH_CHECK(x.scalar_type() == xs[0].scalar_type() && x.device() == xs[0].device(), "xs: expected tensors of one type and device");
        Tensor q = fresh(x.sizes(), x.options().dtype(torch::kInt8)), s = fresh(scale_shape(x), x.options().dtype(scale_dtype));
        xp[k] = x.data_ptr(); Rs[k] = (int)R; Cs[k] = (int)C; qp[k] = (int8_t *)q.data_ptr(); sp[k] = s.data_ptr();
        out.emplace_back(std::move(q), std::move(s));
    }
    pybind11::gil_scoped_release nogil;
    check_rc(jf_quantize_many(n, xp, Rs, Cs, xc, qp, sp, sc, current_stream(xs[0])), "quantize_many");
    return out;
}

// per-row mean and 1/sqrt(biased variance) of a floating tensor (qmodel.py:429-430)
std::tuple<Tensor, Tensor> rowstats_fp(const Tensor &x)
{
    int64_t R, C;
    rows_of(x, "x", R, C);
    mult32(C);
    const int xc = fp_code(x.scalar_type(), "x");
    c10::DeviceGuard guard(x.device());
    Tensor mean = fresh(row_shape(x), x.options().dtype(torch::kFloat32)), rstd = fresh_like(mean);
    pybind11::gil_scoped_release nogil;
    check_rc(jf_rowstats_fp(x.data_ptr(), xc, (int)R, (int)C, mean.data_ptr<float>(), rstd.data_ptr<float>(), current_stream(x)), "rowstats_fp");
    return std::make_tuple(mean, rstd);
}

// the block tensor of torch.cat(slabs, dim=1) without the concatenation (jf_quantize_slabs)
std::tuple<Tensor, Tensor> quantize_slabs(const std::vector<Tensor> &slabs, int64_t rounding, OptDtype scale_dtype_o,
                                          double amax_eps, OptU64 seed, OptU64 offset)
{
    TORCH_CHECK(!slabs.empty() && slabs.size() <= 4, "between 1 and 4 slabs");
    const Tensor &x0 = slabs[0];
    const int64_t R = x0.dim() == 2 ? x0.size(0) : -1;
    int64_t Ct = 0;
    const void *xs[4];
    int ld[4], wd[4];
    for (size_t k = 0; k < slabs.size(); ++k) {
        const Tensor &x = slabs[k];
        TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.size(0) == R && x.stride(1) == 1 && x.device() == x0.device() &&
                        x.scalar_type() == x0.scalar_type(),
                    "slabs: expected 2-D GPU tensors of one dtype with the same number of rows and unit column stride");
        mult32(x.size(1));
        xs[k] = x.data_ptr(); ld[k] = (int)x.stride(0); wd[k] = (int)x.size(1);
        Ct += x.size(1);
    }
    mult32(R);
    const int xc = fp_code(x0.scalar_type(), "slabs");
    check_rounding(rounding, true);
    const torch::ScalarType scale_dtype = scale_dtype_o.value_or(torch::kFloat16);
    const int sc = scale_code_of(scale_dtype);
    c10::DeviceGuard guard(x0.device());
    Tensor q = fresh({R, Ct}, x0.options().dtype(torch::kInt8));
    Tensor s = fresh({R / QB, Ct / QB}, x0.options().dtype(scale_dtype));
    const auto so = rng(rounding, x0, R * Ct, seed, offset);
    {
        pybind11::gil_scoped_release nogil;
        check_rc(jf_quantize_slabs(xs, ld, wd, (int)slabs.size(), xc, (int)R, (int8_t *)q.data_ptr(), s.data_ptr(), sc,
                                   (int)rounding, so.first, so.second, (float)amax_eps, current_stream(x0)),
                 "quantize_slabs");
    }
    return std::make_tuple(q, s);
}

// dequantize.py:86-116
Tensor dequantize(const Tensor &q, const Tensor &s, OptDtype out_dtype_o)
{
    const torch::ScalarType out_dtype = out_dtype_o.value_or(torch::kFloat32);
    int64_t R, C;
    const int sc = block_tensor(q, s, "x", R, C);
    const int oc = fp_code(out_dtype, "out_dtype");
    c10::DeviceGuard guard(q.device());
    Tensor out = fresh(q.sizes(), q.options().dtype(out_dtype));
    pybind11::gil_scoped_release nogil;
    check_rc(jf_dequantize((const int8_t *)q.data_ptr(), s.data_ptr(), (int)R, (int)C, sc, out.data_ptr(), oc, current_stream(q)),
             "dequantize");
    return out;
}

// transpose.py:69-97
Tensor transpose_s8(const Tensor &q)
{
    int64_t R, C;
    rows_of(q, "x", R, C);
    TORCH_CHECK(q.scalar_type() == torch::kInt8, "x must be int8");
    TORCH_CHECK(R > 0 && C > 0 && R % 16 == 0 && C % 16 == 0, "transpose: dimensions must be positive multiples of 16");
    c10::DeviceGuard guard(q.device());
    Tensor out = fresh({C, R}, q.options());
    pybind11::gil_scoped_release nogil;
    check_rc(jf_transpose_s8((const int8_t *)q.data_ptr(), (int)R, (int)C, (int8_t *)out.data_ptr(), current_stream(q)), "transpose");
    return out;
}

// ---- LayerNorm -----------------------------------------------------------------------------------------------------

std::tuple<Tensor, Tensor> rowstats(const Tensor &q, const Tensor &s, double eps)
{
    int64_t R, C;
    const int sc = block_tensor(q, s, "x", R, C);
    c10::DeviceGuard guard(q.device());
    Tensor mean = fresh(row_shape(q), q.options().dtype(torch::kFloat32)), rstd = fresh_like(mean);
    pybind11::gil_scoped_release nogil;
    check_rc(jf_rowstats((const int8_t *)q.data_ptr(), s.data_ptr(), (int)R, (int)C, sc, (float)eps, mean.data_ptr<float>(),
                         rstd.data_ptr<float>(), current_stream(q)),
             "rowstats");
    return std::make_tuple(mean, rstd);
}

// layernorm.py:430-465
std::tuple<Tensor, Tensor> layernorm_fwd(const Tensor &q, const Tensor &s, const Tensor &gamma, const OptTensor &beta,
                                         const Tensor &mean, const Tensor &rstd)
{
    int64_t R, C;
    const int sc = block_tensor(q, s, "x", R, C);
    const float *g = vec(gamma, C, q, "gamma"), *b = beta ? vec(*beta, C, q, "beta") : nullptr;
    const float *m = vec(mean, R, q, "mean"), *r = vec(rstd, R, q, "rstd");
    c10::DeviceGuard guard(q.device());
    Tensor qy = fresh_like(q), sy = scales_for(q, s);
    pybind11::gil_scoped_release nogil;
    check_rc(jf_layernorm_fwd((const int8_t *)q.data_ptr(), s.data_ptr(), g, b, m, r, (int)R, (int)C, sc, (int8_t *)qy.data_ptr(),
                              sy.data_ptr(), current_stream(q)),
             "layernorm_fwd");
    return std::make_tuple(qy, sy);
}

// layernorm.py:467-526
std::tuple<Tensor, Tensor, Tensor, OptTensor> layernorm_bwd(const Tensor &qx, const Tensor &sx, const Tensor &qg, const Tensor &sg,
                                                            const Tensor &gamma, const Tensor &mean, const Tensor &rstd,
                                                            int64_t rounding, bool want_dbeta, OptU64 seed, OptU64 offset)
{
    int64_t R, C, R2, C2;
    const int sc = block_tensor(qx, sx, "x", R, C);
    TORCH_CHECK(block_tensor(qg, sg, "g", R2, C2) == sc && R2 == R && C2 == C && qg.device() == qx.device(),
                "x and g must have the same shape, scale dtype and device");
    const float *g = vec(gamma, C, qx, "gamma"), *m = vec(mean, R, qx, "mean"), *r = vec(rstd, R, qx, "rstd");
    check_rounding(rounding, true);
    c10::DeviceGuard guard(qx.device());
    const size_t nbytes = jf_layernorm_bwd_workspace_bytes((int)R, (int)C);
    Tensor ws = scratch(qx, nbytes);
    Tensor qdx = fresh_like(qx), sdx = scales_for(qx, sx);
    Tensor dgamma = fresh({C}, qx.options().dtype(torch::kFloat32));
    OptTensor dbeta;
    if (want_dbeta) dbeta = fresh_like(dgamma);
    const auto so = rng(rounding, qx, R * C, seed, offset);
    {
        pybind11::gil_scoped_release nogil;
        check_rc(jf_layernorm_bwd((const int8_t *)qx.data_ptr(), sx.data_ptr(), (const int8_t *)qg.data_ptr(), sg.data_ptr(), g, m, r,
                                  (int)R, (int)C, sc, (int)rounding, so.first, so.second, (int8_t *)qdx.data_ptr(), sdx.data_ptr(),
                                  dgamma.data_ptr<float>(), want_dbeta ? dbeta->data_ptr<float>() : nullptr, ws.data_ptr(), nbytes,
                                  current_stream(qx)),
                 "layernorm_bwd");
    }
    return std::make_tuple(qdx, sdx, dgamma, dbeta);
}

// add.py:164-211 / add_mean_var.py:179-230 (with_stats: the row statistics are finished here as well, :219-221)
std::tuple<Tensor, Tensor, Tensor, OptTensor, OptTensor> add(const Tensor &x1, const Tensor &q2, const Tensor &s2, int64_t rounding,
                                                             bool with_stats, OptDtype out_dtype_o, OptU64 seed, OptU64 offset)
{
    const torch::ScalarType out_dtype = out_dtype_o.value_or(torch::kFloat32);
    int64_t R, C;
    const int sc = block_tensor(q2, s2, "x2", R, C);
    int64_t R1, C1;
    rows_of(x1, "x1", R1, C1);
    const int xc = fp_code(x1.scalar_type(), "x1"), oc = fp_code(out_dtype, "out_dtype");
    TORCH_CHECK(R1 == R && C1 == C && x1.device() == q2.device(), "x1 must be a float tensor of the shape and device of x2");
    check_rounding(rounding, true);
    c10::DeviceGuard guard(x1.device());
    Tensor y1 = fresh(x1.sizes(), x1.options().dtype(out_dtype));
    Tensor q = fresh(x1.sizes(), q2.options()), s = fresh(scale_shape(x1), s2.options());
    Tensor ws;
    OptTensor mean, rstd;
    size_t nbytes = 0;
    if (with_stats) {
        nbytes = jf_add_rowstats_workspace_bytes((int)R, (int)C);
        if (nbytes) ws = scratch(x1, nbytes);
        mean = fresh(row_shape(x1), x1.options().dtype(torch::kFloat32));
        rstd = fresh_like(*mean);
    }
    const auto so = rng(rounding, x1, R * C, seed, offset);
    {
        pybind11::gil_scoped_release nogil;
        const jf_stream_t st = current_stream(x1);
        if (with_stats)
            check_rc(jf_add_rowstats(x1.data_ptr(), xc, (const int8_t *)q2.data_ptr(), s2.data_ptr(), (int)R, (int)C, sc, (int)rounding, so.first,
                                     so.second, y1.data_ptr(), oc, (int8_t *)q.data_ptr(), s.data_ptr(), mean->data_ptr<float>(),
                                     rstd->data_ptr<float>(), nbytes ? ws.data_ptr() : nullptr, nbytes, st), "add");
        else
            check_rc(jf_add(x1.data_ptr(), xc, (const int8_t *)q2.data_ptr(), s2.data_ptr(), (int)R, (int)C, sc, (int)rounding, so.first,
                            so.second, y1.data_ptr(), oc, (int8_t *)q.data_ptr(), s.data_ptr(), nullptr, nullptr, st), "add");
    }
    return std::make_tuple(y1, q, s, mean, rstd);
}

// the pair layernorm.py:467-526 + add.py:164-211 (qmodel.py:125-128, 258-261): one kernel for rows of up to 2048 columns,
// the two calls (same noise counters, same bits) beyond
std::tuple<Tensor, Tensor, Tensor, Tensor, OptTensor> layernorm_bwd_add(const Tensor &qx, const Tensor &sx, const Tensor &qg,
                                                                        const Tensor &sg, const Tensor &gamma, const Tensor &mean,
                                                                        const Tensor &rstd, const Tensor &x1, int64_t rounding,
                                                                        int64_t add_rounding, bool want_dbeta,
                                                                        OptDtype out_dtype_o, OptU64 seed, OptU64 offset,
                                                                        OptU64 add_seed, OptU64 add_offset)
{
    const torch::ScalarType out_dtype = out_dtype_o.value_or(torch::kFloat32);
    int64_t R, C, R2, C2;
    const int sc = block_tensor(qx, sx, "x", R, C);
    TORCH_CHECK(block_tensor(qg, sg, "g", R2, C2) == sc && R2 == R && C2 == C && qg.device() == qx.device(),
                "x and g must have the same shape, scale dtype and device");
    const float *g = vec(gamma, C, qx, "gamma"), *m = vec(mean, R, qx, "mean"), *r = vec(rstd, R, qx, "rstd");
    int64_t R1, C1;
    rows_of(x1, "x1", R1, C1);
    const int xc = fp_code(x1.scalar_type(), "x1"), oc = fp_code(out_dtype, "out_dtype");
    TORCH_CHECK(R1 == R && C1 == C && x1.device() == qx.device(), "x1 must be a float tensor of the shape and device of x");
    check_rounding(rounding, true);
    check_rounding(add_rounding, true);
    const auto so = rng(rounding, qx, R * C, seed, offset);
    const auto ao = rng(add_rounding, qx, R * C, add_seed, add_offset);
    if (C / QB > 64) {
        auto [qdx, sdx, dgamma, dbeta] = layernorm_bwd(qx, sx, qg, sg, gamma, mean, rstd, rounding, want_dbeta, so.first, so.second);
        auto [y1, q, s, _m, _r] = add(x1.view(qx.sizes()), qdx, sdx, add_rounding, false, out_dtype, ao.first, ao.second);
        return std::make_tuple(y1, q, s, dgamma, dbeta);
    }
    c10::DeviceGuard guard(qx.device());
    const size_t nbytes = jf_layernorm_bwd_workspace_bytes((int)R, (int)C);
    Tensor ws = scratch(qx, nbytes);
    Tensor y1 = fresh(qx.sizes(), x1.options().dtype(out_dtype));
    Tensor q = fresh_like(qx), s = scales_for(qx, sx);
    Tensor dgamma = fresh({C}, qx.options().dtype(torch::kFloat32));
    OptTensor dbeta;
    if (want_dbeta) dbeta = fresh_like(dgamma);
    {
        pybind11::gil_scoped_release nogil;
        check_rc(jf_layernorm_bwd_add((const int8_t *)qx.data_ptr(), sx.data_ptr(), (const int8_t *)qg.data_ptr(), sg.data_ptr(), g, m, r,
                                      (int)R, (int)C, sc, (int)rounding, so.first, so.second, x1.data_ptr(), xc, (int)add_rounding,
                                      ao.first, ao.second, y1.data_ptr(), oc, (int8_t *)q.data_ptr(), s.data_ptr(),
                                      dgamma.data_ptr<float>(), want_dbeta ? dbeta->data_ptr<float>() : nullptr, ws.data_ptr(), nbytes,
                                      current_stream(qx)),
                 "layernorm_bwd_add");
    }
    return std::make_tuple(y1, q, s, dgamma, dbeta);
}

// ---- GELU ----------------------------------------------------------------------------------------------------------

void check_approx(int64_t a) { TORCH_CHECK(a == JF_GELU_ERF || a == JF_GELU_TANH, "unknown GELU form ", a); }

// gelu_fwd.py:128-162
std::tuple<Tensor, Tensor> gelu_fwd(const Tensor &q, const Tensor &s, int64_t approx, double amax_eps)
{
    int64_t R, C;
    const int sc = block_tensor(q, s, "x", R, C);
    check_approx(approx);
    c10::DeviceGuard guard(q.device());
    Tensor qy = fresh_like(q), sy = scales_for(q, s);
    pybind11::gil_scoped_release nogil;
    check_rc(jf_gelu_fwd((const int8_t *)q.data_ptr(), s.data_ptr(), (int)R, (int)C, sc, (int)approx, (float)amax_eps,
                         (int8_t *)qy.data_ptr(), sy.data_ptr(), current_stream(q)),
             "gelu_fwd");
    return std::make_tuple(qy, sy);
}

// gelu_bwd.py:173-215
std::tuple<Tensor, Tensor> gelu_bwd(const Tensor &qx, const Tensor &sx, const Tensor &qg, const Tensor &sg, int64_t approx,
                                    int64_t rounding, OptU64 seed, OptU64 offset)
{
    int64_t R, C, R2, C2;
    const int sc = block_tensor(qx, sx, "x", R, C);
    TORCH_CHECK(block_tensor(qg, sg, "g", R2, C2) == sc && R2 == R && C2 == C && qg.device() == qx.device(),
                "x and g must have the same shape, scale dtype and device");
    check_approx(approx);
    check_rounding(rounding, true);
    c10::DeviceGuard guard(qx.device());
    Tensor qy = fresh_like(qx), sy = scales_for(qx, sx);
    const auto so = rng(rounding, qx, R * C, seed, offset);
    pybind11::gil_scoped_release nogil;
    check_rc(jf_gelu_bwd((const int8_t *)qx.data_ptr(), sx.data_ptr(), (const int8_t *)qg.data_ptr(), sg.data_ptr(), (int)R, (int)C, sc,
                         (int)approx, (int)rounding, so.first, so.second, (int8_t *)qy.data_ptr(), sy.data_ptr(), current_stream(qx)),
             "gelu_bwd");
    return std::make_tuple(qy, sy);
}

// ---- causal self-attention (qmodel.py:134) ---------------------------------------------------------------------------

// q, k, v: [B*T, C] binary16 views of one row stride (column ranges of the QKV projection's output), heads D = C/heads wide
struct AttentionOperands {
    int B, H, T, D, ld;
    int64_t C;
    float scale;
};
AttentionOperands attention_operands(const Tensor &q, const Tensor &k, const Tensor &v, int64_t batch, int64_t heads)
{
    for (const Tensor *t : {&q, &k, &v})
        TORCH_CHECK(t->is_cuda() && t->dim() == 2 && t->scalar_type() == torch::kFloat16 && t->stride(1) == 1 && t->sizes() == q.sizes() &&
                        t->stride(0) == q.stride(0) && t->device() == q.device(),
                    "attention: q, k, v must be float16 [tokens, C] GPU tensors of one shape, row stride and device");
    const int64_t M = q.size(0), C = q.size(1);
    TORCH_CHECK(batch > 0 && heads > 0 && M % batch == 0 && C % heads == 0, "attention: ", q.sizes(), " does not split into ", batch,
                " sequences and ", heads, " heads");
    const int64_t D = C / heads;
    return {(int)batch, (int)heads, (int)(M / batch), (int)D, (int)q.stride(0), C, (float)(1.0 / std::sqrt((double)D))};
}

std::tuple<Tensor, Tensor> attention_fwd(const Tensor &q, const Tensor &k, const Tensor &v, int64_t batch, int64_t heads)
{
    const AttentionOperands a = attention_operands(q, k, v, batch, heads);
    c10::DeviceGuard guard(q.device());
    Tensor out = fresh({q.size(0), a.C}, q.options()), lse = fresh({(int64_t)a.B * a.H, a.T}, q.options().dtype(torch::kFloat32));
    pybind11::gil_scoped_release nogil;
    check_rc(jf_attention_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), a.ld, a.B, a.H, a.T, a.D, a.scale, out.data_ptr(),
                              lse.data_ptr<float>(), current_stream(q)),
             "attention_fwd");
    return std::make_tuple(out, lse);
}

void attention_gradient_operands(const Tensor &q, const Tensor &out, const Tensor &lse, const Tensor &gout, const AttentionOperands &a)
{
    for (const Tensor *t : {&out, &gout}) {
        need(*t, "attention: out / its gradient", 2);
        TORCH_CHECK(t->scalar_type() == torch::kFloat16 && t->sizes() == q.sizes() && t->device() == q.device(),
                    "attention: out and its gradient must be float16 tensors of the shape of q");
    }
    vec(lse, q.size(0) * a.H, q, "lse");
}

// the gradients side by side, [B*T, 3C]
Tensor attention_bwd(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &out, const Tensor &lse, const Tensor &gout,
                     int64_t batch, int64_t heads)
{
    const AttentionOperands a = attention_operands(q, k, v, batch, heads);
    attention_gradient_operands(q, out, lse, gout, a);
    c10::DeviceGuard guard(q.device());
    Tensor g = fresh({q.size(0), 3 * a.C}, q.options()), delta = fresh_like(lse);
    c10::Half *gp = g.data_ptr<c10::Half>();
    pybind11::gil_scoped_release nogil;
    check_rc(jf_attention_bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), a.ld, out.data_ptr(), gout.data_ptr(), lse.data_ptr<float>(), a.B,
                              a.H, a.T, a.D, a.scale, gp, gp + a.C, gp + 2 * a.C, (int)(3 * a.C), delta.data_ptr<float>(), current_stream(q)),
             "attention_bwd");
    return g;
}

// attention_fwd with the block quantisation of its result: (out, lse, codes, scales)
std::tuple<Tensor, Tensor, Tensor, Tensor> attention_fwd_q(const Tensor &q, const Tensor &k, const Tensor &v, int64_t batch, int64_t heads)
{
    const AttentionOperands a = attention_operands(q, k, v, batch, heads);
    c10::DeviceGuard guard(q.device());
    const int64_t M = q.size(0);
    Tensor out = fresh({M, a.C}, q.options()), lse = fresh({(int64_t)a.B * a.H, a.T}, q.options().dtype(torch::kFloat32));
    Tensor codes = fresh({M, a.C}, q.options().dtype(torch::kInt8)), scales = fresh({M / QB, a.C / QB}, q.options());
    pybind11::gil_scoped_release nogil;
    check_rc(jf_attention_fwd_q(q.data_ptr(), k.data_ptr(), v.data_ptr(), a.ld, a.B, a.H, a.T, a.D, a.scale, out.data_ptr(), lse.data_ptr<float>(),
                                (int8_t *)codes.data_ptr(), scales.data_ptr(), current_stream(q)),
             "attention_fwd_q");
    return std::make_tuple(out, lse, codes, scales);
}

// attention_bwd with the gradients quantised: (codes, scales)
std::tuple<Tensor, Tensor> attention_bwd_q(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &out, const Tensor &lse,
                                           const Tensor &gout, int64_t batch, int64_t heads, OptU64 seed, OptU64 offset)
{
    const AttentionOperands a = attention_operands(q, k, v, batch, heads);
    attention_gradient_operands(q, out, lse, gout, a);
    c10::DeviceGuard guard(q.device());
    const int64_t M = q.size(0);
    Tensor codes = fresh({M, 3 * a.C}, q.options().dtype(torch::kInt8)), scales = fresh({M / QB, 3 * a.C / QB}, q.options());
    Tensor delta = fresh_like(lse);
    const auto so = rng(JF_ROUND_STOCHASTIC, q, 3 * M * a.C, seed, offset);
    pybind11::gil_scoped_release nogil;
    check_rc(jf_attention_bwd_q(q.data_ptr(), k.data_ptr(), v.data_ptr(), a.ld, out.data_ptr(), gout.data_ptr(), lse.data_ptr<float>(), a.B, a.H, a.T,
                                a.D, a.scale, (int8_t *)codes.data_ptr(), scales.data_ptr(), so.first, so.second, delta.data_ptr<float>(),
                                current_stream(q)),
             "attention_bwd_q");
    return std::make_tuple(codes, scales);
}

// ---- column sums (bias gradient; QBlockLinear.py:63-66) -------------------------------------------------------------

Tensor block_colsum(const Tensor &q, const Tensor &s)
{
    int64_t R, C;
    const int sc = block_tensor(q, s, "x", R, C);
    c10::DeviceGuard guard(q.device());
    const size_t nbytes = jf_block_colsum_workspace_bytes((int)R, (int)C);
    Tensor ws = scratch(q, nbytes);
    Tensor out = fresh({C}, q.options().dtype(torch::kFloat32));
    pybind11::gil_scoped_release nogil;
    check_rc(jf_block_colsum((const int8_t *)q.data_ptr(), s.data_ptr(), (int)R, (int)C, sc, out.data_ptr<float>(), ws.data_ptr(), nbytes,
                             current_stream(q)),
             "block_colsum");
    return out;
}

// ---- GEMMs with fused epilogues ------------------------------------------------------------------------------------

struct GemmOperands {
    int M, N, K, code, la, lb;
    const float *bias = nullptr, *biasmax = nullptr;
};

// A [M,K] contiguous; B [N,K] (layout JF_B_NK) or [K,N] (JF_B_KN) contiguous; scale operands [K/32, rows/32], contiguous or
// the .t() view of the block tensor's own scales; bias [N] / biasmax [1] float32 or None
GemmOperands gemm_operands(const Tensor &A, const Tensor &B, const Tensor &sa, const Tensor &sb, int64_t layout, const OptTensor &bias,
                           const OptTensor &biasmax)
{
    TORCH_CHECK(layout == JF_B_NK || layout == JF_B_KN, "b_layout must be B_NK (0) or B_KN (1)");
    need(A, "A", 2); need(B, "B", 2);
    TORCH_CHECK(A.scalar_type() == torch::kInt8 && B.scalar_type() == torch::kInt8, "A and B must be int8");
    TORCH_CHECK(B.device() == A.device(), "A and B are on different devices");
    GemmOperands g;
    const int64_t M = A.size(0), K = A.size(1), N = layout == JF_B_NK ? B.size(0) : B.size(1);
    TORCH_CHECK((layout == JF_B_NK ? B.size(1) : B.size(0)) == K, "inner dimensions differ: A is ", A.sizes(), ", B is ", B.sizes());
    check_dims(M, N, K);
    g.M = (int)M; g.N = (int)N; g.K = (int)K;
    g.code = check_scales(sa, sb, A, M, N, K, g.la, g.lb);
    TORCH_CHECK(bias.has_value() == biasmax.has_value(), "bias and biasmax come together");
    if (bias) {
        TORCH_CHECK(bias->is_cuda() && bias->device() == A.device() && bias->scalar_type() == torch::kFloat32 && bias->is_contiguous() &&
                        bias->numel() == N, "bias must be a contiguous float32 GPU tensor of N elements");
        TORCH_CHECK(biasmax->is_cuda() && biasmax->device() == A.device() && biasmax->scalar_type() == torch::kFloat32 &&
                        biasmax->numel() >= 1, "biasmax must be a float32 GPU tensor with one element");
        g.bias = bias->data_ptr<float>();
        g.biasmax = biasmax->data_ptr<float>();
    }
    return g;
}

// linear_fwd.py:23 followed by gelu_fwd.py:128-162 (qmodel.py:210-214), one kernel
std::tuple<Tensor, Tensor, Tensor, Tensor> igemm_block_q_gelu(const Tensor &A, const Tensor &B, const Tensor &sa, const Tensor &sb,
                                                              int64_t approx, double amax_eps, const OptTensor &bias,
                                                              const OptTensor &biasmax)
{
    const GemmOperands g = gemm_operands(A, B, sa, sb, JF_B_NK, bias, biasmax);
    check_approx(approx);
    c10::DeviceGuard guard(A.device());
    Tensor q = fresh({g.M, g.N}, A.options());
    Tensor s = fresh({g.M / QB, g.N / QB}, sa.options().memory_format(c10::MemoryFormat::Contiguous));
    Tensor qg = fresh_like(q), sg = fresh_like(s);
    pybind11::gil_scoped_release nogil;
    check_rc(jf_igemm_block_q_gelu((const int8_t *)A.data_ptr(), (const int8_t *)B.data_ptr(), sa.data_ptr(), sb.data_ptr(), g.bias,
                                   g.biasmax, (int8_t *)q.data_ptr(), s.data_ptr(), (int8_t *)qg.data_ptr(), sg.data_ptr(), g.M, g.N, g.K,
                                   g.code, g.la, g.lb, (int)approx, (float)amax_eps, current_stream(A)),
             "igemm_block_q_gelu");
    return std::make_tuple(q, s, qg, sg);
}

// linear_bwd.py:17 followed by gelu_bwd.py:173-215 (qmodel.py:249-253), one kernel; the two draw their noise in that order
std::tuple<Tensor, Tensor> igemm_block_q_gelu_bwd(const Tensor &A, const Tensor &B, const Tensor &sa, const Tensor &sb, const Tensor &xq,
                                                  const Tensor &xs, int64_t approx, int64_t gelu_rounding, OptU64 seed, OptU64 offset,
                                                  OptU64 gelu_seed, OptU64 gelu_offset)
{
    const GemmOperands g = gemm_operands(A, B, sa, sb, JF_B_KN, c10::nullopt, c10::nullopt);
    int64_t R2, C2;
    TORCH_CHECK(block_tensor(xq, xs, "x", R2, C2) == g.code && R2 == g.M && C2 == g.N && xq.device() == A.device(),
                "x must be an [M,N] block tensor with the scale dtype of sa / sb");
    check_approx(approx);
    check_rounding(gelu_rounding, false);
    c10::DeviceGuard guard(A.device());
    const auto so = rng(JF_ROUND_STOCHASTIC, A, (int64_t)g.M * g.N, seed, offset);
    const auto go = rng(gelu_rounding, A, (int64_t)g.M * g.N, gelu_seed, gelu_offset);
    Tensor out = fresh({g.M, g.N}, A.options());
    Tensor sc = fresh({g.M / QB, g.N / QB}, sa.options().memory_format(c10::MemoryFormat::Contiguous));
    pybind11::gil_scoped_release nogil;
    check_rc(jf_igemm_block_q_gelu_bwd((const int8_t *)A.data_ptr(), (const int8_t *)B.data_ptr(), sa.data_ptr(), sb.data_ptr(),
                                       (const int8_t *)xq.data_ptr(), xs.data_ptr(), (int8_t *)out.data_ptr(), sc.data_ptr(), g.M, g.N, g.K,
                                       g.code, g.la, g.lb, (int)approx, so.first, so.second, (int)gelu_rounding, go.first, go.second,
                                       current_stream(A)),
             "igemm_block_q_gelu_bwd");
    return std::make_tuple(out, sc);
}

// linear_fwd.py:22-32 / linear_bwd.py:17-29 with output_quantized / dgrad_quantize = False, one kernel
Tensor igemm_block_q_dequant(const Tensor &A, const Tensor &B, const Tensor &sa, const Tensor &sb, int64_t layout,
                             c10::optional<torch::ScalarType> out_dtype, const OptTensor &bias, const OptTensor &biasmax, int64_t rounding,
                             OptU64 seed, OptU64 offset)
{
    const GemmOperands g = gemm_operands(A, B, sa, sb, layout, bias, biasmax);
    const torch::ScalarType odt = out_dtype.value_or(sa.scalar_type());
    const int oc = fp_code(odt, "out_dtype");
    check_rounding(rounding, false);
    c10::DeviceGuard guard(A.device());
    const auto so = rng(rounding, A, (int64_t)g.M * g.N, seed, offset);
    Tensor out = fresh({g.M, g.N}, A.options().dtype(odt));
    pybind11::gil_scoped_release nogil;
    check_rc(jf_igemm_block_q_dequant((const int8_t *)A.data_ptr(), (const int8_t *)B.data_ptr(), sa.data_ptr(), sb.data_ptr(), g.bias,
                                      g.biasmax, out.data_ptr(), g.M, g.N, g.K, (int)layout, g.code, g.la, g.lb, oc, (int)rounding,
                                      so.first, so.second, current_stream(A)),
             "igemm_block_q_dequant");
    return out;
}

// the requantising GEMM with every option of the C ABI (the reference's four variants fix them: bqc_ext.cpp)
std::tuple<Tensor, Tensor> igemm_block_q(const Tensor &A, const Tensor &B, const Tensor &sa, const Tensor &sb, int64_t layout,
                                         const OptTensor &bias, const OptTensor &biasmax, int64_t rounding, OptU64 seed, OptU64 offset)
{
    const GemmOperands g = gemm_operands(A, B, sa, sb, layout, bias, biasmax);
    check_rounding(rounding, false);
    c10::DeviceGuard guard(A.device());
    const auto so = rng(rounding, A, (int64_t)g.M * g.N, seed, offset);
    Tensor out = fresh({g.M, g.N}, A.options());
    Tensor sc = fresh({g.M / QB, g.N / QB}, sa.options().memory_format(c10::MemoryFormat::Contiguous));
    pybind11::gil_scoped_release nogil;
    check_rc(jf_igemm_block_q((const int8_t *)A.data_ptr(), (const int8_t *)B.data_ptr(), sa.data_ptr(), sb.data_ptr(), g.bias, g.biasmax,
                              (int8_t *)out.data_ptr(), sc.data_ptr(), g.M, g.N, g.K, (int)layout, g.code, g.la, g.lb, (int)rounding,
                              so.first, so.second, nullptr, 0, current_stream(A)),
             "igemm_block_q");
    return std::make_tuple(out, sc);
}

// ---- package Linear (linear_fwd.py:4-32, linear_bwd.py:4-29) -------------------------------------------------------------

// an int8 operand [.., rows, cols] with its scales in the block tensor's own layout
struct Operand {
    Tensor q, s;
    int64_t R, C;
    int code;
    Operand(const Tensor &q_, const Tensor &s_, const char *name) : q(q_.contiguous()), s(s_.contiguous()) { code = block_tensor(q, s, name, R, C, 8); }
    int8_t *qp() const { return (int8_t *)q.data_ptr(); }
    void *sp() const { return s.data_ptr(); }
};

void same_kind(const Operand &a, const Operand &b)
{
    TORCH_CHECK(a.code == b.code, "scales must have the same dtype");
    TORCH_CHECK(a.q.device() == b.q.device(), "operands are on different devices");
}

// the sizes of x with another last dimension
std::vector<int64_t> with_last(const Tensor &x, int64_t n)
{
    std::vector<int64_t> v = x.sizes().vec();
    v.back() = n;
    return v;
}

void linear_bias(const OptTensor &bias, const OptTensor &biasmax, const Operand &x, int64_t N, const float *&b, const float *&bm)
{
    b = bm = nullptr;
    TORCH_CHECK(bias.has_value() == biasmax.has_value(), "bias and biasmax come together");
    if (!bias) return;
    b = vec(*bias, N, x.q, "bias");
    TORCH_CHECK(biasmax->is_cuda() && biasmax->device() == x.q.device() && biasmax->scalar_type() == torch::kFloat32 && biasmax->numel() >= 1,
                "biasmax must be a float32 GPU tensor with one element");
    bm = biasmax->data_ptr<float>();
}

// Y = X W^T (+ bias): (codes, scales), or (values in the scale type, None) with quantized = false
std::tuple<Tensor, OptTensor> linear_forward(const Tensor &X, const Tensor &SX, const Tensor &W, const Tensor &SW, bool quantized,
                                             const OptTensor &bias, const OptTensor &biasmax)
{
    const Operand x(X, SX, "X"), w(W, SW, "W");
    same_kind(x, w);
    TORCH_CHECK(w.q.dim() == 2 && x.C == w.C, "inner dimensions differ: X is ", X.sizes(), ", W is ", W.sizes());
    const float *b, *bm;
    linear_bias(bias, biasmax, x, w.R, b, bm);
    c10::DeviceGuard guard(x.q.device());
    if (!quantized) {
        Tensor out = fresh(with_last(x.q, w.R), x.s.options());
        pybind11::gil_scoped_release nogil;
        check_rc(jf_igemm_block_q_dequant(x.qp(), w.qp(), x.sp(), w.sp(), b, bm, out.data_ptr(), (int)x.R, (int)w.R, (int)x.C, JF_B_NK, x.code,
                                          JF_SCALES_ROWMAJOR, JF_SCALES_ROWMAJOR, x.code == JF_SCALE_F16 ? JF_FP_F16 : JF_FP_F32,
                                          JF_ROUND_NEAREST, 0, 0, current_stream(x.q)),
                 "linear_forward");
        return std::make_tuple(out, OptTensor());
    }
    Tensor o = fresh(with_last(x.q, w.R), x.q.options()), so = fresh(with_last(x.s, w.R / QB), x.s.options());
    pybind11::gil_scoped_release nogil;
    check_rc(jf_igemm_block_q(x.qp(), w.qp(), x.sp(), w.sp(), b, bm, (int8_t *)o.data_ptr(), so.data_ptr(), (int)x.R, (int)w.R, (int)x.C,
                              JF_B_NK, x.code, JF_SCALES_ROWMAJOR, JF_SCALES_ROWMAJOR, JF_ROUND_NEAREST, 0, 0, nullptr, 0, current_stream(x.q)),
             "linear_forward");
    return std::make_tuple(o, OptTensor(so));
}

std::tuple<Tensor, Tensor, Tensor, Tensor> linear_forward_gelu(const Tensor &X, const Tensor &SX, const Tensor &W, const Tensor &SW,
                                                               int64_t approx, double amax_eps, const OptTensor &bias, const OptTensor &biasmax)
{
    const Operand x(X, SX, "X"), w(W, SW, "W");
    same_kind(x, w);
    TORCH_CHECK(w.q.dim() == 2 && x.C == w.C, "inner dimensions differ: X is ", X.sizes(), ", W is ", W.sizes());
    check_approx(approx);
    const float *b, *bm;
    linear_bias(bias, biasmax, x, w.R, b, bm);
    c10::DeviceGuard guard(x.q.device());
    Tensor o = fresh(with_last(x.q, w.R), x.q.options()), so = fresh(with_last(x.s, w.R / QB), x.s.options());
    Tensor g = fresh_like(o), sg = fresh_like(so);
    pybind11::gil_scoped_release nogil;
    check_rc(jf_igemm_block_q_gelu(x.qp(), w.qp(), x.sp(), w.sp(), b, bm, (int8_t *)o.data_ptr(), so.data_ptr(), (int8_t *)g.data_ptr(),
                                   sg.data_ptr(), (int)x.R, (int)w.R, (int)x.C, x.code, JF_SCALES_ROWMAJOR, JF_SCALES_ROWMAJOR, (int)approx,
                                   (float)amax_eps, current_stream(x.q)),
             "linear_forward_gelu");
    return std::make_tuple(o, so, g, sg);
}

// dW = dY^T X of a gradient read where it lies, or of its transposed copy [C_out, tokens]
Tensor weight_gradient(const Operand &x, const Operand &g, const OptTensor &gT, int64_t splitk, OptDtype dtype)
{
    const torch::ScalarType odt = dtype.value_or(torch::kFloat16);
    const int oc = fp_code(odt, "wgrad_dtype");
    TORCH_CHECK(splitk >= 0, "splitk must be >= 0");
    const int M = (int)g.C, N = (int)x.C, K = (int)x.R;
    const int8_t *a = g.qp();
    int la = JF_A_KM;
    if (gT) {
        TORCH_CHECK(gT->device() == x.q.device(), "operands are on different devices");
        la = check_a_any_layout(*gT, M, K);
        a = (const int8_t *)gT->data_ptr();
    }
    Tensor out = fresh({M, N}, x.q.options().dtype(odt));
    const size_t nbytes = jf_igemm_block_fp_workspace_bytes(M, N, K, JF_B_KN, (int)splitk);
    Tensor ws;
    if (nbytes) ws = scratch(x.q, nbytes);
    pybind11::gil_scoped_release nogil;
    check_rc(jf_igemm_block_fp(a, x.qp(), g.sp(), x.sp(), out.data_ptr(), M, N, K, la, JF_B_KN, x.code, JF_SCALES_KMAJOR, JF_SCALES_KMAJOR, oc,
                               (int)splitk, nbytes ? ws.data_ptr() : nullptr, nbytes, current_stream(x.q)),
             "weight_gradient");
    return out;
}

// (dX codes, dX scales, dW[, db]) or (dX values, dW[, db])
std::vector<Tensor> linear_backward(const Tensor &X, const Tensor &SX, const Tensor &G, const Tensor &SG, const OptTensor &GT, const Tensor &W,
                                    const Tensor &SW, bool dgrad_quantize, int64_t splitk, OptDtype wgrad_dtype, bool bias_grad)
{
    const Operand x(X, SX, "X"), g(G, SG, "G"), w(W, SW, "W");
    same_kind(x, g); same_kind(x, w);
    TORCH_CHECK(x.R == g.R && w.q.dim() == 2 && w.R == g.C && w.C == x.C, "operands do not match: X ", X.sizes(), ", G ", G.sizes(), ", W ", W.sizes());
    c10::DeviceGuard guard(x.q.device());
    std::vector<Tensor> out;
    const auto so = rng(JF_ROUND_STOCHASTIC, g.q, g.R * w.C, c10::nullopt, c10::nullopt);
    if (!GT) {
        const torch::ScalarType odt = wgrad_dtype.value_or(torch::kFloat16);
        const int oc = fp_code(odt, "wgrad_dtype");
        TORCH_CHECK(splitk >= 0, "splitk must be >= 0");
        out.push_back(fresh(with_last(g.q, w.C), dgrad_quantize ? g.q.options() : g.s.options()));
        if (dgrad_quantize) out.push_back(fresh(with_last(g.s, w.C / QB), g.s.options()));
        out.push_back(fresh({g.C, x.C}, x.q.options().dtype(odt)));
        const size_t nbytes = jf_igemm_block_fp_workspace_bytes((int)g.C, (int)x.C, (int)x.R, JF_B_KN, (int)splitk);
        Tensor ws;
        if (nbytes) ws = scratch(x.q, nbytes);
        {
            pybind11::gil_scoped_release nogil;
            check_rc(jf_linear_bwd(x.qp(), x.sp(), g.qp(), g.sp(), w.qp(), w.sp(), (int)g.R, (int)w.C, (int)g.C, g.code, out[0].data_ptr(),
                                   dgrad_quantize ? out[1].data_ptr() : nullptr, g.code == JF_SCALE_F16 ? JF_FP_F16 : JF_FP_F32, so.first, so.second,
                                   out.back().data_ptr(), oc, (int)splitk, nbytes ? ws.data_ptr() : nullptr, nbytes, current_stream(x.q)),
                     "linear_backward");
        }
        if (bias_grad) out.push_back(block_colsum(g.q, g.s));
        return out;
    }
    if (dgrad_quantize) {
        out.push_back(fresh(with_last(g.q, w.C), g.q.options()));
        out.push_back(fresh(with_last(g.s, w.C / QB), g.s.options()));
        pybind11::gil_scoped_release nogil;
        check_rc(jf_igemm_block_q(g.qp(), w.qp(), g.sp(), w.sp(), nullptr, nullptr, (int8_t *)out[0].data_ptr(), out[1].data_ptr(), (int)g.R,
                                  (int)w.C, (int)g.C, JF_B_KN, g.code, JF_SCALES_ROWMAJOR, JF_SCALES_KMAJOR, JF_ROUND_STOCHASTIC, so.first,
                                  so.second, nullptr, 0, current_stream(g.q)),
                 "linear_backward");
    } else {
        out.push_back(fresh(with_last(g.q, w.C), g.s.options()));
        pybind11::gil_scoped_release nogil;
        check_rc(jf_igemm_block_q_dequant(g.qp(), w.qp(), g.sp(), w.sp(), nullptr, nullptr, out[0].data_ptr(), (int)g.R, (int)w.C, (int)g.C,
                                          JF_B_KN, g.code, JF_SCALES_ROWMAJOR, JF_SCALES_KMAJOR, g.code == JF_SCALE_F16 ? JF_FP_F16 : JF_FP_F32,
                                          JF_ROUND_STOCHASTIC, so.first, so.second, current_stream(g.q)),
                 "linear_backward");
    }
    out.push_back(weight_gradient(x, g, GT, splitk, wgrad_dtype));
    if (bias_grad) out.push_back(block_colsum(g.q, g.s));
    return out;
}

// linear_backward followed by the GELU backward of its activation gradient (qmodel.py:249-253): (codes, scales, dW[, db])
std::vector<Tensor> linear_backward_gelu(const Tensor &X, const Tensor &SX, const Tensor &G, const Tensor &SG, const Tensor &W, const Tensor &SW,
                                         const Tensor &P, const Tensor &SP, int64_t approx, int64_t gelu_rounding, int64_t splitk,
                                         OptDtype wgrad_dtype, bool bias_grad)
{
    const Operand x(X, SX, "X"), g(G, SG, "G"), w(W, SW, "W"), p(P, SP, "PRE");
    same_kind(x, g); same_kind(x, w); same_kind(x, p);
    TORCH_CHECK(x.R == g.R && w.q.dim() == 2 && w.R == g.C && w.C == x.C && p.R == x.R && p.C == x.C, "operands do not match: X ", X.sizes(), ", G ",
                G.sizes(), ", W ", W.sizes(), ", PRE ", P.sizes());
    check_approx(approx);
    check_rounding(gelu_rounding, false);
    c10::DeviceGuard guard(x.q.device());
    const auto so = rng(JF_ROUND_STOCHASTIC, g.q, g.R * w.C, c10::nullopt, c10::nullopt);
    const auto go = rng(gelu_rounding, g.q, g.R * w.C, c10::nullopt, c10::nullopt);
    std::vector<Tensor> out{fresh(with_last(g.q, w.C), g.q.options()), fresh(with_last(g.s, w.C / QB), g.s.options())};
    {
        pybind11::gil_scoped_release nogil;
        check_rc(jf_igemm_block_q_gelu_bwd(g.qp(), w.qp(), g.sp(), w.sp(), p.qp(), p.sp(), (int8_t *)out[0].data_ptr(), out[1].data_ptr(), (int)g.R,
                                           (int)w.C, (int)g.C, g.code, JF_SCALES_ROWMAJOR, JF_SCALES_KMAJOR, (int)approx, so.first, so.second,
                                           (int)gelu_rounding, go.first, go.second, current_stream(g.q)),
                 "linear_backward_gelu");
    }
    out.push_back(weight_gradient(x, g, c10::nullopt, splitk, wgrad_dtype));
    if (bias_grad) out.push_back(block_colsum(g.q, g.s));
    return out;
}

}  // namespace

void register_jetfire_ops(pybind11::module &m)
{
    namespace py = pybind11;
    const py::object none = py::none();
    m.attr("ROUND_NEAREST") = JF_ROUND_NEAREST;
    m.attr("ROUND_STOCHASTIC") = JF_ROUND_STOCHASTIC;
    m.attr("ROUND_TRUNC") = JF_ROUND_TRUNC;
    m.attr("ROUND_STOCHASTIC_TRUNC") = JF_ROUND_STOCHASTIC_TRUNC;
    m.attr("GELU_ERF") = JF_GELU_ERF;
    m.attr("GELU_TANH") = JF_GELU_TANH;
    m.attr("B_NK") = JF_B_NK;
    m.attr("B_KN") = JF_B_KN;
    m.def("quantize", &quantize, py::arg("x"), py::arg("rounding") = JF_ROUND_NEAREST, py::arg("scale_dtype") = none,
          py::arg("transpose") = false, py::arg("amax_eps") = 0.0, py::arg("seed") = none, py::arg("offset") = none,
          "(codes, scales, transposed codes or None) of a float [R,C] tensor");
    m.def("quantize_slabs", &quantize_slabs, py::arg("slabs"), py::arg("rounding") = JF_ROUND_NEAREST,
          py::arg("scale_dtype") = none, py::arg("amax_eps") = 0.0, py::arg("seed") = none, py::arg("offset") = none,
          "block tensor of the column-wise concatenation of up to 4 slabs, read where they lie");
    m.def("quantize_many", &quantize_many, py::arg("xs"), py::arg("scale_dtype") = none,
          "[(codes, scales), ...] of up to 8 float tensors of one type, one launch, round to nearest");
    m.def("rowstats_fp", &rowstats_fp, py::arg("x"), "(mean, 1/sqrt(biased variance)) of the rows of a float tensor");
    m.def("dequantize", &dequantize, py::arg("q"), py::arg("s"), py::arg("out_dtype") = none);
    m.def("transpose_s8", &transpose_s8, py::arg("q"));
    m.def("rowstats", &rowstats, py::arg("q"), py::arg("s"), py::arg("eps") = 1e-5);
    m.def("layernorm_fwd", &layernorm_fwd, py::arg("q"), py::arg("s"), py::arg("gamma"), py::arg("beta"), py::arg("mean"), py::arg("rstd"));
    m.def("layernorm_bwd", &layernorm_bwd, py::arg("qx"), py::arg("sx"), py::arg("qg"), py::arg("sg"), py::arg("gamma"), py::arg("mean"),
          py::arg("rstd"), py::arg("rounding") = JF_ROUND_NEAREST, py::arg("want_dbeta") = true, py::arg("seed") = none,
          py::arg("offset") = none);
    m.def("layernorm_bwd_add", &layernorm_bwd_add, py::arg("qx"), py::arg("sx"), py::arg("qg"), py::arg("sg"), py::arg("gamma"),
          py::arg("mean"), py::arg("rstd"), py::arg("x1"), py::arg("rounding") = JF_ROUND_NEAREST, py::arg("add_rounding") = JF_ROUND_TRUNC,
          py::arg("want_dbeta") = true, py::arg("out_dtype") = none, py::arg("seed") = none, py::arg("offset") = none,
          py::arg("add_seed") = none, py::arg("add_offset") = none);
    m.def("gelu_fwd", &gelu_fwd, py::arg("q"), py::arg("s"), py::arg("approx") = JF_GELU_ERF, py::arg("amax_eps") = 5e-5);
    m.def("gelu_bwd", &gelu_bwd, py::arg("qx"), py::arg("sx"), py::arg("qg"), py::arg("sg"), py::arg("approx") = JF_GELU_ERF,
          py::arg("rounding") = JF_ROUND_NEAREST, py::arg("seed") = none, py::arg("offset") = none);
    m.def("add", &add, py::arg("x1"), py::arg("q2"), py::arg("s2"), py::arg("rounding") = JF_ROUND_TRUNC, py::arg("with_stats") = false,
          py::arg("out_dtype") = none, py::arg("seed") = none, py::arg("offset") = none,
          "(y1, codes, scales, mean or None, rstd or None)");
    m.def("attention_fwd", &attention_fwd, py::arg("q"), py::arg("k"), py::arg("v"), py::arg("batch"), py::arg("heads"),
          "(out [tokens, C], lse [batch*heads, T]) of causal self-attention; heads 32 or 64 wide");
    m.def("attention_bwd", &attention_bwd, py::arg("q"), py::arg("k"), py::arg("v"), py::arg("out"), py::arg("lse"), py::arg("gout"),
          py::arg("batch"), py::arg("heads"), "gradients of q, k, v side by side, [tokens, 3C]");
    m.def("attention_fwd_q", &attention_fwd_q, py::arg("q"), py::arg("k"), py::arg("v"), py::arg("batch"), py::arg("heads"),
          "attention_fwd and the block quantisation of its result: (out, lse, codes, scales)");
    m.def("attention_bwd_q", &attention_bwd_q, py::arg("q"), py::arg("k"), py::arg("v"), py::arg("out"), py::arg("lse"), py::arg("gout"),
          py::arg("batch"), py::arg("heads"), py::arg("seed") = none, py::arg("offset") = none, "(codes, scales) of attention_bwd's result, rounded stochastically");
    m.def("block_colsum", &block_colsum, py::arg("q"), py::arg("s"), "fp32 column sums of a block tensor (bias gradient)");
    m.def("linear_forward", &linear_forward, py::arg("x"), py::arg("sx"), py::arg("w"), py::arg("sw"), py::arg("quantized"),
          py::arg("bias") = none, py::arg("biasmax") = none);
    m.def("linear_forward_gelu", &linear_forward_gelu, py::arg("x"), py::arg("sx"), py::arg("w"), py::arg("sw"), py::arg("approx"),
          py::arg("amax_eps"), py::arg("bias") = none, py::arg("biasmax") = none);
    m.def("linear_backward", &linear_backward, py::arg("x"), py::arg("sx"), py::arg("g"), py::arg("sg"), py::arg("gt"), py::arg("w"),
          py::arg("sw"), py::arg("dgrad_quantize"), py::arg("splitk"), py::arg("wgrad_dtype"), py::arg("bias_grad"));
    m.def("linear_backward_gelu", &linear_backward_gelu, py::arg("x"), py::arg("sx"), py::arg("g"), py::arg("sg"), py::arg("w"), py::arg("sw"),
          py::arg("pre"), py::arg("spre"), py::arg("approx"), py::arg("gelu_rounding"), py::arg("splitk"), py::arg("wgrad_dtype"),
          py::arg("bias_grad"));
    m.def("igemm_block_q", &igemm_block_q, py::arg("A"), py::arg("B"), py::arg("sa"), py::arg("sb"), py::arg("b_layout") = JF_B_KN,
          py::arg("bias") = none, py::arg("biasmax") = none, py::arg("rounding") = JF_ROUND_NEAREST, py::arg("seed") = none,
          py::arg("offset") = none);
    m.def("igemm_block_q_gelu", &igemm_block_q_gelu, py::arg("A"), py::arg("B"), py::arg("sa"), py::arg("sb"),
          py::arg("approx") = JF_GELU_ERF, py::arg("amax_eps") = 5e-5, py::arg("bias") = none, py::arg("biasmax") = none);
    m.def("igemm_block_q_gelu_bwd", &igemm_block_q_gelu_bwd, py::arg("A"), py::arg("B"), py::arg("sa"), py::arg("sb"), py::arg("xq"),
          py::arg("xs"), py::arg("approx") = JF_GELU_ERF, py::arg("gelu_rounding") = JF_ROUND_STOCHASTIC, py::arg("seed") = none,
          py::arg("offset") = none, py::arg("gelu_seed") = none, py::arg("gelu_offset") = none);
    m.def("igemm_block_q_dequant", &igemm_block_q_dequant, py::arg("A"), py::arg("B"), py::arg("sa"), py::arg("sb"),
          py::arg("b_layout") = JF_B_KN, py::arg("out_dtype") = none, py::arg("bias") = none, py::arg("biasmax") = none,
          py::arg("rounding") = JF_ROUND_NEAREST, py::arg("seed") = none, py::arg("offset") = none);
}

}  // namespace jfext
