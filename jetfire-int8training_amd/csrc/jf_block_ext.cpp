// BlockQuantizeCUDA.jetfire.qblock -- one transformer block of the recipe (Jetfire/recipe.py: LayerNorm -> QKV -> attention ->
// projection -> residual add -> LayerNorm -> fc + GELU -> projection -> residual add, qmodel.py:86-268) as ONE autograd node in
// C++.  The same kernels in the same order with the same Philox counters as the recipe's separate Functions; what goes is the
// host work between them: some forty Python-level operator calls, views and autograd nodes per block and step, and one
// allocation per intermediate.  What the backward needs lives in one buffer, what only the call needs in another.
#include "bqc_common.h"

#include <algorithm>
#include <cmath>
#include <vector>

namespace jfext {
namespace {

using torch::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
using OptTensor = c10::optional<Tensor>;

// Carves a buffer into 256-byte aligned pieces: first pass (base = null) adds up the size, second hands out the addresses.
struct Carver {
    uint8_t *base;
    size_t used = 0;
    explicit Carver(uint8_t *b) : base(b) {}
    template <typename T = void> T *take(size_t bytes)
    {
        T *p = base ? (T *)(base + used) : nullptr;
        used += (bytes + 255) & ~(size_t)255;
        return p;
    }
};

struct Dims {
    int B, T, C, H, M;
    size_t m, c;
    size_t codes(size_t cols) const { return m * cols; }                     // INT8 codes of [M, cols]
    size_t scales(size_t cols) const { return m / 32 * (cols / 32) * 2; }    // binary16 scales
};

// kept for the backward
struct Saved {
    int8_t *qn, *qy, *q2, *qn2, *qh, *qa;
    void *sn, *sy, *s2, *sn2, *sh, *sa;
    void *qkv, *y;
    float *lse, *mean2, *rstd2;
    size_t carve(uint8_t *b, const Dims &d)
    {
        Carver k(b);
        auto block = [&](int8_t *&q, void *&s, size_t cols) { q = k.take<int8_t>(d.codes(cols)); s = k.take(d.scales(cols)); };
        block(qn, sn, d.c); block(qy, sy, d.c); block(q2, s2, d.c); block(qn2, sn2, d.c); block(qh, sh, 4 * d.c); block(qa, sa, 4 * d.c);
        qkv = k.take(d.m * 3 * d.c * 2); y = k.take(d.m * d.c * 2);
        lse = k.take<float>(d.m * d.H * 4); mean2 = k.take<float>(d.m * 4); rstd2 = k.take<float>(d.m * 4);
        return k.used;
    }
};

// needed by the forward only
struct ForwardTemp {
    float *mid, *rowsum, *rowsq;
    size_t carve(uint8_t *b, const Dims &d)
    {
        Carver k(b);
        mid = k.take<float>(d.m * d.c * 4);
        rowsum = k.take<float>(d.c / 32 * d.m * 4); rowsq = k.take<float>(d.c / 32 * d.m * 4);
        return k.used;
    }
};

// Both of them where no backward follows: what is dead makes room for what comes after it.  Of two block tensors of [M, C] one
// serves in turn as qn, qy and qn2, the other as q2; Q, K, V and the attention's result make room for the float sum and the hidden layer.  14
// bytes per element of [M, C] and the scales, where a call whose backward follows holds 25.
size_t carve_inference(uint8_t *b, const Dims &d, Saved &v, ForwardTemp &t)
{
    Carver k(b);
    v.qn = v.qy = v.qn2 = k.take<int8_t>(d.codes(d.c)); v.sn = v.sy = v.sn2 = k.take(d.scales(d.c));
    v.q2 = k.take<int8_t>(d.codes(d.c)); v.s2 = k.take(d.scales(d.c));
    v.lse = k.take<float>(d.m * d.H * 4); v.mean2 = k.take<float>(d.m * 4); v.rstd2 = k.take<float>(d.m * 4);
    t.rowsum = k.take<float>(d.c / 32 * d.m * 4); t.rowsq = k.take<float>(d.c / 32 * d.m * 4);
    Carver attention(b ? b + k.used : nullptr), mlp(attention.base);
    v.qkv = attention.take(d.m * 3 * d.c * 2); v.y = attention.take(d.m * d.c * 2);
    t.mid = mlp.take<float>(d.m * d.c * 4);
    v.qh = mlp.take<int8_t>(d.codes(4 * d.c)); v.sh = mlp.take(d.scales(4 * d.c));
    v.qa = mlp.take<int8_t>(d.codes(4 * d.c)); v.sa = mlp.take(d.scales(4 * d.c));
    return k.used + std::max(attention.used, mlp.used);
}

struct BackwardTemp {
    int8_t *qp, *qd, *qr, *qq;
    void *sp, *sd, *sr, *sq;
    void *res, *gy;
    float *delta, *ln1_terms, *ln2_terms;
    void *ws;
    size_t carve(uint8_t *b, const Dims &d, size_t res_bytes, size_t ws_bytes)
    {
        Carver k(b);
        qp = k.take<int8_t>(d.codes(4 * d.c)); sp = k.take(d.scales(4 * d.c));      // gradient at the GELU's input
        qd = k.take<int8_t>(d.codes(d.c)); sd = k.take(d.scales(d.c));              // at a LayerNorm's output
        qr = k.take<int8_t>(d.codes(d.c)); sr = k.take(d.scales(d.c));              // at the sum inside the block
        qq = k.take<int8_t>(d.codes(3 * d.c)); sq = k.take(d.scales(3 * d.c));      // at Q, K, V
        res = k.take(d.m * d.c * res_bytes); gy = k.take(d.m * d.c * 2);
        delta = k.take<float>(d.m * d.H * 4);
        ln1_terms = k.take<float>(d.m / 32 * d.c * 4); ln2_terms = k.take<float>(d.m / 32 * d.c * 4);
        ws = k.take(ws_bytes);
        return k.used;
    }
};

int fp_of(const Tensor &t, const char *name)
{
    if (t.scalar_type() == torch::kFloat16) return JF_FP_F16;
    if (t.scalar_type() == torch::kFloat32) return JF_FP_F32;
    TORCH_CHECK(t.scalar_type() == torch::kBFloat16, name, ": expected float16, float32 or bfloat16");
    return JF_FP_BF16;
}

// the tensors of a call, in the order the node's inputs have
enum { X, QX, SX, MEAN, RSTD, LN1, LN2, W_QKV, W_PROJ, W_FC, W_FC2, B_QKV, B_PROJ, B_FC, B_FC2, N_GRAD };   // differentiable
struct WeightOperand { Tensor q, s; };
struct BiasOperand { Tensor b, bmax; };

// What the kernels are told about a tensor is checked here, as the separate operators check theirs: all tensors of a call live on
// the GPU that its kernels are launched on (`like`), and codes and scales split into rows of the width they are read with.
bool matrix_of(const Tensor &t, int64_t R, int64_t C)
{
    return t.dim() >= 2 && t.size(-1) == C && t.numel() == R * C && t.is_contiguous();
}
void check_codes(const Tensor &q, const Tensor &s, int64_t R, int64_t C, const Tensor &like, const char *name)
{
    TORCH_CHECK(q.is_cuda() && s.is_cuda(), name, ": expected GPU tensors");
    TORCH_CHECK(q.device() == like.device() && s.device() == like.device(), name, ": codes and scales must be on ", like.device(), ", got ", q.device(),
                " and ", s.device());
    TORCH_CHECK(q.element_size() == 1 && s.scalar_type() == torch::kFloat16 && matrix_of(q, R, C) && matrix_of(s, R / QB, C / QB), name,
                ": expected contiguous codes of [", R, ", ", C, "] with float16 scales, got ", q.sizes(), " and ", s.sizes());
}
const float *f32_vec(const Tensor &v, int64_t n, const Tensor &like, const char *name)
{
    TORCH_CHECK(v.is_cuda(), name, ": expected a GPU tensor");
    TORCH_CHECK(v.scalar_type() == torch::kFloat32 && v.is_contiguous() && v.numel() == n && v.device() == like.device(), name, ": expected ", n,
                " contiguous float32 values on ", like.device());
    return v.data_ptr<float>();
}
void check_residual(const Tensor &x, int64_t R, int64_t C, const Tensor &like, const char *name)
{
    TORCH_CHECK(x.is_cuda(), name, ": expected a GPU tensor");
    TORCH_CHECK(x.device() == like.device() && matrix_of(x, R, C), name, ": expected a contiguous [B, T, C] tensor of ", R, " rows of ", C, " on ",
                like.device());
}

struct BlockForward {
    Tensor saved, fp, q, s, mean, rstd;
};

// Forward of a block.  weights: qkv, projection, fc, second projection.  biases: empty or one (bias, max|bias|) pair each.
// keep: leave what the backward needs in `saved` (else it stays undefined).
BlockForward forward_impl(const Dims &d, const Tensor &x, const Tensor &qx, const Tensor &sx, const Tensor &mean, const Tensor &rstd,
                          const Tensor &ln1, const Tensor &ln2, const std::vector<WeightOperand> &w, const std::vector<BiasOperand> &bias,
                          torch::ScalarType out_dtype, bool keep)
{
    const int64_t M = d.M, C = d.C;
    check_residual(x, M, C, x, "x");
    check_codes(qx, sx, M, C, x, "qx");
    check_codes(w[0].q, w[0].s, 3 * C, C, x, "w_qkv"); check_codes(w[1].q, w[1].s, C, C, x, "w_attn_proj");
    check_codes(w[2].q, w[2].s, 4 * C, C, x, "w_fc"); check_codes(w[3].q, w[3].s, C, 4 * C, x, "w_mlp_proj");
    const float *g1 = f32_vec(ln1, C, x, "ln_1"), *g2 = f32_vec(ln2, C, x, "ln_2"), *mu = f32_vec(mean, M, x, "mean"), *rs = f32_vec(rstd, M, x, "rstd");
    const float *bp[4] = {}, *bm[4] = {};
    const int64_t widths[4] = {3 * C, C, 4 * C, C};
    for (size_t i = 0; i < bias.size(); ++i) { bp[i] = f32_vec(bias[i].b, widths[i], x, "bias"); bm[i] = f32_vec(bias[i].bmax, 1, x, "biasmax"); }
    const int xc = fp_of(x, "x");

    c10::DeviceGuard guard(x.device());
    const auto opt = x.options().requires_grad(false);
    Saved v;
    ForwardTemp t;
    BlockForward r;
    Tensor temp = fresh({(int64_t)(keep ? t.carve(nullptr, d) : carve_inference(nullptr, d, v, t))}, opt.dtype(torch::kUInt8));
    if (keep) {
        r.saved = fresh({(int64_t)v.carve(nullptr, d)}, opt.dtype(torch::kUInt8));
        v.carve((uint8_t *)r.saved.data_ptr(), d);
        t.carve((uint8_t *)temp.data_ptr(), d);
    } else {
        carve_inference((uint8_t *)temp.data_ptr(), d, v, t);
    }
    r.fp = fresh({d.B, d.T, C}, opt.dtype(out_dtype));
    r.q = fresh({d.B, d.T, C}, opt.dtype(torch::kFloat8_e4m3fn));
    r.s = fresh({d.B, d.T / QB, C / QB}, opt.dtype(torch::kFloat16));
    r.mean = fresh({d.B, d.T}, opt.dtype(torch::kFloat32));
    r.rstd = fresh({d.B, d.T}, opt.dtype(torch::kFloat32));
    const jf_stream_t st = current_stream(x);
    constexpr int RM = JF_SCALES_ROWMAJOR, F16 = JF_SCALE_F16;
    const int m = d.M, c = d.C;
    auto codes = [](const Tensor &a) { return (const int8_t *)a.data_ptr(); };
    const int8_t *qx_ = codes(qx);
    auto project_add = [&](const int8_t *a, const void *sa, int i, int k, const void *x1, int x1c, void *y, int yc, int8_t *q, void *s) {
        check_rc(jf_igemm_block_q_add(a, codes(w[i].q), sa, w[i].s.data_ptr(), bp[i], bm[i], x1, x1c, JF_ROUND_TRUNC, y, yc, q, s, t.rowsum,
                                      t.rowsq, m, c, k, F16, RM, RM, st), "projection and residual add");
    };
    check_rc(jf_layernorm_fwd(qx_, sx.data_ptr(), g1, nullptr, mu, rs, m, c, F16, v.qn, v.sn, st), "layernorm");
    check_rc(jf_igemm_block_q_dequant(v.qn, codes(w[0].q), v.sn, w[0].s.data_ptr(), bp[0], bm[0], v.qkv, m, 3 * c, c, JF_B_NK, F16, RM, RM, JF_FP_F16,
                                      JF_ROUND_NEAREST, 0, 0, st), "qkv projection");
    c10::Half *qkv = (c10::Half *)v.qkv;
    check_rc(jf_attention_fwd_q(qkv, qkv + c, qkv + 2 * c, 3 * c, d.B, d.H, d.T, c / d.H, (float)(1.0 / std::sqrt((double)(c / d.H))), v.y, v.lse,
                                v.qy, v.sy, st),
             "attention");
    project_add(v.qy, v.sy, 1, c, x.data_ptr(), xc, t.mid, JF_FP_F32, v.q2, v.s2);
    check_rc(jf_layernorm_fwd_sums(v.q2, v.s2, g2, nullptr, t.rowsum, t.rowsq, m, c, F16, v.mean2, v.rstd2, v.qn2, v.sn2, st), "layernorm");
    check_rc(jf_igemm_block_q_gelu(v.qn2, codes(w[2].q), v.sn2, w[2].s.data_ptr(), bp[2], bm[2], v.qh, v.sh, v.qa, v.sa, m, 4 * c, c, F16, RM, RM,
                                   JF_GELU_ERF, 5e-5f, st), "fc");
    project_add(v.qa, v.sa, 3, 4 * c, t.mid, JF_FP_F32, r.fp.data_ptr(), fp_of(r.fp, "out"), (int8_t *)r.q.data_ptr(), r.s.data_ptr());
    check_rc(jf_rowstats_finish(t.rowsum, t.rowsq, m, c / QB, c, r.mean.data_ptr<float>(), r.rstd.data_ptr<float>(), st), "row statistics");
    return r;
}

// (seed, offset) pairs of the backward's stochastic operators, in the order the separate Functions draw them
struct Noise {
    uint64_t seed, offset;
};

struct BlockNode : torch::autograd::Function<BlockNode> {
    // the N_GRAD differentiable inputs (absent biases: no value), the coded weights and the bias pairs
    static variable_list forward(AutogradContext *ctx, Tensor x_, Tensor qx, Tensor sx, Tensor mean, Tensor rstd, Tensor ln1, Tensor ln2, Tensor w1,
                                 Tensor w2, Tensor w3, Tensor w4, OptTensor b1, OptTensor b2, OptTensor b3, OptTensor b4,
                                 const std::vector<WeightOperand> &w,
                                 const std::vector<BiasOperand> &bias, int64_t heads, torch::ScalarType out_dtype, bool keep)
    {
        const variable_list in{x_, qx, sx, mean, rstd, ln1, ln2, w1, w2, w3, w4};
        const Tensor &x = in[X];
        const Dims d = dims_of(x, heads);
        BlockForward r = forward_impl(d, x, in[QX], in[SX], in[MEAN], in[RSTD], in[LN1], in[LN2], w, bias, out_dtype, keep);
        if (!keep) return {r.fp, r.q, r.s, r.mean, r.rstd};
        ctx->set_materialize_grads(false);
        variable_list held{in[QX], in[SX], in[MEAN], in[RSTD], in[LN1], in[LN2]};
        for (auto &o : w) { held.push_back(o.q); held.push_back(o.s); }
        held.push_back(r.saved);
        ctx->save_for_backward(std::move(held));
        auto &data = ctx->saved_data;
        data["shape"] = std::vector<int64_t>{d.B, d.T, d.C, d.H};
        data["types"] = std::vector<int64_t>{(int64_t)x.scalar_type(), (int64_t)in[W_QKV].scalar_type(), (int64_t)(b1 ? b1->scalar_type() : torch::kFloat32)};
        data["bias"] = !bias.empty();
        return {r.fp, r.q, r.s, r.mean, r.rstd};
    }

    static Dims dims_of(const Tensor &x, int64_t heads)
    {
        TORCH_CHECK(x.dim() == 3, "x: expected [B, T, C]");
        const int64_t B = x.size(0), T = x.size(1), C = x.size(2);
        TORCH_CHECK(T % QB == 0 && C % QB == 0 && heads > 0 && C % heads == 0, "x ", x.sizes(), " does not split into blocks and ", heads, " heads");
        return {(int)B, (int)T, (int)C, (int)heads, (int)(B * T), (size_t)(B * T), (size_t)C};
    }

    static variable_list backward(AutogradContext *ctx, const variable_list &grads)
    {
        const auto shape = ctx->saved_data["shape"].toIntVector(), types = ctx->saved_data["types"].toIntVector();
        const bool with_bias = ctx->saved_data["bias"].toBool();
        const int64_t B = shape[0], T = shape[1], C = shape[2], M = B * T;
        const Dims d = {(int)B, (int)T, (int)C, (int)shape[3], (int)M, (size_t)M, (size_t)C};
        const auto res_type = (torch::ScalarType)types[0], w_type = (torch::ScalarType)types[1], b_type = (torch::ScalarType)types[2];
        TORCH_CHECK(grads[0].defined() && grads[1].defined() && grads[2].defined(), "the block's gradient needs its floating part, codes and scales");
        const variable_list s = ctx->get_saved_variables();
        const Tensor &qx = s[0], &sx = s[1], &mean = s[2], &rstd = s[3], &ln1 = s[4], &ln2 = s[5];
        const WeightOperand w[4] = {{s[6], s[7]}, {s[8], s[9]}, {s[10], s[11]}, {s[12], s[13]}};
        const Tensor fpg = grads[0].contiguous(), qg = grads[1].contiguous(), sg = grads[2].contiguous();
        check_residual(fpg, M, C, qx, "gradient");
        check_codes(qg, sg, M, C, qx, "gradient");

        c10::DeviceGuard guard(qx.device());
        const auto opt = qx.options().requires_grad(false);
        Saved v;
        v.carve((uint8_t *)s[14].data_ptr(), d);
        const int m = d.M, c = d.C;
        // [C_out, C_in] of the weights
        const int wrows[4] = {3 * c, c, 4 * c, c}, wcols[4] = {c, c, c, 4 * c};
        size_t ws_bytes = jf_wgrad_many_workspace_bytes(4, wrows, wcols, m);
        if (with_bias) ws_bytes = std::max(ws_bytes, jf_block_colsum_workspace_bytes(m, 4 * c));
        BackwardTemp t;
        const size_t res_bytes = torch::elementSize(res_type);
        Tensor temp = fresh({(int64_t)t.carve(nullptr, d, res_bytes, ws_bytes)}, opt.dtype(torch::kUInt8));
        t.carve((uint8_t *)temp.data_ptr(), d, res_bytes, ws_bytes);

        variable_list out(N_GRAD + 5);                         // (one entry per argument of forward)
        out[X] = fresh({B, T, C}, opt.dtype(res_type));
        out[QX] = fresh({B, T, C}, opt.dtype(torch::kFloat8_e4m3fn));
        out[SX] = fresh({B, T / QB, C / QB}, opt.dtype(torch::kFloat16));
        out[LN1] = fresh({C}, opt.dtype(torch::kFloat32));
        out[LN2] = fresh({C}, opt.dtype(torch::kFloat32));
        for (int i = 0; i < 4; ++i) out[W_QKV + i] = fresh({wrows[i], wcols[i]}, opt.dtype(w_type));
        if (with_bias)
            for (int i = 0; i < 4; ++i) out[B_QKV + i] = fresh({wrows[i]}, opt.dtype(torch::kFloat32));
        const int resc = fp_of(out[X], "residual"), wc = fp_of(out[W_QKV], "weight"), fpgc = fp_of(fpg, "gradient");

        // Philox counters, drawn in the order of the separate Functions (the reservations below are what each would make)
        const int64_t n1 = M * C, n3 = 3 * M * C, n4 = 4 * M * C;
        Noise z[10];
        {
            const int64_t sizes[10] = {n4, n4, n1, n1, n1, n1, n3, n1, n1, n1};
            at::Generator gen = default_generator(qx.device().index());
            std::lock_guard<std::mutex> g(gen.mutex());
            const uint64_t seed = gen.current_seed();
            uint64_t off = gen.get_offset();
            for (int i = 0; i < 10; ++i) { z[i] = {seed, off}; off += reserve_calls(sizes[i]); }
            gen.set_offset(off);
        }
        const jf_stream_t st = current_stream(qx);
        constexpr int RM = JF_SCALES_ROWMAJOR, KM = JF_SCALES_KMAJOR, F16 = JF_SCALE_F16, SR = JF_ROUND_STOCHASTIC;
        auto codes = [](const Tensor &a) { return (const int8_t *)a.data_ptr(); };
        // The weight gradients run together, with the last activation gradient: one launch has tiles for the whole chip where each
        // alone leaves a last round half empty, and one more at the end adds what is left to add, the parts of K splits and the
        // LayerNorm weights' gradients.
        const int8_t *wg[4], *wx[4];
        const void *wgs[4], *wxs[4];
        auto wgrad = [&](int i, const int8_t *g, const void *gs, const int8_t *xq, const void *xs) {
            wg[i] = g; wgs[i] = gs; wx[i] = xq; wxs[i] = xs;
            if (with_bias) check_rc(jf_block_colsum(g, gs, m, wrows[i], F16, out[B_QKV + i].data_ptr<float>(), t.ws, ws_bytes, st), "bias gradient");
        };
        // MLP: second projection with the GELU's backward in its epilogue, fc, LayerNorm with the residual add behind it
        check_rc(jf_igemm_block_q_gelu_bwd(codes(qg), codes(w[3].q), sg.data_ptr(), w[3].s.data_ptr(), v.qh, v.sh, t.qp, t.sp, m, 4 * c, c, F16, RM, KM,
                                           JF_GELU_ERF, z[0].seed, z[0].offset, SR, z[1].seed, z[1].offset, st), "gradient of the MLP's projection");
        wgrad(3, codes(qg), sg.data_ptr(), v.qa, v.sa);
        check_rc(jf_igemm_block_q(t.qp, codes(w[2].q), t.sp, w[2].s.data_ptr(), nullptr, nullptr, t.qd, t.sd, m, c, 4 * c, JF_B_KN, F16, RM, KM, SR,
                                  z[2].seed, z[2].offset, nullptr, 0, st), "gradient of fc");
        wgrad(2, t.qp, t.sp, v.qn2, v.sn2);
        check_rc(jf_layernorm_bwd_add_strips(v.q2, v.s2, t.qd, t.sd, ln2.data_ptr<float>(), v.mean2, v.rstd2, m, c, F16, SR, z[3].seed, z[3].offset,
                                      fpg.data_ptr(), fpgc, JF_ROUND_STOCHASTIC_TRUNC, z[4].seed, z[4].offset, t.res, resc, t.qr, t.sr,
                                      t.ln2_terms, st), "gradient of layernorm");
        // attention: output projection, the attention itself, QKV, LayerNorm with the residual add behind it
        check_rc(jf_igemm_block_q_dequant(t.qr, codes(w[1].q), t.sr, w[1].s.data_ptr(), nullptr, nullptr, t.gy, m, c, c, JF_B_KN, F16, RM, KM, JF_FP_F16,
                                          SR, z[5].seed, z[5].offset, st), "gradient of the attention's projection");
        wgrad(1, t.qr, t.sr, v.qy, v.sy);
        const c10::Half *qkv = (const c10::Half *)v.qkv;
        check_rc(jf_attention_bwd_q(qkv, qkv + c, qkv + 2 * c, 3 * c, v.y, t.gy, v.lse, d.B, d.H, d.T, c / d.H, (float)(1.0 / std::sqrt((double)(c / d.H))),
                                    t.qq, t.sq, z[6].seed, z[6].offset, t.delta, st), "gradient of attention");
        wgrad(0, t.qq, t.sq, v.qn, v.sn);
        void *const gw[4] = {out[W_QKV].data_ptr(), out[W_PROJ].data_ptr(), out[W_FC].data_ptr(), out[W_FC2].data_ptr()};
        check_rc(jf_wgrad_many_dgrad(codes(w[0].q), w[0].s.data_ptr(), t.qd, t.sd, z[7].seed, z[7].offset, 4, wg, wgs, wx, wxs, gw, wrows, wcols, m, F16,
                                     wc, t.ws, ws_bytes, st), "gradient of qkv and weight gradients");
        check_rc(jf_layernorm_bwd_add_strips(codes(qx), sx.data_ptr(), t.qd, t.sd, ln1.data_ptr<float>(), mean.data_ptr<float>(), rstd.data_ptr<float>(), m, c, F16,
                                      SR, z[8].seed, z[8].offset, t.res, resc, JF_ROUND_STOCHASTIC_TRUNC, z[9].seed, z[9].offset, out[X].data_ptr(), resc,
                                      (int8_t *)out[QX].data_ptr(), out[SX].data_ptr(), t.ln1_terms, st),
                 "gradient of layernorm");
        const float *const terms[2] = {t.ln1_terms, t.ln2_terms};
        float *const gln[2] = {out[LN1].data_ptr<float>(), out[LN2].data_ptr<float>()};
        const int widths[2] = {c, c};
        check_rc(jf_wgrad_many_finish(4, wg, wgs, wx, wxs, gw, wrows, wcols, m, F16, wc, 2, terms, widths, gln, t.ws, ws_bytes, st), "weight gradients");
        if (with_bias && b_type != torch::kFloat32)
            for (int i = 0; i < 4; ++i) out[B_QKV + i] = out[B_QKV + i].to(b_type);
        return out;
    }
};

// (fp, codes as float8, scales, mean, rstd) of a block.  params: ln_1, ln_2, w_qkv, w_attn_proj, w_fc, w_mlp_proj (the
// parameters: where their gradients go); codes: (codes, scales) of the four weights; biases: the four bias parameters and
// their (float32 bias, max|bias|) pairs, or empty.
variable_list qblock(const Tensor &x_, const Tensor &qx_, const Tensor &sx_, const Tensor &mean_, const Tensor &rstd_, std::vector<Tensor> params,
                     const std::vector<std::tuple<Tensor, Tensor>> &codes, const std::vector<Tensor> &bias_params,
                     const std::vector<std::tuple<Tensor, Tensor>> &bias_pairs, int64_t heads, torch::ScalarType out_dtype)
{
    TORCH_CHECK(params.size() == 6 && codes.size() == 4 && (bias_params.empty() || bias_params.size() == 4) && bias_pairs.size() == bias_params.size(),
                "qblock: expected 6 parameters, 4 coded weights and 0 or 4 biases");
    // strides, and types of the statistics, are brought to what the kernels read, as the separate operators do
    const Tensor x = x_.contiguous(), qx = qx_.contiguous(), sx = sx_.contiguous();
    const Tensor mean = mean_.to(torch::kFloat32).contiguous(), rstd = rstd_.to(torch::kFloat32).contiguous();
    params[0] = params[0].contiguous(); params[1] = params[1].contiguous();
    std::vector<WeightOperand> w;
    std::vector<BiasOperand> bias;
    for (auto &p : codes) w.push_back({std::get<0>(p), std::get<1>(p)});
    for (auto &p : bias_pairs) bias.push_back({std::get<0>(p), std::get<1>(p)});
    const auto b = [&](size_t i) { return bias_params.empty() ? OptTensor() : OptTensor(bias_params[i]); };
    // the condition under which autograd will ask for a backward
    variable_list inputs{x, qx, sx, mean, rstd};
    inputs.insert(inputs.end(), params.begin(), params.end());
    inputs.insert(inputs.end(), bias_params.begin(), bias_params.end());
    const bool keep = c10::GradMode::is_enabled() && std::any_of(inputs.begin(), inputs.end(), [](const Tensor &t) { return t.requires_grad(); });
    return BlockNode::apply(x, qx, sx, mean, rstd, params[0], params[1], params[2], params[3], params[4], params[5], b(0), b(1), b(2), b(3), w, bias,
                            heads, out_dtype, keep);
}

}  // namespace

void register_block(pybind11::module &m)
{
    namespace py = pybind11;
    m.def("qblock", &qblock, py::arg("x"), py::arg("qx"), py::arg("sx"), py::arg("mean"), py::arg("rstd"), py::arg("params"), py::arg("codes"),
          py::arg("bias_params"), py::arg("bias_pairs"), py::arg("heads"), py::arg("out_dtype"), py::call_guard<py::gil_scoped_release>());
}

}  // namespace jfext
