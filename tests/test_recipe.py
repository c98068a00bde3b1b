"""End-to-end check of the operator sequence of the INT8 GPT-2 recipe (our counterpart of the autograd
Functions of INT8_GPT2/qmodel.py) against an fp32 torch transformer block: outputs and gradients agree within
quantisation noise, and a small stack trains."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def ref_block(x, blk):
    C = x.shape[-1]
    B, T, _ = x.shape
    h = F.layer_norm(x, (C,), blk.ln_1, None, 0.0)
    qkv = F.linear(h, blk.w_qkv, blk.b_qkv)
    q, k, v = (t.view(B, T, blk.n_head, C // blk.n_head).transpose(1, 2) for t in qkv.split(C, dim=2))
    y = F.scaled_dot_product_attention(q, k, v, is_causal=True).transpose(1, 2).contiguous().view(B, T, C)
    x = x + F.linear(y, blk.w_attn_proj, blk.b_attn_proj)
    h = F.layer_norm(x, (C,), blk.ln_2, None, 0.0)
    return x + F.linear(F.gelu(F.linear(h, blk.w_fc, blk.b_fc)), blk.w_mlp_proj, blk.b_mlp_proj)


def cos(a, b):
    return float(F.cosine_similarity(a.detach().reshape(-1).float(), b.detach().reshape(-1).float(), dim=0))


def test_one_block_matches_fp32_reference():
    from recipe import QStack
    torch.manual_seed(0)
    B, T, C, H = 2, 64, 128, 4
    model = QStack(1, C, H).cuda()
    with torch.no_grad():
        for p in model.parameters():
            if p.dim() == 1:
                p.add_(0.1 * torch.randn_like(p))
    x = torch.randn(B, T, C, device="cuda", requires_grad=True)
    w = torch.randn(B, T, C, device="cuda")
    out = model(x)
    assert out.shape == x.shape and out.dtype == torch.float32
    (out * w).sum().backward()
    got = {n: p.grad.clone() for n, p in model.named_parameters()}
    gx = x.grad.clone()
    for p in model.parameters():
        p.grad = None
    x2 = x.detach().clone().requires_grad_(True)
    ref = ref_block(x2, model.blocks[0])
    (ref * w).sum().backward()
    assert cos(out, ref) > 0.999
    assert cos(gx, x2.grad) > 0.99
    for n, p in model.named_parameters():
        assert got[n].shape == p.shape and got[n].dtype == p.dtype
        assert cos(got[n], p.grad) > 0.97, n


def test_block_with_linear_biases_matches_fp32_reference():
    """QBlock(bias=True): the four biases enter in the GEMM epilogues and their gradients are the column sums of the
    layers' quantised output gradients; against the fp32 block with the same biases."""
    from recipe import QStack
    torch.manual_seed(4)
    B, T, C, H = 2, 128, 256, 4
    model = QStack(1, C, H, bias=True).cuda()
    names = [n for n, _ in model.named_parameters()]
    assert sum(".b_" in n for n in names) == 4
    with torch.no_grad():
        for n, p in model.named_parameters():
            if p.dim() == 1:
                p.add_((0.3 if ".b_" in n else 0.1) * torch.randn_like(p))
    x = torch.randn(B, T, C, device="cuda", requires_grad=True)
    w = torch.randn(B, T, C, device="cuda")
    out = model(x)
    (out * w).sum().backward()
    got = {n: p.grad.clone() for n, p in model.named_parameters()}
    gx = x.grad.clone()
    for p in model.parameters():
        p.grad = None
    x2 = x.detach().clone().requires_grad_(True)
    ref = ref_block(x2, model.blocks[0])
    (ref * w).sum().backward()
    assert cos(out, ref) > 0.999
    assert cos(gx, x2.grad) > 0.99
    for n, p in model.named_parameters():
        assert got[n].shape == p.shape and got[n].dtype == p.dtype
        assert cos(got[n], p.grad) > (0.99 if ".b_" in n else 0.97), (n, cos(got[n], p.grad))
    # without the biases the output differs: they are really applied
    with torch.no_grad():
        saved = [p.clone() for n, p in model.named_parameters() if ".b_" in n]
        for n, p in model.named_parameters():
            if ".b_" in n:
                p.zero_()
        assert cos(model(x), ref) < 0.999
        for (n, p), v in zip([(n, p) for n, p in model.named_parameters() if ".b_" in n], saved):
            p.copy_(v)
        assert torch.equal(model(x), out)                          # cached bias operands follow the parameter's version


def test_xl_width_block_matches_fp32_reference():
    """One block at the GPT-2 XL widths (1600 / 4800 / 6400, 25 heads) on 2048 tokens: every operator at its real
    row length (LayerNorm rows of 50 blocks, GELU rows of 200), weight gradients through the K split."""
    from recipe import QStack
    torch.manual_seed(3)
    B, T, C, H = 2, 1024, 1600, 25
    model = QStack(1, C, H).cuda()
    x = torch.randn(B, T, C, device="cuda", requires_grad=True)
    w = torch.randn(B, T, C, device="cuda")
    out = model(x)
    (out * w).sum().backward()
    got = {n: p.grad.clone() for n, p in model.named_parameters()}
    gx = x.grad.clone()
    for p in model.parameters():
        p.grad = None
    x2 = x.detach().clone().requires_grad_(True)
    ref = ref_block(x2, model.blocks[0])
    (ref * w).sum().backward()
    assert torch.isfinite(out).all() and cos(out, ref) > 0.999
    assert cos(gx, x2.grad) > 0.99
    for n, p in model.named_parameters():
        assert torch.isfinite(got[n]).all() and cos(got[n], p.grad) > 0.97, (n, cos(got[n], p.grad))


def test_twelve_layer_stack_matches_fp32_reference():
    """Twelve blocks (the depth of GPT-2 small; the reference stacks n_layer blocks, INT8_GPT2/qmodel.py:418-446):
    forward output after every depth and the gradients of every layer's weights against the same stack in fp32.
    Quantisation noise grows through the depth (each block requantises its residual stream, every backward GEMM rounds
    stochastically), so the thresholds are per depth (measured: forward 0.99995 at depth 12, weight gradients 0.9988
    and better at every depth); a wrong operand, scale or layout anywhere in the chain fails them by far."""
    from recipe import QStack
    torch.manual_seed(7)
    L, B, T, C, H = 12, 2, 128, 256, 4
    model = QStack(L, C, H).cuda()
    with torch.no_grad():
        for p in model.parameters():
            if p.dim() == 1:
                p.add_(0.1 * torch.randn_like(p))
    x = torch.randn(B, T, C, device="cuda", requires_grad=True)
    w = torch.randn(B, T, C, device="cuda")
    # forward at every depth: a prefix of the stack is a stack
    x_ref = x.detach()
    depth_cos = []
    for d in range(1, L + 1):
        x_ref = ref_block(x_ref, model.blocks[d - 1])
        prefix = QStack(0, C, H)
        prefix.blocks = model.blocks[:d]
        with torch.no_grad():
            depth_cos.append(cos(prefix(x.detach()), x_ref))
    print("forward cosine per depth:", [round(c, 5) for c in depth_cos], flush=True)
    for d, c in enumerate(depth_cos, 1):
        assert c > 0.9999 - 1e-5 * d, (d, c)
    # backward through all twelve
    out = model(x)
    (out * w).sum().backward()
    got = {n: p.grad.clone() for n, p in model.named_parameters()}
    gx = x.grad.clone()
    for p in model.parameters():
        p.grad = None
    x2 = x.detach().clone().requires_grad_(True)
    h = x2
    for blk in model.blocks:
        h = ref_block(h, blk)
    (h * w).sum().backward()
    print("output / input-gradient cosine:", round(cos(out, h), 5), round(cos(gx, x2.grad), 5), flush=True)
    assert cos(out, h) > 0.9998
    assert cos(gx, x2.grad) > 0.99, cos(gx, x2.grad)
    worst = {}
    for n, p in model.named_parameters():
        layer = int(n.split(".")[1])
        c = cos(got[n], p.grad)
        worst[layer] = min(worst.get(layer, 1.0), c)
        assert torch.isfinite(got[n]).all()
    print("worst weight-gradient cosine per layer:", {k: round(v, 4) for k, v in sorted(worst.items())}, flush=True)
    for layer, c in worst.items():
        # the gradient reaching layer l has passed through L-1-l quantised backward blocks
        assert c > 0.997 - 0.0003 * (L - 1 - layer), (layer, c)


def test_bfloat16_stream_between_blocks():
    """The reference casts the fp sum that leaves a block to bfloat16 (qmodel.py:228); here the add kernels write it (and
    the gradient that flows back into a bfloat16 residual) in that type.  Input and its gradient keep float32; the INT8
    stream is quantised from the float32 sums, so the result is as close to the fp32 stack as with a float32 stream up to
    the rounding of the residual."""
    from recipe import QStack
    torch.manual_seed(11)
    L, B, T, C, H = 3, 2, 128, 256, 4
    model = QStack(L, C, H, stream_dtype=torch.bfloat16).cuda()
    x = torch.randn(B, T, C, device="cuda", requires_grad=True)
    w = torch.randn(B, T, C, device="cuda")
    out = model(x)
    assert out.dtype == torch.bfloat16
    out.backward(w.to(torch.bfloat16))
    assert x.grad.dtype == torch.float32
    got = {n: p.grad.clone() for n, p in model.named_parameters()}
    gx = x.grad.clone()
    for p in model.parameters():
        p.grad = None
    x2 = x.detach().clone().requires_grad_(True)
    h = x2
    for blk in model.blocks:
        h = ref_block(h, blk)
    (h * w).sum().backward()
    print("bf16 stream: output / input-gradient cosine:", round(cos(out, h), 5), round(cos(gx, x2.grad), 5), flush=True)
    assert cos(out, h) > 0.9995
    assert cos(gx, x2.grad) > 0.99
    for n, p in model.named_parameters():
        assert got[n].dtype == p.dtype and torch.isfinite(got[n]).all()
        assert cos(got[n], p.grad) > 0.99, (n, cos(got[n], p.grad))


def test_merged_node_equals_the_two_functions():
    """AttentionOutMLP is AttentionOut followed by MLPResidual: same kernels in the same order, so with the same noise
    offsets the outputs and every gradient are the same bits."""
    import recipe
    torch.manual_seed(5)
    B, T, C = 2, 64, 128
    blk = recipe.QBlock(C, 4).cuda()
    res = torch.randn(B, T, C, device="cuda")
    y = torch.randn(B, T, C, device="cuda").half()
    gout = torch.randn(B, T, C, device="cuda")

    def run(merged):
        torch.manual_seed(123)                                    # rewinds the stochastic-rounding stream
        r, yy = res.clone().requires_grad_(True), y.clone().requires_grad_(True)
        for p in blk.parameters():
            p.grad = None
        if merged:
            fp, q, s, m, rs = recipe.AttentionOutMLP.apply(r, yy, blk.w_attn_proj, blk.w_fc, blk.w_mlp_proj, blk.ln_2, torch.float32)
        else:
            a = recipe.AttentionOut.apply(r, yy, blk.w_attn_proj)
            fp, q, s, m, rs = recipe.MLPResidual.apply(*a[:3], blk.w_fc, blk.w_mlp_proj, blk.ln_2, a[3], a[4])
        out = recipe.StreamEnd.apply(fp, q, s)
        out.backward(gout)
        return [fp.detach(), q.view(torch.int8), s, m, rs, r.grad, yy.grad, blk.w_attn_proj.grad, blk.w_fc.grad,
                blk.w_mlp_proj.grad, blk.ln_2.grad]
    for i, (a, b) in enumerate(zip(run(True), run(False))):
        assert torch.equal(a, b), i


def test_small_stack_trains():
    from recipe import QStack
    torch.manual_seed(1)
    B, T, C, H = 2, 64, 128, 4
    model = QStack(2, C, H).cuda()
    opt = torch.optim.AdamW(model.parameters(), lr=3e-3)
    x = torch.randn(B, T, C, device="cuda")
    target = torch.roll(x, 1, dims=1) * 0.5 + 0.1
    losses = []
    for _ in range(20):
        opt.zero_grad(set_to_none=True)
        loss = F.mse_loss(model(x), target)
        loss.backward()
        opt.step()
        losses.append(float(loss.detach()))
    assert losses[-1] < 0.8 * losses[0], losses
    assert all(torch.isfinite(p).all() for p in model.parameters())


def test_weight_codes_are_cached_per_weight_version():
    """A weight is quantised once per value: repeated forwards reuse its codes, an optimizer-style in-place update
    re-quantises it, and cached codes are the ones a fresh quantisation gives."""
    import recipe
    from Nonlinear import int8_quantize
    torch.manual_seed(2)
    model = recipe.QStack(1, 128, 4).cuda()
    x = torch.randn(2, 64, 128, device="cuda")
    recipe.weight_codes.clear()
    recipe.weight_codes.hits = recipe.weight_codes.misses = 0
    with torch.no_grad():
        y0 = model(x)
        assert (recipe.weight_codes.misses, recipe.weight_codes.hits) == (4, 0)
        y1 = model(x)
        assert (recipe.weight_codes.misses, recipe.weight_codes.hits) == (4, 4)
        assert torch.equal(y0, y1)
        w = model.blocks[0].w_fc
        q, s = recipe.weight_codes.get(w)
        q2, s2 = int8_quantize(w.detach(), 32)
        assert torch.equal(q, q2) and torch.equal(s, s2)
        w.mul_(2.0)                                               # what an optimizer step does: in place, new version
        q3, s3 = recipe.weight_codes.get(w)
        assert recipe.weight_codes.misses == 5
        assert torch.equal(q3, q) and not torch.equal(s3, s)      # same codes (exact rescale by 2), doubled scales
        y2 = model(x)
        assert not torch.equal(y2, y1)
    del model, w
    import gc
    gc.collect()
    assert len(recipe.weight_codes._entries) == 0


@pytest.mark.parametrize("B,T,C,H,bias,res,out", [(1, 32, 64, 2, False, torch.float32, torch.float32), (2, 96, 192, 3, True, torch.bfloat16, torch.float32),
                                                  (3, 160, 128, 4, False, torch.float32, torch.bfloat16),
                                                  # 64 K blocks: the weight gradients are sums of four parts, together as alone
                                                  (2, 1024, 512, 8, True, torch.bfloat16, torch.bfloat16)])
def test_block_as_one_node_equals_the_functions(B, T, C, H, bias, res, out):
    """QBlock's single node runs the kernels of AttentionIn, the attention and AttentionOutMLP in their order with their noise
    counters: outputs and every gradient are the same bits."""
    import BlockQuantizeCUDA as BQC
    import recipe
    from Nonlinear import int8_quantize
    jf = BQC.jetfire

    class Attention(torch.autograd.Function):
        @staticmethod
        def forward(ctx, q, k, v):
            q, k, v = (t.reshape(B * T, C) for t in (q, k, v))
            y, lse = jf.attention_fwd(q, k, v, B, H)
            ctx.save_for_backward(q, k, v, y, lse)
            return y.view(B, T, C)

        @staticmethod
        def backward(ctx, g):
            return jf.attention_bwd(*ctx.saved_tensors, g.reshape(B * T, C).contiguous(), B, H).view(B, T, 3 * C).split(C, dim=-1)

    torch.manual_seed(5)
    blk = recipe.QBlock(C, H, out, bias).cuda()
    with torch.no_grad():
        for p in blk.parameters():
            if p.dim() == 1:
                p.add_(0.1 * torch.randn_like(p))
    x = torch.randn(B, T, C, device="cuda").to(res)
    g = torch.randn(B, T, C, device="cuda").to(out)

    def run(one):
        torch.manual_seed(77)
        xi = x.clone().requires_grad_(True)
        for p in blk.parameters():
            p.grad = None
        h, qx, sx = recipe.StreamBegin.apply(xi)
        mean, rstd = jf.rowstats_fp(h.detach())
        assert torch.allclose(mean, h.detach().float().mean(-1), atol=1e-6)
        assert torch.allclose(rstd, torch.rsqrt(h.detach().float().var(-1, unbiased=False)), rtol=1e-5)
        if one:
            assert blk._one_node(h, sx)
            fp, q, s, m, r = blk(h, qx, sx, mean, rstd)
        else:
            a, qq, k, v = recipe.AttentionIn.apply(h, qx, sx, blk.w_qkv, blk.ln_1, mean, rstd, blk.b_qkv)
            fp, q, s, m, r = recipe.AttentionOutMLP.apply(a, Attention.apply(qq, k, v), blk.w_attn_proj, blk.w_fc, blk.w_mlp_proj, blk.ln_2, out,
                                                          blk.b_attn_proj, blk.b_fc, blk.b_mlp_proj)
        recipe.StreamEnd.apply(fp, q, s).backward(g)
        return [fp.detach(), q.view(torch.int8), s, m, r, xi.grad] + [p.grad for p in blk.parameters()]
    for i, (a, b) in enumerate(zip(run(True), run(False))):
        assert a.dtype == b.dtype and torch.equal(a, b), i
    # several weights quantised in one launch: the codes of one by one
    for (q, s), w in zip(jf.quantize_many([blk.w_qkv.detach(), blk.w_fc.detach()]), (blk.w_qkv, blk.w_fc)):
        q2, s2 = int8_quantize(w.detach(), 32)
        assert torch.equal(q, q2) and torch.equal(s, s2)


def block_arguments(B=1, T=64, C=128, H=4, bias=True):
    """What QBlock.forward hands to the extension: [x, qx, sx, mean, rstd, params, codes, biases, (bias, max) pairs, heads, type]."""
    import BlockQuantizeCUDA as BQC
    import recipe
    torch.manual_seed(6)
    blk = recipe.QBlock(C, H, torch.float32, bias).cuda()
    x = torch.randn(B, T, C, device="cuda")
    x, qx, sx = recipe.StreamBegin.apply(x)
    mean, rstd = BQC.jetfire.rowstats_fp(x)
    ws, bs = [blk.w_qkv, blk.w_attn_proj, blk.w_fc, blk.w_mlp_proj], [blk.b_qkv, blk.b_attn_proj, blk.b_fc, blk.b_mlp_proj]
    codes = [tuple(p) for p in recipe.weight_codes.get_many(ws)]
    return [x, qx, sx, mean, rstd, [blk.ln_1, blk.ln_2] + ws, codes, bs, [recipe.weight_codes.get_bias(b) for b in bs], H, torch.float32]


def test_block_refuses_tensors_of_another_device_or_shape():
    """Every tensor of the block's single node is looked at before anything is launched: on the GPU of x, of its own width."""
    import BlockQuantizeCUDA as BQC
    qblock = BQC.jetfire.qblock
    assert len(qblock(*block_arguments())) == 5
    X, QX, SX, MEAN, RSTD, PARAMS, CODES, BPARAMS, BPAIRS = range(9)

    def host(t):
        return t.detach().cpu()

    def other_shape(t):                                            # the same number of elements in rows of another width
        return t.detach().reshape(*t.shape[:-2], t.shape[-2] // 2, t.shape[-1] * 2)

    def swap(i, f, *path):
        a = block_arguments()
        if not path:
            a[i] = f(a[i])
        else:
            inner = list(a[i])
            if len(path) == 1:
                inner[path[0]] = f(inner[path[0]])
            else:
                pair = list(inner[path[0]])
                pair[path[1]] = f(pair[path[1]])
                inner[path[0]] = tuple(pair)
            a[i] = inner
        return a

    cases = [(i, host) for i in (X, QX, SX, MEAN, RSTD)] + [(PARAMS, host, 0), (PARAMS, host, 1)]
    cases += [(CODES, host, k, part) for k in range(4) for part in range(2)] + [(BPAIRS, host, k, part) for k in range(4) for part in range(2)]
    cases += [(i, other_shape) for i in (QX, SX)] + [(CODES, other_shape, k, part) for k in range(4) for part in range(2)]
    cases += [(MEAN, lambda t: t[..., :-32].contiguous()), (PARAMS, lambda t: t.detach()[:-32], 0), (BPAIRS, lambda t: t[:-32], 2, 0)]
    for case in cases:
        args = swap(*case)
        with pytest.raises(RuntimeError, match="expected|must be"):
            qblock(*args)
            raise AssertionError(f"accepted: {case}")


def test_block_calls_its_hooks():
    """Forward, full backward and full backward pre-hooks of a block see its five outputs and their gradients."""
    import recipe
    torch.manual_seed(8)
    model = recipe.QStack(2, 128, 4).cuda()
    seen = []
    for i, blk in enumerate(model.blocks):
        blk.register_forward_hook(lambda m, a, out, i=i: seen.append(("forward", i, type(out), len(out))))
        blk.register_full_backward_pre_hook(lambda m, go, i=i: seen.append(("pre", i, type(go), len(go))))
        blk.register_full_backward_hook(lambda m, gi, go, i=i: seen.append(("backward", i, type(go), len(go))))
    x = torch.randn(2, 64, 128, device="cuda", requires_grad=True)
    w = torch.randn(2, 64, 128, device="cuda")
    torch.manual_seed(9)
    (model(x) * w).sum().backward()
    assert seen == [("forward", 0, tuple, 5), ("forward", 1, tuple, 5), ("pre", 1, tuple, 5), ("backward", 1, tuple, 5), ("pre", 0, tuple, 5),
                    ("backward", 0, tuple, 5)]
    got = [x.grad] + [p.grad for p in model.parameters()]
    plain = recipe.QStack(2, 128, 4).cuda()                        # the hooks change nothing
    plain.load_state_dict(model.state_dict())
    x2 = x.detach().clone().requires_grad_(True)
    torch.manual_seed(9)
    (plain(x2) * w).sum().backward()
    for a, b in zip(got, [x2.grad] + [p.grad for p in plain.parameters()]):
        assert torch.equal(a, b)


def test_block_without_a_backward_keeps_nothing_for_one():
    """Under no_grad (and where nothing requires a gradient) a block holds what its next operators need, not what a backward
    would: 14 bytes per element of [tokens, C] and its results; same bits as with a gradient.  A gradient of one parameter
    alone, or of the input alone, is still computed."""
    import recipe
    torch.manual_seed(12)
    B, T, C, H = 16, 512, 256, 4
    blk = recipe.QBlock(C, H, torch.float32, True).cuda()
    args = block_arguments(B, T, C, H)[:5]
    want = [t.detach().clone() for t in blk(*args)]                # (also quantises the weights)

    def peak(f):
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        out = f()
        torch.cuda.synchronize()
        return torch.cuda.max_memory_allocated() - before, out

    def check(held, out):
        for a, b in zip(out, want):
            assert torch.equal(a.view(torch.int8), b.view(torch.int8)) and not a.requires_grad
        # 14 inside, a float32 sum and codes as results, 0.5 for scales, statistics and row sums; the allocator counts up to 1 MiB
        # more for each of the three large tensors (it does not split off less)
        assert held < (14 + 5 + 0.5) * B * T * C + (3 << 20), held / (B * T * C)

    with torch.no_grad():
        check(*peak(lambda: blk(*args)))
    with torch.inference_mode():
        check(*peak(lambda: blk(*args)))
    for p in blk.parameters():
        p.requires_grad_(False)
    check(*peak(lambda: blk(*args)))
    blk.w_fc.requires_grad_(True)
    blk(*args)[0].sum()                                            # a graph that is never used
    fp, q, s, _, _ = blk(*args)
    recipe.StreamEnd.apply(fp, q, s).backward(torch.ones_like(fp))
    assert blk.w_fc.grad.isfinite().all() and blk.w_fc.grad.abs().sum() > 0 and blk.w_qkv.grad is None


def test_block_takes_strided_operands_and_statistics_of_other_types():
    """Codes, scales, residual, statistics and LayerNorm weights that are not contiguous, or statistics in float64: the same bits."""
    import recipe
    torch.manual_seed(13)
    B, T, C, H = 2, 64, 128, 4
    blk = recipe.QBlock(C, H).cuda()
    args = block_arguments(B, T, C, H)[:5]
    w = torch.randn(B, T, C, device="cuda")

    def strided(t):                                                # the same values, every other element of the storage
        if t.element_size() == 1:
            return torch.stack([t.view(torch.int8)] * 2, -1)[..., 0].view(t.dtype)
        return torch.stack([t, t], -1)[..., 0]

    def run(blk, args):
        torch.manual_seed(14)
        for p in blk.parameters():
            p.grad = None
        x = args[0].detach().clone(memory_format=torch.preserve_format).requires_grad_(True)
        fp, q, s, m, r = blk(x, *args[1:])
        recipe.StreamEnd.apply(fp, q, s).backward(w)
        return [fp, q.view(torch.int8), s, m, r, x.grad] + [p.grad for p in blk.parameters()]

    want = run(blk, args)
    odd = recipe.QBlock(C, H).cuda()
    odd.load_state_dict(blk.state_dict())
    for name in ("ln_1", "ln_2"):
        setattr(odd, name, torch.nn.Parameter(strided(getattr(odd, name).detach())))
        assert not getattr(odd, name).is_contiguous()
    views = [strided(t.detach()) for t in args]
    assert not any(t.is_contiguous() for t in views)
    for other in (views, [*views[:3], views[3].double(), views[4].double()]):
        for i, (a, b) in enumerate(zip(want, run(odd, other))):
            assert torch.equal(a, b), i


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_autocast_reaches_the_attention(dtype, monkeypatch):
    """The recipe's attention runs in binary16; under an autocast to another type it is torch's attention that is called, within
    the autocast (here a stand-in that records it)."""
    import recipe
    torch.manual_seed(15)
    calls = []

    def attention(q, k, v, is_causal):
        calls.append((torch.is_autocast_enabled("cuda"), torch.get_autocast_dtype("cuda"), is_causal))
        return v.to(torch.get_autocast_dtype("cuda"))
    monkeypatch.setattr(recipe.F, "scaled_dot_product_attention", attention)
    blk = recipe.QBlock(128, 4).cuda()
    args = block_arguments()[:5]
    with torch.no_grad():
        plain = blk(*args)
        assert not calls
        with torch.autocast("cuda", dtype=dtype):
            cast = blk(*args)
    assert calls == ([] if dtype == torch.float16 else [(True, dtype, True)])
    assert cast[0].isfinite().all() and torch.equal(cast[0], plain[0]) == (dtype == torch.float16)


def test_block_with_some_of_its_biases():
    """A block some of whose biases were taken out applies the ones that are left."""
    import recipe
    torch.manual_seed(16)
    blk = recipe.QBlock(128, 4, torch.float32, True).cuda()
    args = block_arguments()[:5]
    with torch.no_grad():
        for b in (blk.b_qkv, blk.b_attn_proj, blk.b_fc, blk.b_mlp_proj):
            b.normal_()
        for keep in (("b_qkv",), ("b_attn_proj", "b_mlp_proj"), ("b_qkv", "b_fc", "b_mlp_proj")):
            some, zeros = recipe.QBlock(128, 4, torch.float32, True).cuda(), recipe.QBlock(128, 4, torch.float32, True).cuda()
            for other in (some, zeros):
                other.load_state_dict(blk.state_dict())
            for name in ("b_qkv", "b_attn_proj", "b_fc", "b_mlp_proj"):
                if name not in keep:
                    setattr(some, name, None)
                    getattr(zeros, name).zero_()
            got, want = some(*args), zeros(*args)
            none = recipe.QBlock(128, 4).cuda()
            none.load_state_dict({n: p for n, p in blk.state_dict().items() if not n.startswith("b_")})
            assert cos(got[0], want[0]) > 0.9999 and cos(none(*args)[0], want[0]) < 0.999
