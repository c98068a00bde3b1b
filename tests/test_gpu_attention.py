"""The recipe's causal attention kernels against attention evaluated in float32 on the CPU, at the edges of their tiles: one
row block, ragged last tiles, workgroups with waves that have no rows, head counts that do not divide by the 8 XCDs, operands
that are column ranges of one tensor."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def reference(qkv, g, B, H, T, D):
    x = qkv.float().cpu().view(B, T, 3, H, D).permute(2, 0, 3, 1, 4).contiguous().requires_grad_(True)
    s = (x[0] @ x[1].transpose(-1, -2).contiguous()) * D ** -0.5
    s = s.masked_fill(~torch.ones(T, T, dtype=torch.bool).tril(), float("-inf"))
    o = (torch.softmax(s, -1) @ x[2]).transpose(1, 2).reshape(B * T, H * D)
    o.backward(g.float().cpu())
    return o.detach(), x.grad.permute(1, 3, 0, 2, 4).reshape(B * T, 3 * H * D)


def rel(a, b):
    return float((a.float().cpu() - b).norm() / b.norm())


@pytest.mark.parametrize("B,H,T,D", [(1, 1, 32, 64), (2, 3, 64, 64), (1, 5, 96, 32), (2, 4, 160, 64), (37, 7, 160, 64), (70, 8, 96, 32),
                                     (20, 9, 288, 64), (1, 2, 1056, 64)])
@pytest.mark.parametrize("scale", [1.0, 6.0])
def test_causal_attention(B, H, T, D, scale):
    import BlockQuantizeCUDA as BQC
    jf, C = BQC.jetfire, H * D
    gen = torch.Generator().manual_seed(B * 1000 + T)
    qkv = (torch.randn(B * T, 3 * C, generator=gen) * scale).half().cuda()     # (scale 6: peaked rows, the running maximum moves)
    g = (torch.randn(B * T, C, generator=gen) * 1e-2).half().cuda()
    q, k, v = qkv.split(C, dim=1)
    print(f"case B={B} H={H} T={T} D={D} scale={scale}", flush=True)
    out, lse = jf.attention_fwd(q, k, v, B, H)
    grads = jf.attention_bwd(q, k, v, out, lse, g, B, H)
    want, want_g = reference(qkv, g, B, H, T, D)
    assert rel(out, want) < 1e-3
    for i in range(3):
        assert rel(grads[:, i * C:(i + 1) * C], want_g[:, i * C:(i + 1) * C]) < 2e-3, i
    out2, lse2 = jf.attention_fwd(q.contiguous(), k.contiguous(), v.contiguous(), B, H)
    assert torch.equal(out, out2) and torch.equal(lse, lse2)                   # operands of their own: same bits
    assert torch.equal(grads, jf.attention_bwd(q, k, v, out, lse, g, B, H))    # and on every run
    with pytest.raises(RuntimeError):
        jf.attention_fwd(q, k, v.float(), B, H)
    with pytest.raises(RuntimeError):
        jf.attention_fwd(q[: 16 * B], k[: 16 * B], v[: 16 * B], B, H)          # rows that are not whole blocks
    # the same with the block quantisation inside: what quantising the stored tensors gives
    out3, lse3, qo, so = jf.attention_fwd_q(q, k, v, B, H)
    assert torch.equal(out, out3) and torch.equal(lse, lse3)
    wq, ws, _ = jf.quantize(out, jf.ROUND_NEAREST)
    assert torch.equal(qo, wq) and torch.equal(so, ws)
    qg, sg = jf.attention_bwd_q(q, k, v, out, lse, g, B, H, 3, 40)
    wq, ws, _ = jf.quantize(grads, jf.ROUND_STOCHASTIC, torch.float16, False, 0.0, 3, 40)
    assert torch.equal(qg, wq) and torch.equal(sg, ws)


def half(x):
    return x.to(torch.float16).to(x.dtype)


def attention64(q, k, v, g, rounded):
    """One head in float64: (out, dq, dk, dv).  rounded: with the roundings to binary16 that the kernels state, and no others: the
    probabilities and score gradients that enter a second product, and the results (the forward's is what the backward reads).  The
    forward's probabilities are relative to the maximum over a row's first 32 keys unless the row has one 2^8 times larger."""
    r = half if rounded else (lambda x: x)
    T, scale = q.shape[0], q.shape[1] ** -0.5
    mask = ~torch.ones(T, T, dtype=torch.bool).tril()
    s = ((q @ k.t()) * scale).masked_fill(mask, float("-inf"))
    first, top = s[:, :32].amax(1, keepdim=True), s.amax(1, keepdim=True)
    e = torch.exp(s - torch.where(top - first > 8 * 0.6931, top, first))
    out = r((r(e) @ v) / e.sum(1, keepdim=True))
    p = torch.softmax(s, 1)
    ds = r(p * (g @ v.t() - (out * g).sum(1, keepdim=True)))
    return out, r(ds @ k * scale), r(ds.t() @ q * scale), r(r(p).t() @ g)


@pytest.mark.parametrize("B,H,T,D,scale,kind", [(1, 3, 1024, 64, 1.0, "plain"), (1, 3, 1024, 64, 6.0, "plain"), (1, 2, 512, 64, 20.0, "plain"),
                                                (1, 3, 1024, 32, 1.0, "plain"), (1, 3, 512, 32, 0.1, "plain"), (1, 3, 1024, 64, 1.0, "rising"),
                                                (1, 3, 1024, 32, 3.0, "rising"), (2, 4, 416, 64, 1.0, "channel"), (37, 7, 160, 64, 1.0, "plain"),
                                                (37, 7, 160, 64, 3.0, "channel"), (70, 8, 96, 32, 3.0, "plain")])
def test_attention_rounds_only_where_it_says(B, H, T, D, scale, kind):
    """The error against float64 is that of float64 with the stated roundings.  Bound: a result's own rounding is in both; what else can
    differ is whether a row's largest probability is exactly 1 (the kernel's maximum may be raised on the way, then it is not), which is
    one more rounding of the same size, the square root of 2 in norm.  (Seen: 0.94 to 1.02, and 1.11 where keys rise.)  Binary32 leaves a
    probability a relative error of 2^-23 times its exponent.  rising: keys that grow along the sequence, so that the running maximum is
    raised again and again; channel: one channel in fifty twenty times larger, as activations have."""
    import BlockQuantizeCUDA as BQC
    jf, C = BQC.jetfire, H * D
    gen = torch.Generator().manual_seed(B * 1000 + T + D)
    x = torch.randn(B * T, 3 * C, generator=gen) * scale
    if kind == "rising":
        x[:, C: 2 * C] *= torch.linspace(0.2, 3.0, T).repeat(B).unsqueeze(1)
    elif kind == "channel":
        x[:, 7::50] *= 20
    qkv, g = x.half(), (torch.randn(B * T, C, generator=gen) * 1e-2).half()
    print(f"case B={B} H={H} T={T} D={D} scale={scale} {kind}", flush=True)
    q, k, v = qkv.cuda().split(C, dim=1)
    out, lse = jf.attention_fwd(q, k, v, B, H)
    grads = jf.attention_bwd(q, k, v, out, lse, g.cuda(), B, H)
    got = torch.cat([out, grads], 1).cpu().double().view(B, T, 4, H, D)
    err, model, norm, exponent = torch.zeros(4, dtype=torch.float64), torch.zeros(4, dtype=torch.float64), torch.zeros(4, dtype=torch.float64), 0.0
    for b in range(B):
        for h in range(H):
            a = [t.double().contiguous() for t in qkv.view(B, T, 3, H, D)[b, :, :, h].unbind(1)] + [g.view(B, T, H, D)[b, :, h].double()]
            want, rounded = attention64(*a, False), attention64(*a, True)
            exponent = max(exponent, float((a[0] @ a[1].t()).abs().max()) * D ** -0.5 * 1.4427)
            for i in range(4):
                err[i] += (got[b, :, i, h] - want[i]).square().sum()
                model[i] += (rounded[i] - want[i]).square().sum()
                norm[i] += want[i].square().sum()
    err, model = (err / norm).sqrt(), (model / norm).sqrt()
    print("  out dq dk dv", " ".join("%.2e" % e for e in err.tolist()), "| rounded", " ".join("%.2e" % e for e in model.tolist()),
          "ratio", " ".join("%.3f" % e for e in (err / model).tolist()), "exponent %.0f" % exponent, flush=True)
    assert (err <= 2.0 ** 0.5 * model + 2.0 ** -23 * exponent).all()


def causal_rows(qkv, B, H, T, D):
    """Attention in float32 on the CPU, every query over its own keys only: what lies behind a query cannot reach it."""
    x = qkv.float().cpu().view(B, T, 3, H, D).permute(2, 0, 3, 1, 4)
    rows = []
    for i in range(T):
        s = (x[1][:, :, : i + 1] * x[0][:, :, i: i + 1]).sum(-1) * D ** -0.5
        p = torch.softmax(s, -1)
        rows.append(torch.where(p == 0, torch.zeros(()), p).unsqueeze(-1).mul(x[2][:, :, : i + 1]).sum(2))
    return torch.stack(rows, 2).transpose(1, 2).reshape(B * T, H * D)


INF, NAN = float("inf"), float("nan")


@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("what,value", [("q", NAN), ("k", NAN), ("v", NAN), ("q", INF), ("k", INF), ("v", INF), ("v", -INF)])
def test_a_value_that_is_not_finite_reaches_the_result(D, what, value):
    """An infinity or NaN in q, k or v: the result is not finite wherever it is not in float32, and untouched in the row blocks
    before it.  The quantised results are those of the stored ones, and a NaN gradient reaches every gradient it belongs to."""
    import BlockQuantizeCUDA as BQC
    jf, B, H, T, at = BQC.jetfire, 1, 2, 160, 70
    C = H * D
    gen = torch.Generator().manual_seed(D)
    qkv = torch.randn(T, 3 * C, generator=gen).half()
    g = (torch.randn(T, C, generator=gen) * 1e-2).half().cuda()
    qkv[:, 5] = qkv[:, C + 5] = 1.0                                # (head 0: one column of q and k with a known sign)
    qkv[at, {"q": 0, "k": C, "v": 2 * C}[what] + 5] = value
    print(f"case {what}={value} D={D}", flush=True)
    q, k, v = qkv.cuda().split(C, dim=1)
    out, lse, qo, so = jf.attention_fwd_q(q, k, v, B, H)
    want = causal_rows(qkv, B, H, T, D)
    bad = ~want.isfinite()
    assert bad.any() and not out.cpu()[bad].isfinite().any()
    assert out.cpu()[:64].isfinite().all() and rel(out[:64], want[:64]) < 1e-3                        # row blocks before it
    assert out.cpu()[:, D:].isfinite().all() and rel(out[:, D:], want[:, D:]) < 1e-3                  # the other head
    wq, ws, _ = jf.quantize(out, jf.ROUND_NEAREST)
    assert torch.equal(qo, wq) and torch.equal(so.view(torch.int16), ws.view(torch.int16))
    grads = jf.attention_bwd(q, k, v, out, lse, g, B, H)
    qg, sg = jf.attention_bwd_q(q, k, v, out, lse, g, B, H, 3, 40)
    wq, ws, _ = jf.quantize(grads, jf.ROUND_STOCHASTIC, torch.float16, False, 0.0, 3, 40)
    assert torch.equal(qg, wq) and torch.equal(sg.view(torch.int16), ws.view(torch.int16))
    if what == "q":                                                # a query's row of scores: its own dq, dk and dv of its keys
        rows = grads.cpu()
        assert rows[at, :D].isnan().all() and rows[: at + 1, C: C + D].isnan().all() and rows[: at + 1, 2 * C: 2 * C + D].isnan().all()
        assert rows[96:, :D].isfinite().all() and rows[:, D: C].isfinite().all()


@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("keys", [range(0, 32), range(0, 64), range(0, 96), [3, 40, 159]])
def test_scores_of_minus_infinity_count_for_nothing(D, keys):
    """Keys whose scores are -inf (k infinite against a positive q): the other keys decide; a query with no other key has no result."""
    import BlockQuantizeCUDA as BQC
    jf, B, H, T = BQC.jetfire, 1, 1, 160
    gen = torch.Generator().manual_seed(D)
    qkv = torch.randn(T, 3 * D, generator=gen).half()
    qkv[:, 5] = 1.0
    qkv[list(keys), D + 5] = -INF
    print(f"case keys={keys} D={D}", flush=True)
    out, _ = jf.attention_fwd(*qkv.cuda().split(D, dim=1), B, H)
    want = causal_rows(qkv, B, H, T, D)
    finite = want.isfinite().all(1)
    assert finite.sum() >= 64 and not out.cpu()[~finite].isfinite().any()
    assert rel(out.cpu()[finite], want[finite]) < 1e-3


# both gradients in one launch (up to one and a half workgroups per CU, sequences of up to 4096 rows) against the two launches that many copies
# of the same sequences take: one workgroup, waves without rows, ragged last tiles, the most workgroups, the longest sequence
@pytest.mark.parametrize("B,H,T,D,copies", [(1, 1, 32, 64, 385), (1, 3, 96, 32, 130), (3, 4, 416, 64, 9), (3, 16, 1024, 64, 2), (2, 1, 4096, 32, 7)])
def test_both_gradients_in_one_launch(B, H, T, D, copies):
    import BlockQuantizeCUDA as BQC
    jf, C = BQC.jetfire, H * D
    print(f"case B={B} H={H} T={T} D={D}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(T)
    qkv = torch.randn(B * T, 3 * C, device="cuda", generator=gen).half()
    g = (torch.randn(B * T, C, device="cuda", generator=gen) * 1e-2).half()
    out, lse = jf.attention_fwd(*qkv.split(C, dim=1), B, H)
    grads = jf.attention_bwd(*qkv.split(C, dim=1), out, lse, g, B, H)
    qg, sg = jf.attention_bwd_q(*qkv.split(C, dim=1), out, lse, g, B, H, 3, 40)
    wq, ws, _ = jf.quantize(grads, jf.ROUND_STOCHASTIC, torch.float16, False, 0.0, 3, 40)
    assert torch.equal(qg, wq) and torch.equal(sg, ws)
    many = jf.attention_bwd(*qkv.repeat(copies, 1).split(C, dim=1), out.repeat(copies, 1), lse.repeat(copies, 1).reshape(-1, T).contiguous(),
                            g.repeat(copies, 1), copies * B, H)
    for part in many.split(B * T):
        assert torch.equal(part, grads)


def test_one_row_block_more_than_one_launch_takes():
    """4128 rows take the two launches.  With no gradient behind row 4095 they return what the one launch returns for the first 4096 rows."""
    import BlockQuantizeCUDA as BQC
    jf, T, D = BQC.jetfire, 4128, 64
    gen = torch.Generator(device="cuda").manual_seed(T)
    qkv = torch.randn(T, 3 * D, device="cuda", generator=gen).half()
    g = (torch.randn(T, D, device="cuda", generator=gen) * 1e-2).half()
    out, lse = jf.attention_fwd(*qkv.split(D, dim=1), 1, 1)
    grads = jf.attention_bwd(*qkv.split(D, dim=1), out, lse, g, 1, 1)
    want, want_g = reference(qkv, g, 1, 1, T, D)
    assert rel(out, want) < 1e-3
    for i in range(3):
        assert rel(grads[:, i * D:(i + 1) * D], want_g[:, i * D:(i + 1) * D]) < 2e-3, i
    g[4096:] = 0
    long = jf.attention_bwd(*qkv.split(D, dim=1), out, lse, g, 1, 1)
    short = jf.attention_bwd(*qkv[:4096].split(D, dim=1), out[:4096].contiguous(), lse.view(1, T)[:, :4096].contiguous(), g[:4096].contiguous(), 1, 1)
    assert torch.equal(long[:4096], short) and not long[4096:, :D].any()


# gradients that lie where operands were (the kernels of one launch read those to the end) or between the columns of the operands' matrix
@pytest.mark.parametrize("B,H,T,D", [(1, 1, 32, 64), (3, 4, 416, 64), (2, 16, 1024, 32)])
def test_gradients_in_the_place_of_operands(jf, B, H, T, D):
    import BlockQuantizeCUDA as BQC
    C, p = H * D, jf._ptr
    print(f"case B={B} H={H} T={T} D={D}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(T)
    wide = torch.randn(B * T, 6 * C, device="cuda", generator=gen).half()
    g = (torch.randn(B * T, C, device="cuda", generator=gen) * 1e-2).half()
    q, k, v = (wide[:, i * C:(i + 1) * C].contiguous() for i in range(3))
    out, lse = BQC.jetfire.attention_fwd(q, k, v, B, H)
    want = BQC.jetfire.attention_bwd(q, k, v, out, lse, g, B, H)
    delta = torch.empty(B * H, T, device="cuda")

    def bwd(q, k, v, ld, out, gq, gk, gv, ldg):
        jf.check(jf.lib().jf_attention_bwd(p(q), p(k), p(v), ld, p(out), p(g), p(lse), B, H, T, D, D ** -0.5, p(gq), p(gk), p(gv), ldg, p(delta), jf._stream()))
        return torch.cat((gq, gk, gv), dim=1)

    part = [wide[:, i * C:(i + 1) * C] for i in range(6)]
    assert torch.equal(bwd(*part[:3], 6 * C, out, *part[3:], 6 * C), want)
    o, spare = out.clone(), torch.empty_like(out)
    assert torch.equal(bwd(q, k, v, C, o, spare, o, torch.empty_like(v), C), want)
    o, kk, vv = out.clone(), k.clone(), v.clone()
    assert torch.equal(bwd(q, kk, vv, C, o, o, vv, kk, C), want)
