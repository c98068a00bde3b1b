"""GPU parity of the per-block INT8 GEMMs (through the C ABI) against the CPU oracle.

Bars: INT32 results, per-K-block INT32 accumulators, INT8 codes and scales: bit-exact.  The fp32
accumulation is compared bit-exact too (same fmaf chain); fp16 output = RNE of it.
Shapes: the reference's own test lists (JetfireGEMMKernel/tests/*.py) plus shapes that are not
multiples of the 128x128 tile (where the reference drops tiles) and a K with an odd number of blocks.
"""
import ctypes
import os

import numpy as np
import pytest
import torch

from helpers import QB, rand_codes, rand_scales

pytestmark = pytest.mark.gpu

GOLD = os.path.join(os.path.dirname(__file__), "golden")
SHAPES = [(128, 256, 32), (512, 512, 64), (32, 32, 32), (96, 160, 224), (160, 96, 96), (256, 384, 544)]


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def same(got, want, what):
    got = got.cpu().numpy() if isinstance(got, torch.Tensor) else got
    if got.dtype == np.float16:
        g, w = got.view(np.uint16), want.view(np.uint16)
    elif got.dtype == np.float32:
        g, w = got.view(np.uint32), want.view(np.uint32)
    else:
        g, w = got, want
    bad = np.argwhere(g != w)
    assert bad.shape[0] == 0, f"{what}: {bad.shape[0]} of {g.size} differ; first at {bad[0].tolist()}: " \
                              f"got {got[tuple(bad[0])]}, want {want[tuple(bad[0])]}"


def make_problem(seed, M, N, K, f16=True):
    rng = np.random.default_rng(seed)
    A = rand_codes(rng, (M, K))
    Bkn = rand_codes(rng, (K, N))
    sa = rand_scales(rng, (K // QB, M // QB), f16=f16)
    sb = rand_scales(rng, (K // QB, N // QB), f16=f16)
    return A, Bkn, sa, sb


def b_of(Bkn, layout):
    return Bkn if layout == 1 else np.ascontiguousarray(Bkn.T)


def test_reference_fixture(jf, oracle):
    """A/B/CPU dump of the reference's igemm_BasicInt8Gemm_128_128_32 harness."""
    A = np.loadtxt(os.path.join(GOLD, "basic_int8_gemm_128_128_32_A.txt"), dtype=np.int64).reshape(128, 32).astype(np.int8)
    B = np.loadtxt(os.path.join(GOLD, "basic_int8_gemm_128_128_32_B.txt"), dtype=np.int64).reshape(32, 128).astype(np.int8)
    Cw = np.loadtxt(os.path.join(GOLD, "basic_int8_gemm_128_128_32_C.txt"), dtype=np.int64).reshape(128, 128).astype(np.int32)
    same(jf.igemm_s32(dev(A), dev(B), jf.B_KN), Cw, "fixture KN")
    same(jf.igemm_s32(dev(A), dev(np.ascontiguousarray(B.T)), jf.B_NK), Cw, "fixture NK")


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_s32_and_block_accumulators(jf, oracle, M, N, K, layout):
    print(f"case s32 M={M} N={N} K={K} layout={layout}", flush=True)
    A, Bkn, _, _ = make_problem(M * 7 + N * 3 + K, M, N, K)
    B = b_of(Bkn, layout)
    same(jf.igemm_s32(dev(A), dev(B), layout), oracle.igemm_s32(A, B, layout), "s32")
    same(jf.igemm_block_acc(dev(A), dev(B), layout), oracle.igemm_block_acc(A, B, layout), "block acc")


def test_s32_extreme_codes(jf):
    A = np.full((64, 96), -127, np.int8)
    B = np.full((96, 64), 127, np.int8)
    got = jf.igemm_s32(dev(A), dev(B), jf.B_KN).cpu().numpy()
    assert np.all(got == -96 * 127 * 127)


@pytest.mark.parametrize("f16", [True, False])
@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_block_fp(jf, oracle, M, N, K, layout, f16):
    print(f"case fp M={M} N={N} K={K} layout={layout} f16={f16}", flush=True)
    A, Bkn, sa, sb = make_problem(M + N + K + layout, M, N, K, f16)
    B = b_of(Bkn, layout)
    st = np.float16 if f16 else np.float32
    want32 = oracle.igemm_block_f32(A, B, sa, sb, layout)
    got32 = jf.igemm_block_fp(dev(A), dev(B), dev(sa.astype(st)), dev(sb.astype(st)), layout, torch.float32)
    same(got32, want32, "fp32 accumulators")
    got16 = jf.igemm_block_fp(dev(A), dev(B), dev(sa.astype(st)), dev(sb.astype(st)), layout, torch.float16)
    with np.errstate(over="ignore"):
        same(got16, want32.astype(np.float16), "fp16 output")
    gotbf = jf.igemm_block_fp(dev(A), dev(B), dev(sa.astype(st)), dev(sb.astype(st)), layout, torch.bfloat16)
    wantbf = torch.from_numpy(want32).to(torch.bfloat16)
    assert torch.equal(gotbf.cpu(), wantbf)


@pytest.mark.parametrize("f16", [True, False])
@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_block_q_deterministic_and_stochastic(jf, oracle, M, N, K, layout, f16):
    print(f"case q M={M} N={N} K={K} layout={layout} f16={f16}", flush=True)
    A, Bkn, sa, sb = make_problem(M * 3 + N + K + layout, M, N, K, f16)
    B = b_of(Bkn, layout)
    st = np.float16 if f16 else np.float32
    sdt = "f16" if f16 else "f32"
    dA, dB, dsa, dsb = dev(A), dev(B), dev(sa.astype(st)), dev(sb.astype(st))
    q, sc = jf.igemm_block_q(dA, dB, dsa, dsb, layout)
    wq, wsc = oracle.igemm_block_q(A, B, sa, sb, layout, scale_dtype=sdt)
    same(q, wq, "det codes")
    same(sc, wsc, "det scales")
    q2, sc2 = jf.igemm_block_q(dA, dB, dsa, dsb, layout)
    assert torch.equal(q, q2) and torch.equal(sc, sc2), "run-to-run difference"
    for seed, offset in ((0, 0), (0x1234567890ABCDEF, 977)):
        q, sc = jf.igemm_block_q(dA, dB, dsa, dsb, layout, rounding=jf.ROUND_STOCHASTIC, seed=seed, offset=offset)
        wq, wsc = oracle.igemm_block_q(A, B, sa, sb, layout, stochastic=True, seed=seed, offset=offset, scale_dtype=sdt)
        same(q, wq, f"SR codes seed={seed}")
        same(sc, wsc, "SR scales")


@pytest.mark.parametrize("f16", [True, False])
@pytest.mark.parametrize("layout", [0, 1])
def test_row_major_scale_operands(jf, oracle, layout, f16):
    """The scale operands may be the .t() views of the block tensors' own [rows/32, K/32] scale arrays (no transposed
    copy): same bits as with K-major copies, for each operand separately and for both."""
    M, N, K = 160, 352, 544
    A, Bkn, sa, sb = make_problem(99 + layout, M, N, K, f16)
    B = b_of(Bkn, layout)
    st = np.float16 if f16 else np.float32
    dA, dB = dev(A), dev(B)
    ka, kb = dev(sa.astype(st)), dev(sb.astype(st))                                  # [K/32, rows/32] contiguous
    ra, rb = dev(np.ascontiguousarray(sa.astype(st).T)).t(), dev(np.ascontiguousarray(sb.astype(st).T)).t()   # views
    assert not ra.is_contiguous() and not rb.is_contiguous()
    want = oracle.igemm_block_f32(A, B, sa, sb, layout)
    for xa, xb in ((ra, kb), (ka, rb), (ra, rb)):
        same(jf.igemm_block_fp(dA, dB, xa, xb, layout, torch.float32), want, "fp32 accumulators")
        q0, s0 = jf.igemm_block_q(dA, dB, ka, kb, layout, rounding=jf.ROUND_STOCHASTIC, seed=3, offset=5)
        q1, s1 = jf.igemm_block_q(dA, dB, xa, xb, layout, rounding=jf.ROUND_STOCHASTIC, seed=3, offset=5)
        assert torch.equal(q0, q1) and torch.equal(s0, s1)
    with pytest.raises(RuntimeError):
        jf.igemm_block_fp(dA, dB, ka[:, ::2].repeat_interleave(2, 1)[:, : M // QB].t().t()[::1].as_strided((K // QB, M // QB), (M // QB * 2, 2)), kb, layout)


def _largest_noise(oracle, seed):
    """(offset, element) whose rounding noise under `seed` is the largest there is, 1/2 - 2^-17."""
    for offset in range(1 << 17):
        o = oracle.philox4x32([offset, 0, 0, 0], [seed, 0], oracle.NOISE_ROUNDS)
        h = np.stack([o & 0xFFFF, o >> 16], 1).reshape(-1)
        if (h == 0xFFFF).any():
            return offset, int(np.argmax(h == 0xFFFF))
    raise AssertionError("no such counter")


@pytest.mark.parametrize("sign", [1, -1])
@pytest.mark.parametrize("above", [False, True])
def test_largest_noise_on_the_largest_result(jf, oracle, sign, above):
    """127 * amax / amax is 127 or the number after it; with the noise 1/2 - 2^-17 the latter would round to 128, code -128."""
    offset, e = _largest_noise(oracle, 5)
    A, B = np.zeros((QB, QB), np.int8), np.zeros((QB, QB), np.int8)
    A[0, 0], A[1:, 0] = 64, 16
    B[0, :], B[0, e] = 16, sign * 64
    scale = np.linspace(1, 2, 4001, dtype=np.float32)[1:]
    amax = scale * np.float32(4096)
    top = (np.float32(127) * amax) / amax
    sa, sb = np.full((1, 1), scale[top > 127][0] if above else scale[top == 127][0], np.float32), np.ones((1, 1), np.float32)
    got, sc = jf.igemm_block_q(dev(A), dev(B), dev(sa), dev(sb), jf.B_KN, rounding=jf.ROUND_STOCHASTIC, seed=5, offset=offset)
    want, wsc = oracle.igemm_block_q(A, B, sa, sb, 1, stochastic=True, seed=5, offset=offset, scale_dtype="f32")
    same(got, want, "codes")
    same(sc, wsc, "scales")
    assert abs(int(got[0, e])) == 127


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("regime", ["huge_everywhere", "huge_one_block", "huge_last_kblock", "denormal_products"])
def test_extreme_scale_products(jf, oracle, regime, layout):
    """Scale products at the ends of the fp32 range.  sa*sb >= 2^102 is where the kernel's pre-scaled factor
    (sa*sb*2^26) overflows and the wave must fall back to the plain conversion; products in the denormal range
    must keep their (reduced) precision.  Results are finite in every regime, and bit-exact like everywhere else."""
    M, N, K = 160, 288, 160
    A, Bkn, sa, sb = make_problem(1234 + layout, M, N, K, f16=False)
    B = b_of(Bkn, layout)
    sa = (sa / sa.max()).astype(np.float32)
    sb = (sb / sb.max()).astype(np.float32)                      # all in (0, 1]
    if regime == "huge_everywhere":
        sa, sb = sa * np.float32(2.0 ** 53), sb * np.float32(2.0 ** 52)
    elif regime == "huge_one_block":                             # one output block (one wave) takes the fallback
        sa[:, 2] *= np.float32(2.0 ** 53)
        sb[:, 5] *= np.float32(2.0 ** 52)
    elif regime == "huge_last_kblock":
        sa[-1, :] *= np.float32(2.0 ** 53)
        sb[-1, :] *= np.float32(2.0 ** 52)
    else:
        sa, sb = sa * np.float32(2.0 ** -70), sb * np.float32(2.0 ** -70)
    want = oracle.igemm_block_f32(A, B, sa, sb, layout)
    assert np.isfinite(want).all() and np.abs(want).max() > 0
    dA, dB, dsa, dsb = dev(A), dev(B), dev(sa), dev(sb)
    same(jf.igemm_block_fp(dA, dB, dsa, dsb, layout, torch.float32), want, f"{regime}: fp32 accumulators")
    q, sc = jf.igemm_block_q(dA, dB, dsa, dsb, layout)
    wq, wsc = oracle.igemm_block_q(A, B, sa, sb, layout, scale_dtype="f32")
    same(q, wq, f"{regime}: codes")
    same(sc, wsc, f"{regime}: scales")


@pytest.mark.parametrize("f16", [True, False])
@pytest.mark.parametrize("M,N,K", SHAPES + [(160, 288, 1056)])
def test_block_fp_a_given_as_km(jf, oracle, M, N, K, f16):
    """Weight-gradient form with the A operand as it lies in memory ([K, M], e.g. the gradient [tokens, C_out]) and
    B as [K, N]: the same bits as with a materialised transpose."""
    print(f"case fp A_KM M={M} N={N} K={K} f16={f16}", flush=True)
    A, Bkn, sa, sb = make_problem(M + 2 * N + K, M, N, K, f16)
    st = np.float16 if f16 else np.float32
    Akm = np.ascontiguousarray(A.T)
    want32 = oracle.igemm_block_f32(A, Bkn, sa, sb, 1)
    dsa, dsb = dev(sa.astype(st)), dev(sb.astype(st))
    same(jf.igemm_block_fp(dev(Akm), dev(Bkn), dsa, dsb, jf.B_KN, torch.float32, a_layout=jf.A_KM), want32, "fp32 accumulators")
    got16 = jf.igemm_block_fp(dev(Akm), dev(Bkn), dsa, dsb, jf.B_KN, torch.float16, a_layout=jf.A_KM)
    with np.errstate(over="ignore"):
        same(got16, want32.astype(np.float16), "fp16 output")
    with pytest.raises(RuntimeError, match="not implemented"):
        jf.igemm_block_fp(dev(Akm), dev(np.ascontiguousarray(Bkn.T)), dsa, dsb, jf.B_NK, torch.float32, a_layout=jf.A_KM)


@pytest.mark.parametrize("a_km", [False, True])
@pytest.mark.parametrize("M,N,K,req", [(128, 256, 2048, 2), (160, 96, 3104, 4), (96, 160, 2560, 0), (64, 64, 12288, 0),
                                           (128, 128, 512, 3), (32, 32, 992, 2), (256, 384, 544, 0)])
def test_block_fp_split_k(jf, oracle, M, N, K, req, a_km):
    """K cut into ordered partial chains: bit-exact against the oracle's composition with the same plan; request 1
    stays the reference arithmetic; the two differ by fp32 rounding only."""
    print(f"case fp splitk M={M} N={N} K={K} request={req} a_km={a_km}", flush=True)
    A, Bkn, sa, sb = make_problem(M + N + K + req, M, N, K, f16=False)
    parts, per = jf.splitk_plan(M, N, K, req)
    assert parts >= 1 and per % 4 == 0 and (parts - 1) * per < K // QB <= parts * per
    if req == 0:
        assert parts > 1 or K // QB < 32 or 2 * ((M + 127) // 128) * ((N + 127) // 128) > 512
    dA = dev(np.ascontiguousarray(A.T)) if a_km else dev(A)
    kw = dict(a_layout=jf.A_KM if a_km else jf.A_MK)
    dsa, dsb = dev(sa), dev(sb)
    want = oracle.igemm_block_f32_splitk(A, Bkn, sa, sb, 1, parts, per)
    one = oracle.igemm_block_f32(A, Bkn, sa, sb, 1)
    got = jf.igemm_block_fp(dA, dev(Bkn), dsa, dsb, jf.B_KN, torch.float32, splitk=req, **kw)
    same(got, want, f"fp32, {parts} parts of {per} K blocks")
    same(jf.igemm_block_fp(dA, dev(Bkn), dsa, dsb, jf.B_KN, torch.float32, splitk=1, **kw), one, "one chain")
    np.testing.assert_allclose(want, one, rtol=1e-5, atol=1e-5 * np.abs(one).max())
    got16 = jf.igemm_block_fp(dA, dev(Bkn), dsa, dsb, jf.B_KN, torch.float16, splitk=req, **kw)
    with np.errstate(over="ignore"):
        same(got16, want.astype(np.float16), "fp16 output")
    if not a_km:                                                  # B as [N,K] takes the same path
        same(jf.igemm_block_fp(dA, dev(np.ascontiguousarray(Bkn.T)), dsa, dsb, jf.B_NK, torch.float32, splitk=req),
             oracle.igemm_block_f32_splitk(A, np.ascontiguousarray(Bkn.T), sa, sb, 0, parts, per), "B as [N,K]")


def _random_cases(n, seed):
    rng = np.random.default_rng(seed)
    for _ in range(n):
        yield (int(rng.integers(1, 13)) * 32, int(rng.integers(1, 13)) * 32, int(rng.integers(1, 41)) * 32,
               int(rng.integers(0, 2)), bool(rng.integers(0, 2)), int(rng.integers(0, 4)), int(rng.integers(0, 1 << 30)))


@pytest.mark.parametrize("M,N,K,layout,f16,scale_views,seed", list(_random_cases(32, 2024)))
def test_random_shapes(jf, oracle, M, N, K, layout, f16, scale_views, seed):
    """Random small problems (M, N up to 384, K up to 1280, all multiples of 32): every output kind, both B layouts, both
    scale dtypes, K-major copies or row-major views of the scales, the [K,M] form of A where it applies."""
    print(f"case random M={M} N={N} K={K} layout={layout} f16={f16} views={scale_views} seed={seed}", flush=True)
    A, Bkn, sa, sb = make_problem(seed, M, N, K, f16)
    B = b_of(Bkn, layout)
    st = np.float16 if f16 else np.float32
    sdt = "f16" if f16 else "f32"
    dA, dB = dev(A), dev(B)
    dsa = dev(np.ascontiguousarray(sa.astype(st).T)).t() if scale_views & 1 else dev(sa.astype(st))
    dsb = dev(np.ascontiguousarray(sb.astype(st).T)).t() if scale_views & 2 else dev(sb.astype(st))
    same(jf.igemm_s32(dA, dB, layout), oracle.igemm_s32(A, B, layout), "s32")
    acc = oracle.igemm_block_f32(A, B, sa, sb, layout)
    same(jf.igemm_block_fp(dA, dB, dsa, dsb, layout, torch.float32), acc, "fp32")
    q, sc = jf.igemm_block_q(dA, dB, dsa, dsb, layout)
    wq, wsc = oracle.requant(acc, scale_dtype=sdt)
    same(q, wq, "det codes")
    same(sc, wsc, "det scales")
    q, sc = jf.igemm_block_q(dA, dB, dsa, dsb, layout, rounding=jf.ROUND_STOCHASTIC, seed=seed, offset=seed % 1000)
    wq, wsc = oracle.requant(acc, stochastic=True, seed=seed, offset=seed % 1000, scale_dtype=sdt)
    same(q, wq, "SR codes")
    same(sc, wsc, "SR scales")
    if layout == 1:
        same(jf.igemm_block_fp(dev(np.ascontiguousarray(A.T)), dB, dsa, dsb, layout, torch.float32, a_layout=jf.A_KM), acc, "fp32, A as [K,M]")
        parts, per = jf.splitk_plan(M, N, K, 0)
        same(jf.igemm_block_fp(dA, dB, dsa, dsb, layout, torch.float32, splitk=0),
             oracle.igemm_block_f32_splitk(A, B, sa, sb, layout, parts, per), f"fp32, {parts} parts")


@pytest.mark.parametrize("views", [0, 3])
@pytest.mark.parametrize("a_km", [False, True])
def test_block_fp_split_k_binary16_scales(jf, oracle, a_km, views):
    """The K split with binary16 scales (fetched as 32-bit words, half selected by index parity) in both scale layouts."""
    M, N, K, req = 96, 160, 4128, 3
    A, Bkn, sa, sb = make_problem(77, M, N, K, f16=True)
    parts, per = jf.splitk_plan(M, N, K, req)
    assert parts == 3
    dA = dev(np.ascontiguousarray(A.T)) if a_km else dev(A)
    h = np.float16
    dsa = dev(np.ascontiguousarray(sa.astype(h).T)).t() if views & 1 else dev(sa.astype(h))
    dsb = dev(np.ascontiguousarray(sb.astype(h).T)).t() if views & 2 else dev(sb.astype(h))
    want = oracle.igemm_block_f32_splitk(A, Bkn, sa, sb, 1, parts, per)
    got = jf.igemm_block_fp(dA, dev(Bkn), dsa, dsb, jf.B_KN, torch.float32, splitk=req, a_layout=jf.A_KM if a_km else jf.A_MK)
    same(got, want, "fp32")


def test_block_q_bias(jf, oracle):
    """The forward kernel's bias / biasmax inputs (…BiasRowCol.cu:313,341,357)."""
    M, N, K = 128, 256, 96
    A, Bkn, sa, sb = make_problem(5, M, N, K)
    B = b_of(Bkn, 0)
    rng = np.random.default_rng(6)
    acc = oracle.igemm_block_f32(A, B, sa, sb, 0)
    bias = (np.abs(acc).mean() * rng.standard_normal(N)).astype(np.float32)
    biasmax = np.array([np.abs(bias).max()], np.float32)
    q, sc = jf.igemm_block_q(dev(A), dev(B), dev(sa.astype(np.float16)), dev(sb.astype(np.float16)), 0,
                             bias=dev(bias), biasmax=dev(biasmax))
    wq, wsc = oracle.igemm_block_q(A, B, sa, sb, 0, bias=bias, biasmax=float(biasmax[0]), scale_dtype="f16")
    same(q, wq, "bias codes")
    same(sc, wsc, "bias scales")


def test_zero_blocks_and_zero_scales(jf, oracle):
    M, N, K = 64, 64, 64
    A, Bkn, sa, sb = make_problem(9, M, N, K)
    A[:32] = 0
    sb[:, 1] = 0.0
    q, sc = jf.igemm_block_q(dev(A), dev(Bkn), dev(sa.astype(np.float16)), dev(sb.astype(np.float16)), 1)
    wq, wsc = oracle.igemm_block_q(A, Bkn, sa, sb, 1, scale_dtype="f16")
    same(q, wq, "codes")
    same(sc, wsc, "scales")
    assert not q.cpu().numpy()[:32].any() and not sc.cpu().numpy()[0].any()


def test_sr_mean_converges(jf, oracle):
    """Mean of R stochastic runs -> un-rounded product, error ~ R^-1/2
    (JetfireGEMMKernel/tests/test_int8igemmoutputIntQuantizeStochastic.py:70-120)."""
    M, N, K = 128, 128, 64
    A, Bkn, sa, sb = make_problem(11, M, N, K)
    dA, dB, dsa, dsb = dev(A), dev(Bkn), dev(sa.astype(np.float16)), dev(sb.astype(np.float16))
    acc = oracle.igemm_block_f32(A, Bkn, sa, sb, 1)
    amax = np.abs(acc.reshape(M // QB, QB, N // QB, QB)).max(axis=(1, 3))
    t = 127.0 * acc / np.repeat(np.repeat(amax, QB, 0), QB, 1)
    errs = []
    for R in (16, 256):
        m = torch.zeros((M, N), dtype=torch.float64, device="cuda")
        for r in range(R):
            q, _ = jf.igemm_block_q(dA, dB, dsa, dsb, 1, rounding=jf.ROUND_STOCHASTIC, seed=3, offset=r * (M * N // 8))
            m += q
        errs.append(float(np.sqrt(np.mean((m.cpu().numpy() / R - t) ** 2))))
    assert errs[0] < 0.5 / 4 and errs[1] < 0.5 / 16 and 2.5 < errs[0] / errs[1] < 6.5


def test_full_size_small_wgrad_deep_k(jf, oracle):
    """benchmark configuration 2 (GPT-2 small, 12288 tokens): the weight gradient of the qkv layer, K = 12288 deep with few
    output tiles (2304 x 768), both operands read in place from their token-major arrays' natural layouts."""
    T, Cin, Cout = 12288, 768, 2304
    g = torch.Generator().manual_seed(0)
    x = torch.randn(T, Cin, generator=g)
    dy = torch.randn(T, Cout, generator=g) * 1e-3
    qx, sx = jf.quantize(x.cuda(), scale_dtype=torch.float32)
    qg, sg, qgT = jf.quantize(dy.cuda(), rounding=jf.ROUND_STOCHASTIC, scale_dtype=torch.float32, transpose=True, seed=0, offset=0)
    dw = jf.igemm_block_fp(qgT, qx, sg, sx, jf.B_KN, torch.float32)
    torch.cuda.synchronize()
    GT, X, SG, SX = (t.cpu().numpy() for t in (qgT, qx, sg, sx))
    for r0 in (0, 1120, 2272):
        rows, rb = slice(r0, r0 + 32), slice(r0 // 32, r0 // 32 + 1)
        want = oracle.igemm_block_f32(GT[rows], X, np.ascontiguousarray(SG[:, rb]), SX, 1)
        same(dw[rows], want, f"wgrad rows {r0}")


def test_gemm_entry_points_can_be_captured_in_a_graph(jf, oracle):
    """The GEMM entry points only launch kernels (no allocation, no synchronisation, no memset), so a caller can record
    them into a HIP graph: three replays, with eager work and synchronisations in between, all give the eager result."""
    M, N, K = 256, 384, 2048
    A, Bkn, sa, sb = make_problem(5, M, N, K, f16=False)
    dA, dB, dsa, dsb = dev(A), dev(Bkn), dev(sa), dev(sb)
    L = jf.lib()
    nb = L.jf_igemm_block_fp_workspace_bytes(M, N, K, jf.B_KN, 4)
    assert nb > 0
    ws = torch.empty(nb, dtype=torch.int8, device="cuda")
    q = torch.empty((M, N), dtype=torch.int8, device="cuda")
    sc = torch.empty((M // QB, N // QB), dtype=torch.float32, device="cuda")
    w = torch.empty((M, N), dtype=torch.float32, device="cuda")

    def launch(stream):
        jf.check(L.jf_igemm_block_q(dA.data_ptr(), dB.data_ptr(), dsa.data_ptr(), dsb.data_ptr(), None, None, q.data_ptr(),
                                    sc.data_ptr(), M, N, K, jf.B_KN, 1, 0, 0, jf.ROUND_STOCHASTIC, 9, 4, None, 0, stream))
        jf.check(L.jf_igemm_block_fp(dA.data_ptr(), dB.data_ptr(), dsa.data_ptr(), dsb.data_ptr(), w.data_ptr(), M, N, K,
                                     jf.A_MK, jf.B_KN, 1, 0, 0, 1, 4, ws.data_ptr(), nb, stream))

    launch(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    eq, esc, ew = q.clone(), sc.clone(), w.clone()
    parts, per = jf.splitk_plan(M, N, K, 4)
    same(ew, oracle.igemm_block_f32_splitk(A, Bkn, sa, sb, 1, parts, per), "eager split-K")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        launch(torch.cuda.current_stream().cuda_stream)
    for _ in range(3):
        q.zero_(); sc.zero_(); w.zero_(); ws.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(q, eq) and torch.equal(sc, esc) and torch.equal(w, ew)


@pytest.mark.parametrize("approx", [0, 1])
@pytest.mark.parametrize("f16", [True, False])
@pytest.mark.parametrize("M,N,K", [(128, 256, 96), (96, 160, 224), (256, 384, 544), (32, 32, 32)])
def test_forward_gemm_with_fused_gelu(jf, oracle, M, N, K, f16, approx):
    """The fused entry point returns, bit for bit, what the GEMM and then the GELU kernel return (both of which are
    checked against the oracle elsewhere and here)."""
    print(f"case q+gelu M={M} N={N} K={K} f16={f16} approx={approx}", flush=True)
    A, Bkn, sa, sb = make_problem(M + N * 5 + K, M, N, K, f16)
    sa = sa * np.float32(0.05)                                    # outputs of a few units: the interesting range of GELU
    B = b_of(Bkn, 0)
    st = np.float16 if f16 else np.float32
    sa = sa.astype(st).astype(np.float32)
    sdt = "f16" if f16 else "f32"
    dA, dB, dsa, dsb = dev(A), dev(B), dev(sa.astype(st)), dev(sb.astype(st))
    eps = 5e-5 if approx == 0 else 0.0
    q, s, qg, sg = jf.igemm_block_q_gelu(dA, dB, dsa, dsb, approx, eps)
    q0, s0 = jf.igemm_block_q(dA, dB, dsa, dsb, jf.B_NK)
    qg0, sg0 = jf.gelu_fwd(q0, s0, approx, eps)
    assert torch.equal(q, q0) and torch.equal(s, s0) and torch.equal(qg, qg0) and torch.equal(sg, sg0)
    wq, ws = oracle.igemm_block_q(A, B, sa, sb, 0, scale_dtype=sdt)
    wg, wgs = oracle.gelu_fwd(wq, ws.astype(np.float32), approx, eps, scale_dtype=sdt)
    same(q, wq, "codes")
    same(s, ws, "scales")
    same(qg, wg, "gelu codes")
    same(sg, wgs, "gelu scales")
    assert qg.cpu().numpy().any()


@pytest.mark.parametrize("M,N,K,x1,y,f16,bias", [
    (32, 32, 32, torch.float32, torch.float32, True, False),             # one block
    (64, 160, 96, torch.float16, torch.bfloat16, False, True),           # a tile of one block's width
    (1248, 768, 160, torch.bfloat16, torch.float32, True, True),
    (256, 288, 1056, torch.float32, torch.float16, True, False),
    (2048, 1024, 32, torch.float32, torch.float32, True, False),         # the last launch of one kernel ...
    (2080, 1024, 32, torch.float32, torch.float32, True, True),          # ... and the first of two, in place
    (32, 32, 16416, torch.bfloat16, torch.bfloat16, False, False),       # ... by the length of K
])
def test_quantised_with_residual_addition(jf, oracle, M, N, K, x1, y, f16, bias):
    """The fused entry point returns, bit for bit, what the GEMM and then the addition return (both of which are checked against the
    oracle elsewhere)."""
    print(f"case q+add M={M} N={N} K={K} {x1} {y} f16={f16} bias={bias}", flush=True)
    A, Bkn, sa, sb = make_problem(M + N * 3 + K, M, N, K, f16)
    st = np.float16 if f16 else np.float32
    sa = sa * np.float32(0.05)
    dA, dB, dsa, dsb = dev(A), dev(b_of(Bkn, 0)), dev(sa.astype(st)), dev(sb.astype(st))
    gen = torch.Generator("cuda").manual_seed(M + K)
    res = torch.randn((M, N), device="cuda", generator=gen).to(x1)
    res[:32, :32] = 0
    if M > 32:                                                    # blocks with a NaN, an infinity, both
        res[32, 0] = res[33, 64] = float("nan")
        res[34, 32] = res[35, 64] = float("inf")
    b = torch.randn(N, device="cuda", generator=gen) if bias else None
    bmax = b.abs().max().reshape(1) if bias else None
    for rounding in (jf.ROUND_TRUNC, jf.ROUND_NEAREST):
        got = jf.igemm_block_q_add(dA, dB, dsa, dsb, res, rounding, b, bmax, out_dtype=y)
        q0, s0 = jf.igemm_block_q(dA, dB, dsa, dsb, jf.B_NK, bias=b, biasmax=bmax)
        for g, w, name in zip(got, jf.add(res, q0, s0, rounding, with_stats=True, out_dtype=y), ("sum", "codes", "scales", "row sums", "row squares")):
            if g.is_floating_point():
                assert torch.equal(g.isnan(), w.isnan()), name
                g, w = g.nan_to_num(7.0), w.nan_to_num(7.0)
            assert torch.equal(g, w), name
    assert got[1].any()


@pytest.mark.parametrize("R,C_in,C_out,splitk,f16,quantize", [
    (32, 32, 32, 0, True, True),                     # one tile each
    (96, 160, 224, 0, False, False),
    (512, 768, 2304, 0, True, False),
    (512, 768, 2304, 1, False, True),
    (2048, 128, 256, 0, True, True),                 # weight gradient in parts
    (1024, 1024, 64, 1, True, False),                # 256 tiles of 32x128 ...
    (1056, 1024, 64, 1, False, False),               # ... and one row of them more: 128x128
    (1056, 1024, 2080, 0, True, True),               # 32x128 again, for a long K
    (2080, 1056, 96, 0, False, True),                # ragged tiles
    (12288, 1024, 32, 0, True, True),                # the last launch of one kernel on 256 CUs ...
    (12320, 1024, 32, 0, True, True),                # ... and the first of two
])
def test_both_gradients_of_a_linear_layer_in_one_launch(jf, R, C_in, C_out, splitk, f16, quantize):
    """Bit for bit what the two entry points return (both of which are checked against the oracle elsewhere)."""
    print(f"case bwd R={R} C_in={C_in} C_out={C_out} splitk={splitk} f16={f16} quantize={quantize}", flush=True)
    rng = np.random.default_rng(R + C_in * 3 + C_out)
    st = np.float16 if f16 else np.float32
    block = lambda r, c: (dev(rand_codes(rng, (r, c))), dev(rand_scales(rng, (r // QB, c // QB), lo=-8, hi=-4, f16=f16).astype(st)))  # noqa: E731
    (x, sx), (g, sg), (w, sw) = block(R, C_in), block(R, C_out), block(C_out, C_in)
    L, p, seed, offset = jf.lib(), jf._ptr, 17, 8
    code = jf.SCALE_F16 if f16 else jf.SCALE_F32
    want_w = jf.igemm_block_fp(g, x, sg, sx, jf.B_KN, torch.float32, jf.A_KM, splitk)
    if quantize:
        want = jf.igemm_block_q(g, w, sg.t(), sw, jf.B_KN, rounding=jf.ROUND_STOCHASTIC, seed=seed, offset=offset)
    else:
        want = (jf.igemm_block_q_dequant(g, w, sg.t(), sw, jf.B_KN, torch.float16, rounding=jf.ROUND_STOCHASTIC, seed=seed, offset=offset),)
    dx = torch.empty_like(want[0])
    ds = torch.empty_like(want[1]) if quantize else None
    dw = torch.empty_like(want_w)
    nb = L.jf_igemm_block_fp_workspace_bytes(C_out, C_in, R, jf.B_KN, splitk)
    ws = torch.empty(max(nb, 16), dtype=torch.int8, device="cuda")
    jf.check(L.jf_linear_bwd(p(x), p(sx), p(g), p(sg), p(w), p(sw), R, C_in, C_out, code, p(dx), p(ds), jf.FP_F16, seed, offset, p(dw),
                             jf.FP_F32, splitk, p(ws), nb, jf._stream()))
    assert torch.equal(dw, want_w) and torch.equal(dx, want[0])
    assert ds is None or torch.equal(ds, want[1])


@pytest.mark.parametrize("R,C,f16", [(64, 96, True), (1024, 256, True), (2112, 544, False), (4096, 1056, True), (4128, 1056, True)])
def test_weight_gradients_with_an_activation_gradient(jf, R, C, f16):
    """In 32x128 tiles, in 128x128 tiles and, the last one, apart: bit for bit what the two entry points return."""
    print(f"case wgrads+dgrad R={R} C={C} f16={f16}", flush=True)
    rng = np.random.default_rng(R + C)
    st = np.float16 if f16 else np.float32
    block = lambda r, c: (dev(rand_codes(rng, (r, c))), dev(rand_scales(rng, (r // QB, c // QB), lo=-8, hi=-4, f16=f16).astype(st)))  # noqa: E731
    gs, xs = [block(R, 3 * C), block(R, 32)], [block(R, C), block(R, 64)]
    w, sw = block(3 * C, C)
    terms = torch.rand((R // QB, C), device="cuda")
    want, (wsum,) = jf.wgrad_many(gs, xs, terms=[terms])
    wq, ws_ = jf.igemm_block_q(gs[0][0], w, gs[0][1].t(), sw, jf.B_KN, rounding=jf.ROUND_STOCHASTIC, seed=5, offset=16)
    L, p = jf.lib(), jf._ptr
    ptrs = lambda ts: (ctypes.c_void_p * len(ts))(*[t.data_ptr() for t in ts])  # noqa: E731
    ints = lambda *v: (ctypes.c_int * len(v))(*v)  # noqa: E731
    out, total, q, s = [torch.empty_like(t) for t in want], torch.empty_like(wsum), torch.empty_like(wq), torch.empty_like(ws_)
    Ms, Ns = ints(3 * C, 32), ints(C, 64)
    nb = L.jf_wgrad_many_workspace_bytes(2, Ms, Ns, R)
    ws = torch.empty(max(nb, 16), dtype=torch.int8, device="cuda")
    operands = (ptrs([t for t, _ in gs]), ptrs([t for _, t in gs]), ptrs([t for t, _ in xs]), ptrs([t for _, t in xs]), ptrs(out), Ms, Ns, R,
                jf.SCALE_F16 if f16 else jf.SCALE_F32, jf.FP_F32)
    jf.check(L.jf_wgrad_many_dgrad(p(w), p(sw), p(q), p(s), 5, 16, 2, *operands, p(ws), nb, jf._stream()))
    jf.check(L.jf_wgrad_many_finish(2, *operands, 1, ptrs([terms]), ints(C), ptrs([total]), p(ws), nb, jf._stream()))
    assert torch.equal(q, wq) and torch.equal(s, ws_) and torch.equal(total, wsum)
    assert all(torch.equal(a, b) for a, b in zip(out, want))


@pytest.mark.parametrize("approx", [0, 1])
@pytest.mark.parametrize("f16", [True, False])
@pytest.mark.parametrize("M,N,K", [(128, 256, 96), (96, 160, 224), (256, 384, 544), (32, 32, 32)])
def test_dgrad_gemm_with_fused_gelu_backward(jf, oracle, M, N, K, f16, approx):
    """The fused entry point returns, bit for bit, what the stochastic activation-gradient GEMM and then the GELU
    backward kernel return (with the same two noise streams), and what the oracle computes for that sequence."""
    print(f"case dgrad+gelu_bwd M={M} N={N} K={K} f16={f16} approx={approx}", flush=True)
    A, Bkn, sa, sb = make_problem(M * 2 + N + K * 3, M, N, K, f16)
    rng = np.random.default_rng(M + N + K)
    st = np.float16 if f16 else np.float32
    sdt = "f16" if f16 else "f32"
    xq = rand_codes(rng, (M, N))
    xs = (rand_scales(rng, (M // QB, N // QB), lo=-6, hi=-4, f16=f16)).astype(np.float32)    # pre-activations of a few units
    dA, dB, dsa, dsb, dxq, dxs = dev(A), dev(Bkn), dev(sa.astype(st)), dev(sb.astype(st)), dev(xq), dev(xs.astype(st))
    for rounding2, stochastic2 in ((jf.ROUND_STOCHASTIC, True), (jf.ROUND_NEAREST, False)):
        q, s = jf.igemm_block_q_gelu_bwd(dA, dB, dsa, dsb, dxq, dxs, approx, rounding2, seed=11, offset=3, gelu_seed=12, gelu_offset=40)
        q0, s0 = jf.igemm_block_q(dA, dB, dsa, dsb, jf.B_KN, rounding=jf.ROUND_STOCHASTIC, seed=11, offset=3)
        q1, s1 = jf.gelu_bwd(dxq, dxs, q0, s0, approx, rounding2, seed=12, offset=40)
        assert torch.equal(q, q1) and torch.equal(s, s1)
        wq, ws = oracle.igemm_block_q(A, Bkn, sa, sb, 1, stochastic=True, seed=11, offset=3, scale_dtype=sdt)
        wg, wgs = oracle.gelu_bwd(xq, xs, wq, ws.astype(np.float32), approx, stochastic2, 12, 40, scale_dtype=sdt)
        same(q, wg, "codes")
        same(s, wgs, "scales")
        assert q.cpu().numpy().any()
    with pytest.raises(RuntimeError):
        jf.igemm_block_q_gelu_bwd(dA, dB, dsa, dsb, dxq[:, : N // 2].contiguous(), dxs[:, : N // 64].contiguous(), approx)


@pytest.mark.parametrize("f16", [True, False])
@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("M,N,K", [(128, 256, 96), (96, 160, 224), (256, 384, 544), (32, 32, 32), (160, 1632, 64)])
def test_gemm_with_fused_dequantisation(jf, oracle, M, N, K, layout, f16):
    """jf_igemm_block_q_dequant returns, bit for bit, the dequantisation of what jf_igemm_block_q stores (both roundings,
    every output type), and the oracle's requantised result times its stored scale."""
    print(f"case q+dequant M={M} N={N} K={K} layout={layout} f16={f16}", flush=True)
    A, Bkn, sa, sb = make_problem(M + 5 * N + K, M, N, K, f16)
    st = np.float16 if f16 else np.float32
    dA, dB, dsa, dsb = dev(A), dev(b_of(Bkn, layout)), dev(sa.astype(st)), dev(sb.astype(st))
    bias = torch.linspace(-0.5, 0.5, N).cuda()
    biasmax = bias.abs().max().reshape(1)
    for rounding in (jf.ROUND_NEAREST, jf.ROUND_STOCHASTIC):
        q, s = jf.igemm_block_q(dA, dB, dsa, dsb, layout, rounding=rounding, seed=21, offset=8)
        assert q.cpu().numpy().any()
        for odt in (torch.float16, torch.bfloat16, torch.float32):
            got = jf.igemm_block_q_dequant(dA, dB, dsa, dsb, layout, out_dtype=odt, rounding=rounding, seed=21, offset=8)
            want = jf.dequantize(q, s, out_dtype=odt)
            assert got.dtype == odt and torch.equal(got.view(torch.int16 if odt != torch.float32 else torch.int32),
                                                    want.view(torch.int16 if odt != torch.float32 else torch.int32))
        wq, ws = oracle.igemm_block_q(A, Bkn, sa, sb, 1, stochastic=rounding == jf.ROUND_STOCHASTIC, seed=21, offset=8,
                                      scale_dtype="f16" if f16 else "f32")
        want32 = (wq.astype(np.float32).reshape(M // QB, QB, N // QB, QB) * ws.astype(np.float32)[:, None, :, None]).reshape(M, N)
        got32 = jf.igemm_block_q_dequant(dA, dB, dsa, dsb, layout, out_dtype=torch.float32, rounding=rounding, seed=21, offset=8)
        same(got32, want32, "dequantised result")
    # with a bias and its maximum (deterministic forward form), default output type = the scales' type
    qb, sbb = jf.igemm_block_q(dA, dB, dsa, dsb, layout, bias=bias, biasmax=biasmax)
    gotb = jf.igemm_block_q_dequant(dA, dB, dsa, dsb, layout, bias=bias, biasmax=biasmax)
    assert gotb.dtype == dsa.dtype and torch.equal(gotb, jf.dequantize(qb, sbb, out_dtype=dsa.dtype))
    with pytest.raises(RuntimeError):
        jf.igemm_block_q_dequant(dA, dB, dsa, dsb, layout, out_dtype=torch.float64)


@pytest.mark.gpu
def test_phase_recording_build_gives_the_same_bits_and_ordered_phases(jf):
    """The profiling build of the requantising GEMM (jf_prof_igemm_block_q of the measurement library) stores the same
    codes and scales as the product library's kernel, and every workgroup's phase stamps are in order with a plausible
    shader clock."""
    g = torch.Generator().manual_seed(5)
    M, N, K = 384, 416, 256                                     # 3 x 4 tiles, the last tile column a quarter full
    A = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int8).cuda()
    B = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8).cuda()
    sa = (torch.rand(K // 32, M // 32, generator=g) * 0.01 + 1e-3).cuda()
    sb = (torch.rand(K // 32, N // 32, generator=g) * 0.01 + 1e-3).cuda()
    for rounding, kw in ((jf.ROUND_NEAREST, {}), (jf.ROUND_STOCHASTIC, dict(seed=3, offset=8))):
        q0, s0 = jf.igemm_block_q(A, B, sa, sb, jf.B_NK, rounding=rounding, **kw)
        q, s, ph = jf.igemm_phases(A, B, sa, sb, jf.B_NK, rounding=rounding, **kw)
        assert torch.equal(q, q0) and torch.equal(s, s0)
        us = ph["us"]
        assert us.shape == (12, 6) and (us[:, 1:] >= us[:, :-1]).all() and us[:, 5].max() < 1e4
        assert ((ph["k_loop_MHz"] > 300) & (ph["k_loop_MHz"] < 3500)).all()


# 165 workgroups of 32x128 tiles; 297 of 64x128 for the requantised result, 153 of 128x128 for the float one (585 would be small ones).  K: rings of two and of three stages with one stage, fewer
# than, as many as, more than their depth, every length of the last one; the longest row the small tiles take and the next one
@pytest.mark.parametrize("M,N,K", [(m, n, k) for m, n in ((1056, 544), (2080, 1056)) for k in (32, 64, 96, 128, 160, 288, 384, 416, 896)]
                         + [(32, 160, 16384), (32, 160, 16416)])
def test_both_tile_sizes_at_every_ring_fill(jf, oracle, M, N, K):
    print(f"case M={M} N={N} K={K}", flush=True)
    A, Bkn, sa, sb = make_problem(M + N + K, M, N, K)
    dA, dsa, dsb = dev(A), dev(sa.astype(np.float16)), dev(sb.astype(np.float16))
    for layout in (0, 1):
        B = b_of(Bkn, layout)
        want = oracle.igemm_block_f32(A, B, sa, sb, layout)
        same(jf.igemm_block_fp(dA, dev(B), dsa, dsb, layout, torch.float32), want, "fp32 accumulators")
        q, sc = jf.igemm_block_q(dA, dev(B), dsa, dsb, layout, rounding=jf.ROUND_STOCHASTIC, seed=4, offset=8)
        wq, wsc = oracle.igemm_block_q(A, B, sa, sb, layout, stochastic=True, seed=4, offset=8, scale_dtype="f16")
        same(q, wq, "SR codes")
        same(sc, wsc, "SR scales")


# 32x64 tiles whose blocks two waves share (up to one per CU, 256): 15 of them with a ragged last column at every fill of the six-deep ring
# and every length of its last stage, all 256, and the long row; with 288 tiles and a longer row 32x128 again
@pytest.mark.parametrize("M,N,K", [(96, 160, k) for k in (32, 64, 96, 128, 160, 640, 768, 800, 896, 1056, 1632)]
                         + [(1024, 512, 288), (32, 64, 16384), (1024, 544, 288)])
def test_tiles_whose_blocks_two_waves_share(jf, oracle, M, N, K):
    test_both_tile_sizes_at_every_ring_fill(jf, oracle, M, N, K)
    test_two_tile_sizes_in_one_launch(jf, oracle, M, N, K)       # (every other epilogue)
    test_quantised_with_residual_addition(jf, oracle, M, N, K, torch.bfloat16, torch.float32, True, True)


# 64x128 tiles with one block per wave (up to one per CU, more than one of 32x128 each): few, the last row of them half empty, at fills of the two-deep
# ring and lengths of its last stage; many, columns that end inside a tile; all 256; one row of tiles more
@pytest.mark.parametrize("M,N,K", [(1056, 1024, k) for k in (32, 96, 128, 160, 288, 416)] + [(1760, 1056, 448), (2048, 1024, 64), (2080, 1024, 96)])
def test_tiles_of_64_rows_with_one_block_per_wave(jf, oracle, M, N, K):
    test_both_tile_sizes_at_every_ring_fill(jf, oracle, M, N, K)
    test_two_tile_sizes_in_one_launch(jf, oracle, M, N, K)       # (every other epilogue)
    test_quantised_with_residual_addition(jf, oracle, M, N, K, torch.bfloat16, torch.float32, True, True)


def test_the_longest_row_of_the_tiles_of_64_rows(jf):
    gen = torch.Generator(device="cuda").manual_seed(2)
    a, sa = jf.quantize(torch.randn(1056, 16384, device="cuda", generator=gen))
    b, sb = jf.quantize(torch.randn(1024, 16384, device="cuda", generator=gen))
    q, s = jf.igemm_block_q(a, b, sa.t().contiguous(), sb.t().contiguous(), jf.B_NK)
    for r in range(0, 1056, 352):                                # (parts of 32x64 tiles)
        qp, sp = jf.igemm_block_q(a[r:r + 352], b, sa[r // 32:r // 32 + 11].t().contiguous(), sb.t().contiguous(), jf.B_NK)
        assert torch.equal(q[r:r + 352], qp) and torch.equal(s[r // 32:r // 32 + 11], sp)


# the residual addition in the epilogue of every larger tile: 128x128 with ragged rows and columns, both sizes in one launch, 64x128; one K block
# and a short last stage
@pytest.mark.parametrize("M,N,K,x1,y", [(2080, 3104, 32, torch.float32, torch.float32), (2080, 3104, 160, torch.bfloat16, torch.bfloat16),
                                        (5408, 768, 96, torch.float16, torch.float32), (2080, 1056, 288, torch.float32, torch.float16)])
def test_residual_addition_in_the_large_tiles(jf, oracle, M, N, K, x1, y):
    test_quantised_with_residual_addition(jf, oracle, M, N, K, x1, y, True, True)
    test_quantised_with_residual_addition(jf, oracle, M, N, K, x1, y, False, False)


# activation gradients in 32x64 tiles beside weight gradients, one workgroup per CU: 248 and 8 of them, and one row of tiles more (32x128)
@pytest.mark.parametrize("R,C_in,C_out,f16", [(992, 512, 64, True), (1024, 512, 64, True), (160, 544, 1056, False)])
def test_both_gradients_with_tiles_that_two_waves_share(jf, R, C_in, C_out, f16):
    for quantize in (True, False):
        test_both_gradients_of_a_linear_layer_in_one_launch(jf, R, C_in, C_out, 0, f16, quantize)


# 64x128 tiles with a GELU behind them: the fewest and the most big tiles that they take the place of, one row of tiles less (128x128), the last row
# and column of tiles ragged
@pytest.mark.parametrize("M,N,K", [(4096, 1056, 96), (2080, 2080, 32), (2016, 2976, 160), (2048, 2048, 64)])
def test_gelu_in_the_64_row_tiles(jf, oracle, M, N, K):
    test_two_tile_sizes_in_one_launch(jf, oracle, M, N, K)


# weight gradients in 32x128 tiles beside the activation gradient, up to one workgroup per CU (256): columns of the gradient that end inside a staged
# line, every length of the last stage, K splits with a short last part; 256 workgroups with 32x64 tiles of the activation gradient, one row of tiles
# more (its 32x128 tiles), and too many for either (128x128 beside 32x64 tiles); three times as many K blocks of the activation gradient as of the weight
# gradient (128x128 beside 32x128) and one more (beside 32x64)
@pytest.mark.parametrize("R,C_in,C_out", [(r, 160, 288) for r in (32, 64, 96, 128, 160, 288, 416)] + [(1056, 128, 256), (2048, 96, 544), (480, 512, 1088), (480, 512, 1120), (480, 512, 2080), (352, 992, 1056), (352, 992, 1088)])
def test_weight_gradients_in_tiles_of_32_rows(jf, R, C_in, C_out):
    test_both_gradients_of_a_linear_layer_in_one_launch(jf, R, C_in, C_out, 0, True, True)
    test_both_gradients_of_a_linear_layer_in_one_launch(jf, R, C_in, C_out, 1, False, False)


def test_extreme_scales_in_the_weight_gradients_of_32_rows(jf):
    """Products of scales beyond 2^102: the blocks they touch are formed again from memory, also of a later K split."""
    rng = np.random.default_rng(1)
    R, C_in, C_out = 1056, 128, 160
    g, x, w = dev(rand_codes(rng, (R, C_out))), dev(rand_codes(rng, (R, C_in))), dev(rand_codes(rng, (C_out, C_in)))
    sg, sx, sw = (torch.ones((r // 32, c // 32), device="cuda") for r, c in ((R, C_out), (R, C_in), (C_out, C_in)))
    # (2^104 times a block product, below 32 * 128^2 = 2^19, is finite)
    sg[1, 2], sx[1, 1], sg[30, 0], sx[30, 3] = 2.0 ** 52, 2.0 ** 52, 2.0 ** 53, 2.0 ** 51
    dx, ds, dw = torch.empty_like(x), torch.empty_like(sx), torch.empty((C_out, C_in), device="cuda")
    L, p = jf.lib(), jf._ptr
    for splitk in (0, 1):
        nb = L.jf_igemm_block_fp_workspace_bytes(C_out, C_in, R, jf.B_KN, splitk)
        ws = torch.empty(max(nb, 16), dtype=torch.int8, device="cuda")
        jf.check(L.jf_linear_bwd(p(x), p(sx), p(g), p(sg), p(w), p(sw), R, C_in, C_out, jf.SCALE_F32, p(dx), p(ds), jf.FP_F16, 1, 8, p(dw), jf.FP_F32, splitk, p(ws), nb, jf._stream()))
        want = jf.igemm_block_fp(g, x, sg, sx, jf.B_KN, torch.float32, jf.A_KM, splitk)
        assert torch.isfinite(want).all() and torch.equal(dw, want)


# 425 tiles of 128x128 (825 of 64x128, which would not all be resident), the last row and column of them ragged: every ring fill
@pytest.mark.parametrize("K", [32, 64, 96, 128, 160, 288, 384, 416])
def test_the_large_tiles_at_every_ring_fill(jf, oracle, K):
    test_both_tile_sizes_at_every_ring_fill(jf, oracle, 2080, 3104, K)


# 128x128 and 32x128 tiles in one launch (256 CUs): behind one big tile per CU the fewest and the most small ones and one row block more
# (64x128 only, 128x128 with the GELU forward), columns that end inside a tile; behind two the fewest and the most; behind four; behind six
@pytest.mark.parametrize("M,N,K", [(5408, 768, 32), (6720, 768, 416), (6752, 768, 32), (4704, 800, 160), (10912, 768, 160), (13600, 768, 32),
                                   (4352, 4096, 96), (6176, 4096, 32)])
def test_two_tile_sizes_in_one_launch(jf, oracle, M, N, K):
    print(f"case M={M} N={N} K={K}", flush=True)
    A, Bkn, sa, sb = make_problem(M + N + K, M, N, K)
    d = lambda t: dev(t.astype(np.float16))  # noqa: E731
    dA, dsa, dsb, dkn, dnk = dev(A), d(sa), d(sb), dev(Bkn), dev(b_of(Bkn, 0))
    q, sc = jf.igemm_block_q(dA, dnk, dsa, dsb, jf.B_NK)
    wq, wsc = oracle.igemm_block_q(A, b_of(Bkn, 0), sa, sb, 0, scale_dtype="f16")
    same(q, wq, "codes")
    same(sc, wsc, "scales")
    for got, want in zip(jf.igemm_block_q_gelu(dA, dnk, dsa, dsb), (q, sc) + tuple(jf.gelu_fwd(q, sc))):
        assert torch.equal(got, want)
    assert torch.equal(jf.igemm_block_q_dequant(dA, dnk, dsa, dsb, jf.B_NK, torch.float32), jf.dequantize(q, sc, torch.float32))
    g, gs = jf.igemm_block_q(dA, dkn, dsa, dsb, jf.B_KN, rounding=jf.ROUND_STOCHASTIC, seed=4, offset=8)
    wq, wsc = oracle.igemm_block_q(A, Bkn, sa, sb, 1, stochastic=True, seed=4, offset=8, scale_dtype="f16")
    same(g, wq, "SR codes")
    same(gs, wsc, "SR scales")
    got = jf.igemm_block_q_gelu_bwd(dA, dkn, dsa, dsb, q, sc, seed=4, offset=8, gelu_seed=5, gelu_offset=4)
    want = jf.gelu_bwd(q, sc, g, gs, rounding=jf.ROUND_STOCHASTIC, seed=5, offset=4)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


# behind three big tiles per CU one row block of small ones, columns that end inside a tile; as many as CUs, and one row block more (128x128 only);
# behind five the fewest and the most; behind seven and nine; behind four close to two per CU, and one row block more
@pytest.mark.parametrize("M,N,K", [(16416, 736, 160), (13312, 1024, 32), (13344, 1024, 32), (27296, 768, 32), (5376, 4096, 96), (7328, 4096, 32), (12320, 3072, 32),
                                   (6048, 3072, 1536), (6080, 3072, 1536)])
def test_two_tile_sizes_behind_three_and_more(jf, oracle, M, N, K):
    test_two_tile_sizes_in_one_launch(jf, oracle, M, N, K)
    test_quantised_with_residual_addition(jf, oracle, M, N, K, torch.bfloat16, torch.float32, True, True)


@pytest.mark.parametrize("K", [32, 480, 512, 1056])               # one K block, the longest without and the shortest with a K split, a ragged split
@pytest.mark.parametrize("widths", [[(96, 32)], [(384, 160), (128, 160), (512, 128), (32, 544)]])
@pytest.mark.parametrize("f16,out", [(True, torch.float32), (False, torch.bfloat16)])
def test_weight_gradients_in_one_launch(jf, oracle, K, widths, f16, out):
    print(f"case K={K} widths={widths}", flush=True)
    rng = np.random.default_rng(K)
    st = np.float16 if f16 else np.float32
    operand = lambda c: (rand_codes(rng, (K, c)), rand_scales(rng, (K // QB, c // QB), f16=f16))  # noqa: E731
    gs, xs = [operand(m) for m, _ in widths], [operand(n) for _, n in widths]
    terms = [rng.standard_normal((K // QB, c)).astype(np.float32) for c in (32, 544)]
    d = lambda ts: [(dev(q), dev(s.astype(st))) for q, s in ts]  # noqa: E731
    got, sums = jf.wgrad_many(d(gs), d(xs), out, [dev(t) for t in terms])
    for (g, sg), (x, sx), o in zip(gs, xs, got):
        want = torch.from_numpy(oracle.igemm_block_f32(np.ascontiguousarray(g.T), x, sg, sx, 1))
        if K < 512:
            assert torch.equal(o.cpu(), want.to(out))
        else:
            assert float((o.cpu().double() - want.double()).norm() / want.double().norm()) < (1e-5 if out == torch.float32 else 4e-3)
    for t, s in zip(terms, sums):
        np.testing.assert_allclose(s.cpu().numpy(), t.astype(np.float64).sum(0), atol=1e-5)
    assert jf.wgrad_many(d(gs[:1]), d(xs[:1]), out)[0][0].shape == got[0].shape


@pytest.mark.parametrize("C,K", [(256, 1024), (768, 12288), (1600, 8192), (768, 1248), (512, 4096), (192, 2048)])
def test_weight_gradients_in_one_launch_round_no_more_than_alone(jf, C, K):
    """The gradients of a block's four layers against float64: the one launch sums K in an order whose rounding error is no larger
    than that of each gradient in a launch of its own (2 % for the scatter of a norm over a million rounding errors)."""
    print(f"case C={C} K={K}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(C + K)
    codes = lambda c: torch.randint(-127, 128, (K, c), device="cuda", dtype=torch.int8, generator=gen)  # noqa: E731
    scales = lambda c: (1 + torch.rand(K // QB, c // QB, device="cuda", generator=gen))  # noqa: E731
    widths = [(3 * C, C), (C, C), (4 * C, C), (C, 4 * C)]
    gs, xs = [(codes(m), scales(m)) for m, _ in widths], [(codes(n), scales(n)) for _, n in widths]
    got, _ = jf.wgrad_many(gs, xs)
    value = lambda q, s: q.double() * s.double().repeat_interleave(QB, 0).repeat_interleave(QB, 1)  # noqa: E731
    for (g, sg), (x, sx), many in zip(gs, xs, got):
        alone = jf.igemm_block_fp(g, x, sg, sx, jf.B_KN, torch.float32, a_layout=jf.A_KM, splitk=0)
        exact = value(g, sg).t().contiguous() @ value(x, sx)
        error = lambda o: float((o.double() - exact).norm() / exact.norm())  # noqa: E731
        print(f"  {g.shape[1]} x {x.shape[1]}: alone {error(alone):.3e}, together {error(many):.3e}", flush=True)
        assert error(many) <= 1.02 * error(alone) and error(alone) < 1e-6


# (workgroups per tile along K, K blocks of each, K blocks of a part inside them) of each gradient on 256 compute units: parts inside one
# workgroup; a short last stage alone in the last part, and a short last part; parts inside the parts of a K split, ragged tiles and a
# ragged last split; a gradient with a split of its own beside gradients with parts inside workgroups
@pytest.mark.parametrize("C,K,plan", [(512, 2048, [(1, 64, 16)] * 4), (512, 2080, [(1, 65, 16)] * 4), (480, 2144, [(1, 67, 16)] * 4), (512, 1056, [(1, 33, 16)] * 4),
                                      (416, 4128, [(3, 44, 16)] * 4), (768, 4096, [(1, 128, 32), (8, 16, 0), (1, 128, 40), (1, 128, 40)])])
@pytest.mark.parametrize("f16,out", [(True, torch.float16), (False, torch.float32)])
def test_weight_gradients_summed_in_parts(jf, oracle, C, K, plan, f16, out):
    """Bit for bit the sums in the order of the plan, also where a scale product is too large for the kernel's fast accumulation."""
    print(f"case C={C} K={K} f16={f16}", flush=True)
    rng = np.random.default_rng(C + K)
    st = np.float16 if f16 else np.float32
    widths = [(3 * C, C), (C, C), (4 * C, C), (C, 4 * C)]
    operand = lambda c: (rand_codes(rng, (K, c)), rand_scales(rng, (K // QB, c // QB), f16=f16))  # noqa: E731
    gs, xs = [operand(m) for m, _ in widths], [operand(n) for _, n in widths]
    if not f16:
        gs[0][1][20, 1] = xs[0][1][20, 2] = 2.0 ** 53          # one block product beyond 2^102, in the second part or later
    d = lambda ts: [(dev(q), dev(s.astype(st))) for q, s in ts]  # noqa: E731
    for (g, sg), (x, sx), (parts, kb, fold), o in zip(gs, xs, plan, jf.wgrad_many(d(gs), d(xs), out)[0]):
        A, total = np.ascontiguousarray(g.T), None
        for s in range(parts):
            lo, hi = s * kb, min((s + 1) * kb, K // QB)
            f = fold or hi - lo
            part = oracle.igemm_block_f32_splitk(np.ascontiguousarray(A[:, lo * QB:hi * QB]), np.ascontiguousarray(x[lo * QB:hi * QB]),
                                                 np.ascontiguousarray(sg[lo:hi]), np.ascontiguousarray(sx[lo:hi]), 1, -(-(hi - lo) // f), f)
            total = part if total is None else total + part
        same(o, torch.from_numpy(total).to(out).numpy(), f"dW {g.shape[1]} x {x.shape[1]}")
