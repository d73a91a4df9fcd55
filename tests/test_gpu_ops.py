"""GPU parity of every decode op (HipOps over libdryft_decode.so) against the CPU oracle.

Tolerances: bf16 op outputs within rtol 2e-2 / atol 2e-2 of the oracle (
test_fused.py:25-29 uses 0.02 * max(1, |ref|max)); attention within 0.02 of an fp64 loop
(test_attn.py:40); exact-sum known answers, V cache writes, KV indexing and argmax bit-exact.
"""
import pytest
import torch

import known_answers as ka
from oracle.reference import TorchOps, attn_reference_fp64, fake_engine

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _hip(e_cpu):
    """HipOps over a GPU copy of a fake engine namespace."""
    from dryft_amd.hipops import HipOps
    import types
    e = types.SimpleNamespace(**vars(e_cpu))
    e.dev = torch.device("cuda")
    e.cos, e.sin = e_cpu.cos.cuda(), e_cpu.sin.cuda()
    return HipOps(e)


def close(got, ref, rtol=2e-2, atol=2e-2):
    got, ref = got.float().cpu(), ref.float().cpu()
    d = (got - ref).abs()
    ok = (d <= atol + rtol * ref.abs()).all().item()
    assert ok, f"max|diff| {d.max().item():.4g}"
    return d.max().item()


@pytest.fixture(scope="module")
def small(cuda):
    e = fake_engine(nh=8, nkv=2, hd=128, rope_len=64)
    return TorchOps(e), _hip(e), e


# ------------------------------------------------------------------------ known answers
def test_known_silu(small):
    _, hip, _ = small
    out, exp = ka.case_silu(hip, "cuda")
    assert (out - exp).abs().max().item() < 0.05


def test_known_add_rms(small):
    _, hip, _ = small
    hn, h_exp, y, y_exp = ka.case_add_rms(hip, "cuda")
    assert torch.equal(hn, h_exp)
    assert (y - y_exp).abs().max().item() < 0.02


def test_known_gemv_exact(small):
    _, hip, _ = small
    out, exp = ka.case_gemv_exact(hip, "cuda")
    assert torch.equal(out, exp)


def test_known_gemv_splitk_equals_direct(small):
    _, hip, _ = small
    import dryft_amd
    L = dryft_amd.lib()
    M, N, K = 2, 32, 64
    out, exp = ka.case_gemv_exact(hip, "cuda", M, N, K)
    # force 2 splits through the raw ABI: split-K sum must equal the direct result
    x = torch.zeros(M, K)
    for row in range(M):
        x[row, row] = 1.0
        x[row, 32 + row] = 1.0
    w = torch.zeros(N, K)
    for n in range(N):
        w[n, 0] = (n % 4 + 1) * 0.125
        w[n, 32] = (n % 3 + 1) * 0.0625
        w[n, 1] = -(n % 5 + 1) * 0.125
        w[n, 33] = (n % 2 + 1) * 0.25
    xg, wg = x.to(BF).cuda(), w.to(BF).cuda()
    y = torch.empty(M, N, dtype=BF, device="cuda")
    ws = torch.empty(2 * M * N, dtype=torch.float32, device="cuda")
    cnt = torch.zeros(L.dd_gemv_counters(N), dtype=torch.int32, device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    assert L.dd_gemv(xg.data_ptr(), wg.data_ptr(), y.data_ptr(), M, N, K, 2, ws.data_ptr(),
                     cnt.data_ptr(), st) == 0
    assert not cnt.any()                                  # counters left at zero
    assert torch.equal(y.float().cpu(), exp)


def test_known_gate_up_exact(small):
    _, hip, _ = small
    out, exp = ka.case_gate_up_exact(hip, "cuda")
    assert (out - exp).abs().max().item() < 0.02


def test_known_linear_add_norm(small):
    _, hip, _ = small
    hn, h_exp, y, y_exp = ka.case_linear_add_norm_exact(hip, "cuda")
    assert torch.equal(hn, h_exp)
    assert (y - y_exp).abs().max().item() < 0.02


def test_known_attention_structured(cuda):
    q, kc, vc, pos, exp = ka.case_attention_structured()
    B, NKV, W, G, HD = q.shape
    hip = _hip(fake_engine(nh=NKV * G, nkv=NKV, hd=HD))
    out = hip.attn_decode(q.cuda(), kc.cuda(), vc.cuda(), pos.cuda(), W).double().cpu()
    assert (out - exp).abs().max().item() < 0.02


# ------------------------------------------------------------------------ norms / silu (test_fused.py shapes)
def test_rms_add_rms_silu_random(small):
    tor, hip, _ = small
    g = torch.Generator().manual_seed(0)
    h = torch.randn(5, 256, generator=g).to(BF)
    d = torch.randn(5, 256, generator=g).to(BF)
    w = torch.randn(256, generator=g).to(BF)
    close(hip.rms(h.cuda(), w.cuda()), tor.rms(h, w))
    th, ty = tor.add_rms(h, d, w)
    fh, fy = hip.add_rms(h.cuda(), d.cuda(), w.cuda())
    assert torch.equal(fh.cpu(), th)
    close(fy, ty)
    gu = torch.randn(7, 384, generator=g).to(BF)
    close(hip.silu_mul(gu.cuda()), tor.silu_mul(gu))
    # Qwen3 width
    h = torch.randn(16, 2560, generator=g).to(BF)
    w = (1 + 0.02 * torch.randn(2560, generator=g)).to(BF)
    close(hip.rms(h.cuda(), w.cuda()), tor.rms(h, w))


@pytest.mark.parametrize("M,I", [(3, 9728), (80, 1024), (1, 8)])
def test_silu_mul_vector_path(small, M, I):
    """The 16-byte silu_mul path (I % 8 == 0, aligned rows) gives the element-wise path's bits
    (forced here by an output 2 bytes off 16-byte alignment), and the oracle within tolerance."""
    from dryft_amd._lib import lib
    tor, hip, _ = small
    g = torch.Generator().manual_seed(M + I)
    gu = (torch.randn(M, 2 * I, generator=g) * 4).to(BF)
    gd = gu.cuda()
    vec = hip.silu_mul(gd)
    buf = torch.empty(M * I + 1, dtype=BF, device="cuda")
    assert lib().dd_silu_mul(gd.data_ptr(), buf.data_ptr() + 2, M, I,
                             torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(vec.view(-1), buf[1:])
    close(vec, tor.silu_mul(gu))


def test_embed_rms(small):
    tor, hip, _ = small
    g = torch.Generator().manual_seed(1)
    emb = torch.randn(1000, 2560, generator=g).to(BF)
    w = (1 + 0.02 * torch.randn(2560, generator=g)).to(BF)
    tok = torch.tensor([0, 999, 5, 5, 123])
    h, a = hip.embed_rms(tok.cuda(), emb.cuda(), w.cuda())
    assert torch.equal(h.cpu(), emb[tok])
    close(a, tor.rms(emb[tok], w))
    assert hip.err.item() == 0


# ------------------------------------------------------------------------ GEMV at the real shapes
SHAPES = {"qkv": (6144, 2560), "o": (2560, 4096), "gate_up": (19456, 2560), "down": (2560, 9728),
          "lm_head": (151936, 2560)}


@pytest.fixture(scope="module")
def weights():
    g = torch.Generator().manual_seed(0)
    return {k: (torch.randn(n, kk, generator=g) * 0.02).to(BF) for k, (n, kk) in SHAPES.items()}


# The real widths run the streaming kernels (linear.hip); with 8 columns less K is no multiple of 64, which is
# the GEMV's (gemv.hip).
@pytest.mark.parametrize("cut", [0, 8])
@pytest.mark.parametrize("name", list(SHAPES))
def test_linear_real_shapes(small, weights, name, cut):
    tor, hip, _ = small
    w = weights[name][:, :weights[name].shape[1] - cut].contiguous()
    wg = w.cuda()
    g = torch.Generator().manual_seed(2)
    for M in (1, 4, 8, 16):
        x = torch.randn(M, w.shape[1], generator=g).to(BF)
        assert hip._linear_ok(x.cuda(), wg) == (cut == 0) and hip._gemv_ok(x.cuda(), wg)
        got = hip.linear(x.cuda(), wg)
        close(got, tor.linear(x, w))
        # fp64 bound: |err| <= bf16 half-ulp of the output + fp32 accumulation error (a few
        # sqrt(K) fp32 ulps of sum|x||w|, bounded by 2^-16 of it here)
        ref64 = x.double() @ w.double().T
        err = (got.double().cpu() - ref64).abs()
        bound = ref64.abs() * 2 ** -8 + (x.double().abs() @ w.double().abs().T) * 2 ** -16
        assert (err <= bound + 1e-6).all(), (name, M)


@pytest.mark.parametrize("M,N", [(1, 65576), (8, 65576), (13, 65576), (16, 65576), (16, 40008)])
def test_gemv_multi_tile_exact(small, M, N):
    """N = 65,576 (4,099 tiles of 16 rows, not a multiple of 64 rows) at M >= 8 takes the
    unsplit GEMV with four W tiles per workgroup (M = 1: one tile); N = 40,008 (2,501 tiles)
    takes it with two. Integer x and W in [-3, 3] and K = 520 (no multiple of 64: not the streaming
    kernel's) keep every fp32 partial sum exact in any order, so the one rounding is the bf16 store:
    the fp64 product rounded to bf16 is the exact answer, bit for bit."""
    _, hip, _ = small
    K = 520
    g = torch.Generator().manual_seed(40 + M)
    x = torch.randint(-3, 4, (M, K), generator=g).to(BF)
    w = torch.randint(-3, 4, (N, K), generator=g).to(BF)
    assert not hip._linear_ok(x.cuda(), w.cuda())
    got = hip.linear(x.cuda(), w.cuda()).cpu()
    exp = (x.double() @ w.double().T).to(BF)
    assert torch.equal(got, exp)


@pytest.mark.parametrize("cut", [0, 8])
def test_gate_up_silu_real(small, weights, cut):
    tor, hip, _ = small
    w = weights["gate_up"][:, :2560 - cut].contiguous()
    g = torch.Generator().manual_seed(3)
    for M in (1, 16):
        x = torch.randn(M, 2560 - cut, generator=g).to(BF)
        assert hip._linear_ok(x.cuda(), w.cuda()) == (cut == 0)
        close(hip.gate_up_silu(x.cuda(), w.cuda()), tor.gate_up_silu(x, w))


@pytest.mark.parametrize("cut", [0, 8])
@pytest.mark.parametrize("name", ["o", "down"])
def test_linear_add_norm_real(small, weights, name, cut):
    tor, hip, _ = small
    w = weights[name][:, :weights[name].shape[1] - cut].contiguous()
    g = torch.Generator().manual_seed(4)
    lnw = (1 + 0.02 * torch.randn(2560, generator=g)).to(BF)
    for M in (1, 16):
        x = torch.randn(M, w.shape[1], generator=g).to(BF)
        h = torch.randn(M, 2560, generator=g).to(BF)
        assert hip._linear_ok(x.cuda(), w.cuda()) == (cut == 0)
        hn, y = hip.linear_add_norm(x.cuda(), w.cuda(), h.cuda(), lnw.cuda())
        rh, ry = tor.linear_add_norm(x, w, h, lnw)
        close(hn, rh)
        close(y, ry)


# the GEMV family (K % 64 != 0) at one tile and a ragged last one, splits of K, and 1 to 16 rows
@pytest.mark.parametrize("M", [1, 5, 16])
@pytest.mark.parametrize("N,K", [(8, 72), (72, 200), (1000, 1032), (2560, 2568)])
def test_gemv_family_exact(small, M, N, K):
    """x and W of -1, 0, 1: whole-number sums below 256, exact in fp32 in any order and in bf16, through
    the plain product, SiLU * up and the residual add + norm."""
    hip = small[1]
    g = torch.Generator().manual_seed(M * 7 + N)
    x = torch.randint(-1, 2, (M, K), generator=g).to(BF)
    w = torch.randint(-1, 2, (N, K), generator=g).to(BF)
    ref = x.float() @ w.float().t()
    assert ref.abs().max() < 256
    assert hip._gemv_ok(x.cuda(), w.cuda()) and not hip._linear_ok(x.cuda(), w.cuda())
    assert torch.equal(hip.linear(x.cuda(), w.cuda()).float().cpu(), ref)
    _epilogues_exact(hip, x, w, ref, g)


@pytest.mark.parametrize("M", [17, 64, 65, 300])
def test_linear_keeps_what_only_f_linear_takes(small, M):
    """Products above the GEMV's rows: mismatched shapes raise, an operand that needs a gradient gets it,
    an unaligned operand goes to F.linear, and products on two streams do not share a workspace."""
    hip = small[1]
    g = torch.Generator().manual_seed(M)
    x = torch.randint(-1, 2, (M, 192), generator=g).to(BF).cuda()
    w = torch.randint(-1, 2, (80, 192), generator=g).to(BF).cuda()
    ref = x.float() @ w.float().t()
    for rows in (1, 16, M):
        with pytest.raises(RuntimeError):
            hip.linear(x[:rows], w[:, :128].contiguous())
    wg = w.clone().requires_grad_()
    y = hip.linear(x, wg)
    assert torch.equal(y.float(), ref)
    y.backward(torch.ones_like(y))
    assert torch.equal(wg.grad[0].float(), x.float().sum(0).to(BF).float())
    odd = torch.empty(M * 192 + 1, dtype=BF, device="cuda")[1:].view(M, 192).copy_(x)
    assert odd.data_ptr() % 16 != 0 and not hip._linear_ok(odd, w) and not hip._gemm_ok(odd, w)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        z = hip.linear(x, w)
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(z.float(), ref) and torch.equal(hip.linear(x, w).float(), ref)
    if M > 64:
        a, b = (hip._gemm_workspace(x.device, s.cuda_stream) for s in (side, torch.cuda.current_stream()))
        assert a.data_ptr() != b.data_ptr()


def _epilogues_exact(hip, x, w, ref, g):
    """SiLU * up and the residual add + norm of a product whose values `ref` are whole numbers below 256."""
    M, N = ref.shape
    if N % 2 == 0:
        gu, up = ref.chunk(2, -1)
        want = (torch.nn.functional.silu(gu).to(BF).float() * up).to(BF).float()
        got = hip.gate_up_silu(x.cuda(), w.cuda()).cpu().float()
        # silu to one bf16 ulp (another expf): 2^-7 at most; one more from the rounding of the product
        assert ((got - want).abs() <= 2 ** -6 * want.abs() + 1e-30).all()
    if N <= 4096:
        h = torch.randint(-64, 65, (M, N), generator=g).to(BF)
        lnw = torch.ones(N, dtype=BF)
        hn, y = hip.linear_add_norm(x.cuda(), w.cuda(), h.cuda(), lnw.cuda())
        want = (h.float() + ref).to(BF).float()
        assert torch.equal(hn.float().cpu(), want)
        norm = want * torch.rsqrt(want.square().mean(-1, keepdim=True) + hip.e.eps)
        # one rounding of the fp32 norm to bf16 (half an ulp: 2^-9), doubled for its own fp32 sum
        assert ((y.float().cpu() - norm).abs() <= 2 ** -8 * norm.abs() + 1e-30).all()


# rows at the edges of the 16-row tiles; N and K at a ragged last tile, K split over workgroups (few outputs,
# many rows), every stage width, and on 256 CUs (plain, SiLU) tiles of 1 (72 .. 2560), 2 (6144), 4 (12008), 5
# (20002, 40000) and 8 weight tiles (65576; SiLU 24578)
@pytest.mark.parametrize("M", [1, 16, 17, 48, 64])
@pytest.mark.parametrize("N,K", [(72, 256), (1000, 192), (2560, 1024), (6144, 128), (12008, 64), (20002, 64), (24578, 64),
                                 (40000, 128), (65576, 64)])
def test_streamed_linear_exact(small, M, N, K):
    """x and W of -1, 0, 1: every product sum is a whole number of at most K <= 1024 with |sum| < 256
    (a random walk), exact in fp32 in any order and in bf16."""
    hip = small[1]
    g = torch.Generator().manual_seed(M * 7 + N)
    x = torch.randint(-1, 2, (M, K), generator=g).to(torch.bfloat16)
    w = torch.randint(-1, 2, (N, K), generator=g).to(torch.bfloat16)
    ref = x.float() @ w.float().t()
    assert ref.abs().max() < 256
    assert hip._linear_ok(x.cuda(), w.cuda())
    assert torch.equal(hip.linear(x.cuda(), w.cuda()).float().cpu(), ref)
    _epilogues_exact(hip, x, w, ref, g)


# above 64 rows: the edges of the 32-row steps and of the ranges of SiLU (96) and the sums (128), a ragged last
# tile, SiLU with 8 weight tiles (24578)
@pytest.mark.parametrize("M", [65, 80, 96, 97, 128, 129])
@pytest.mark.parametrize("N,K", [(72, 256), (1000, 192), (2560, 1024), (20002, 64), (24578, 64), (40000, 128)])
def test_streamed_epilogues_exact(small, M, N, K):
    """The products of test_streamed_linear_exact (whole numbers below 256) through the epilogues."""
    g = torch.Generator().manual_seed(M * 7 + N)
    x = torch.randint(-1, 2, (M, K), generator=g).to(BF)
    w = torch.randint(-1, 2, (N, K), generator=g).to(BF)
    ref = x.float() @ w.float().t()
    assert ref.abs().max() < 256
    _epilogues_exact(small[1], x, w, ref, g)


def test_linear_dtype_and_layout_fallback(small):
    """test_linear_precision.py:16-27: fp32/fp16/non-contiguous inputs route to F.linear."""
    _, hip, _ = small
    for dtype in (torch.float32, torch.float16):
        x = torch.randn(3, 8, dtype=dtype, device="cuda")
        w = torch.randn(8, 8, dtype=dtype, device="cuda")
        assert torch.equal(hip.linear(x, w), torch.nn.functional.linear(x, w))
    x = torch.randn(3, 8, dtype=BF, device="cuda")
    w = torch.randn(8, 8, dtype=BF, device="cuda").T
    assert not w.is_contiguous()
    assert torch.equal(hip.linear(x, w), torch.nn.functional.linear(x, w))


@pytest.mark.parametrize("M,N,K", [(256, 512, 256), (777, 2560, 1024), (2049, 1536, 512)])
def test_gemm_solutions_match_fp32(small, M, N, K):
    """Prefill-sized products (M >= GEMM_MIN_M) through dd_gemm_bf16: the heuristic's first
    candidate (solution -1) and every candidate dd_gemm_bf16_solutions lists, each within the
    bf16 bar of an fp32 product and each the same bits when called again; a solution index that
    names no hipBLASLt solution runs the heuristic's first candidate (same bits as -1);
    HipOps.linear (the committed table's pick) within the bar."""
    import ctypes
    from dryft_amd.hipops import GEMM_MIN_M
    _, hip, _ = small
    g = torch.Generator().manual_seed(M + N + K)
    x = (torch.randn(M, K, generator=g) * 0.5).to(BF)
    w = (torch.randn(N, K, generator=g) * 0.05).to(BF)
    ref = x.float() @ w.float().T
    xc, wc = x.cuda(), w.cuda()
    assert M >= GEMM_MIN_M
    ws = torch.empty(hip.L.dd_gemm_ws_bytes(), dtype=torch.uint8, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream

    def run(sol):
        y = torch.empty(M, N, dtype=BF, device="cuda")
        assert hip.L.dd_gemm_bf16(xc.data_ptr(), wc.data_ptr(), y.data_ptr(), M, N, K,
                                  ws.data_ptr(), ws.numel(), sol, stream) == 0
        return y

    first = run(-1)
    close(first, ref)
    assert torch.equal(run(-1), first)
    assert torch.equal(run(10 ** 9), first)          # no such solution: heuristic first
    buf = (ctypes.c_int * 16)()
    n = hip.L.dd_gemm_bf16_solutions(M, N, K, ws.numel(), buf, 16)
    assert 1 <= n <= 16
    for sol in list(buf[:n]):
        y = run(sol)
        close(y, ref)
        assert torch.equal(run(sol), y)
    close(hip.linear(xc, wc), ref)
    # argument validation: nothing runs, hipErrorInvalidValue
    y0 = torch.empty(M, N, dtype=BF, device="cuda")
    assert hip.L.dd_gemm_bf16(xc.data_ptr(), wc.data_ptr(), y0.data_ptr(), 0, N, K, ws.data_ptr(),
                              ws.numel(), -1, stream) == 1
    assert hip.L.dd_gemm_bf16_solutions(0, N, K, ws.numel(), buf, 16) == -1


# ------------------------------------------------------------------------ qkv_post decode
@pytest.mark.parametrize("B,S,posl", [(3, 1, [9, 9, 9]), (16, 1, list(range(0, 800, 50))),
                                      (4, 5, [0, 17, 300, 1000])])
def test_qkv_post_decode(cuda, B, S, posl):
    NH, NKV, HD, cap = 32, 8, 128, 2048
    e = fake_engine(nh=NH, nkv=NKV, hd=HD, rope_len=4096)
    tor, hip = TorchOps(e), _hip(e)
    g = torch.Generator().manual_seed(B * 10 + S)
    qkv = torch.randn(B * S, (NH + 2 * NKV) * HD, generator=g).to(BF)

    class L:
        qn = (1 + 0.02 * torch.randn(HD, generator=g)).to(BF)
        kn = (1 + 0.02 * torch.randn(HD, generator=g)).to(BF)

    class LG:
        qn = L.qn.cuda()
        kn = L.kn.cuda()
    kc0 = torch.randn(B, NKV, cap, HD, generator=g).to(BF)
    vc0 = torch.randn(B, NKV, cap, HD, generator=g).to(BF)
    pos = torch.tensor(posl)
    kc, vc = kc0.cuda(), vc0.cuda()
    q = hip.qkv_post(qkv.cuda(), LG, kc, vc, B, S, pos.cuda())
    G = NH // NKV
    qd = q.reshape(B, NKV, S, G, HD).cpu()
    # oracle: token (b, s) at position pos[b] + s, one at a time
    rk, rv = kc0.clone(), vc0.clone()
    rq = torch.empty(B, NKV, S, G, HD, dtype=BF)
    for b in range(B):
        for s in range(S):
            p = torch.tensor([posl[b] + s])
            qq = tor.qkv_post(qkv[b * S + s:b * S + s + 1], L, rk[b:b + 1], rv[b:b + 1], 1, 1, p)
            rq[b, :, s] = qq.reshape(NKV, G, HD)
    close(qd, rq)
    kcc, vcc = kc.cpu(), vc.cpu()
    assert torch.equal(vcc, rv)                       # V copy and every index: bit-exact
    written = torch.zeros(B, cap, dtype=torch.bool)
    for b in range(B):
        written[b, posl[b]:posl[b] + S] = True
    assert torch.equal(kcc.permute(0, 2, 1, 3)[~written], kc0.permute(0, 2, 1, 3)[~written])
    close(kcc, rk)
    nbits = (kcc != rk).sum().item()
    print(f"K cache bf16 elements differing from the oracle: {nbits} of {written.sum().item() * NKV * HD}")
    assert hip.err.item() == 0


# ------------------------------------------------------------------------ attention (test_attn.py cases)
ATTN_CASES = [(1, 1, 640, [512]), (1, 7, 640, [512]), (1, 7, 640, [0]), (2, 7, 384, [200, 11]),
              (3, 5, 2304, [2048, 900, 5]), (4, 4, 640, [512, 512, 300, 0]),
              (16, 1, 640, [512] * 16), (32, 1, 640, [512] * 32)]


@pytest.mark.parametrize("B,W,cap,posl", ATTN_CASES)
def test_attn_decode_cases(cuda, B, W, cap, posl):
    NH, NKV, HD = 32, 8, 128
    G = NH // NKV
    hip = _hip(fake_engine(nh=NH, nkv=NKV, hd=HD))
    g = torch.Generator().manual_seed(B * 100 + W)
    kc = torch.randn(B, NKV, cap, HD, generator=g).to(BF)
    vc = torch.randn(B, NKV, cap, HD, generator=g).to(BF)
    q = torch.randn(B, NKV, W, G, HD, generator=g).to(BF)
    pos = torch.tensor(posl if B > 1 else posl[:1])
    out = hip.attn_decode(q.cuda(), kc.cuda(), vc.cuda(), pos.cuda(), W).double().cpu()
    ref = attn_reference_fp64(q, kc, vc, pos, W, NH, NKV, HD)
    d = (out - ref).abs().max().item()
    assert d < 0.02, d


def test_attn_ragged_long_context(cuda):
    """B=16, ragged lengths U[512, 8192], cap 8192; also checks that a second call
    (counters left at zero by the last split) gives identical bits."""
    NH, NKV, HD, cap, B = 32, 8, 128, 8192, 16
    G = NH // NKV
    hip = _hip(fake_engine(nh=NH, nkv=NKV, hd=HD))
    g = torch.Generator().manual_seed(42)
    lens = torch.randint(512, 8193, (B,), generator=g)
    pos = lens - 1
    kc = torch.randn(B, NKV, cap, HD, generator=g).to(BF)
    vc = torch.randn(B, NKV, cap, HD, generator=g).to(BF)
    q = torch.randn(B, NKV, 1, G, HD, generator=g).to(BF)
    qg, kg, vg, pg = q.cuda(), kc.cuda(), vc.cuda(), pos.cuda()
    out = hip.attn_decode(qg, kg, vg, pg, 1)
    out2 = hip.attn_decode(qg, kg, vg, pg, 1)
    assert torch.equal(out, out2)
    ref = attn_reference_fp64(q, kc, vc, pos, 1, NH, NKV, HD)
    d = (out.double().cpu() - ref).abs().max().item()
    assert d < 0.02, d


# equal shares of the batch (W * G <= 4): contexts at the edges of the 32-key blocks, empty and full
# caches, pairs that lie in one wave, in several, in several workgroups, more pairs than workgroups,
# a capacity that is no multiple of the block, W = 2
@pytest.mark.parametrize("NH,NKV,W,cap,lens", [
    (32, 8, 1, 64, [1]), (32, 8, 1, 64, [64, 1, 33]), (32, 8, 1, 8192, [8192]), (32, 8, 1, 640, [577] * 33),
    (32, 8, 1, 4100, [4100, 1, 31, 32, 33, 4095, 64, 96]), (4, 4, 1, 200, [7 * i % 199 + 1 for i in range(130)]),
    (32, 8, 1, 330, [11 * i % 331 for i in range(1, 300)]),
    (8, 4, 2, 328, [2, 33, 328, 100, 257]), (12, 4, 1, 1000, [999, 3])])
def test_attn_equal_shares(cuda, NH, NKV, W, cap, lens):
    HD = 128
    hip = _hip(fake_engine(nh=NH, nkv=NKV, hd=HD))
    B, g = len(lens), torch.Generator().manual_seed(cap + len(lens))
    kc, vc = (torch.randn(B, NKV, cap, HD, generator=g).to(BF) for _ in range(2))
    q = torch.randn(B, NKV, W, NH // NKV, HD, generator=g).to(BF)
    pos = torch.tensor(lens) - W
    kg, vg = kc.cuda(), vc.cuda()
    for b, n in enumerate(lens):                            # the cache is zero past the last key
        kg[b, :, n:] = vg[b, :, n:] = 0
    args = q.cuda(), kg, vg, pos.cuda(), W
    out = hip.attn_decode(*args)
    assert torch.equal(out, hip.attn_decode(*args))         # same bits, counters left zero
    d = (out.double().cpu() - attn_reference_fp64(q, kc, vc, pos, W, NH, NKV, HD)).abs().max().item()
    assert d < 0.02, d


@pytest.mark.parametrize("lens", [[33, 64, 577, 1, 640], [8190]])
def test_attn_infinite_newest_value(cuda, lens):
    """An infinite value of the newest key makes that dim infinite, and nothing NaN: slots past it count
    as zeros, which they are."""
    NH, NKV, HD, cap, B = 32, 8, 128, max(lens) + 2, len(lens)
    hip = _hip(fake_engine(nh=NH, nkv=NKV, hd=HD))
    g = torch.Generator().manual_seed(B)
    kc, vc = (torch.randn(B, NKV, cap, HD, generator=g).to(BF) for _ in range(2))
    q = torch.randn(B, NKV, 1, NH // NKV, HD, generator=g).to(BF)
    for b, n in enumerate(lens):
        kc[b, :, n:] = vc[b, :, n:] = 0
        vc[b, :, n - 1, 5] = 0
    pos = torch.tensor(lens) - 1
    ref = attn_reference_fp64(q, kc, vc, pos, 1, NH, NKV, HD).view(B, NH, HD)
    for b, n in enumerate(lens):
        vc[b, :, n - 1, 5] = float("inf")
    out = hip.attn_decode(q.cuda(), kc.cuda(), vc.cuda(), pos.cuda()).double().cpu().view(B, NH, HD)
    assert (out[:, :, 5] == float("inf")).all()
    out[:, :, 5] = ref[:, :, 5]
    assert (out - ref).abs().max().item() < 0.02


@torch.inference_mode()
def test_attn_streams_and_graphs_at_once(cuda):
    """Short contexts that lie in several workgroups (65 keys in a 256-slot cache), eagerly on two streams
    and in two replayed graphs at the same time: every result has the bits of a call by itself."""
    NH, NKV, HD, cap, B = 32, 8, 128, 256, 3
    hip = _hip(fake_engine(nh=NH, nkv=NKV, hd=HD))
    g = torch.Generator().manual_seed(9)
    pos = torch.tensor([64, 127, 70]).cuda()
    sets = [[torch.randn(*s, generator=g).to(BF).cuda() for s in
             ((B, NKV, 1, NH // NKV, HD), (B, NKV, cap, HD), (B, NKV, cap, HD))] for _ in range(2)]
    alone = [hip.attn_decode(*t, pos) for t in sets]
    streams = [torch.cuda.Stream() for _ in sets]
    torch.cuda.synchronize()
    outs = [[], []]
    for _ in range(50):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                outs[i].append(hip.attn_decode(*sets[i], pos))
    torch.cuda.synchronize()
    for i in range(2):
        assert all(torch.equal(o, alone[i]) for o in outs[i])
    graphs = []
    for i, t in enumerate(sets):
        if i == 1:
            hip._spare.clear()                              # a graph that clears its own
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            graphs.append((graph, [hip.attn_decode(*t, pos) for _ in range(4)]))
    for _ in range(3):
        for _, out in graphs:
            for o in out:
                o.zero_()
        torch.cuda.synchronize()
        for s, (graph, _) in zip(streams, graphs):
            with torch.cuda.stream(s):
                graph.replay()
        torch.cuda.synchronize()
        for i, (_, out) in enumerate(graphs):
            assert all(torch.equal(o, alone[i]) for o in out)


def test_gemm_record_past_its_bound(cuda):
    """More shapes than the product's record holds (256), an older one in use all along, with no named
    solution, the table's, and one that the library does not know: exact products each time, and the same
    choice after a shape has been dropped and comes again."""
    hip = _hip(fake_engine(nh=8, nkv=2, hd=128))
    from dryft_amd.hipops import load_gemm_table
    sols = (-1, load_gemm_table()[2560, 4096][0][1], 1 << 30)
    g = torch.Generator().manual_seed(5)
    x = torch.randint(-1, 2, (400, 64), generator=g).to(BF).cuda()
    w = torch.randint(-1, 2, (48, 64), generator=g).to(BF).cuda()
    ref = (x.float() @ w.float().t()).to(BF)                # |sum| <= 64: exact in bf16
    for M in (*range(65, 345), 66, 200):
        assert torch.equal(hip._gemm_lib(x[:M], w, sols[M % 3]), ref[:M]), M
        assert torch.equal(hip._gemm_lib(x[:65], w, sols[M % 3]), ref[:65]), M


# ------------------------------------------------------------------------ argmax
def test_argmax_rules_and_pos(cuda):
    from dryft_amd.hipops import HipOps
    hip = _hip(fake_engine(nh=8, nkv=2, hd=128))
    lg = torch.tensor([[1.0, 3.0, 3.0, -1.0, 0.5], [0.0, 2.0, float("nan"), 5.0, float("nan")],
                       [-1.0, -1.0, -1.0, -1.0, -1.0]], dtype=BF).cuda()
    tok = torch.zeros(3, dtype=torch.long, device="cuda")
    pos = torch.tensor([4, 7, 9], device="cuda")
    hip.argmax_(lg, tok, pos)
    assert tok.tolist() == lg.cpu().argmax(-1).tolist() == [1, 2, 0]
    assert pos.tolist() == [5, 8, 10]
    g = torch.Generator().manual_seed(5)
    big = torch.randn(16, 151936, generator=g).to(BF)
    big[3, 100] = big[3, 200] = big[3].max() + 1          # a tie: first index wins
    tok = torch.zeros(16, dtype=torch.long, device="cuda")
    hip.argmax_(big.cuda(), tok)
    assert tok.cpu().tolist() == big.argmax(-1).tolist()
    assert isinstance(hip, HipOps)
