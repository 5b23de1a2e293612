"""GPU parity of the HIP kernels against the CPU oracle (bit-exact exponents and
payloads) and against fp64 (outputs, with the tolerance the north star states:
relative Frobenius error <= 2e-3 and no worse than the reference's own error,
which the oracle emulates)."""
import ctypes

import math

import numpy as np
import pytest
import torch

import workloads as W
from oracle import tbf16_oracle as O
from tbf16 import _ext, attention, autograd, ops
import tbf16

from _ref64 import attn_fwd64, rel

pytestmark = pytest.mark.gpu

TOL = 2e-3
# slack on "no worse than the reference's own error": accumulation order differs
REF_SLACK = 1.02


def bf16_from_bits(bits: np.ndarray) -> torch.Tensor:
    return torch.from_numpy(bits.astype(np.uint16).view(np.int16)).view(torch.bfloat16)


def f16_bits(t: torch.Tensor) -> np.ndarray:
    return t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.uint16)


def row_exps_gpu(x: torch.Tensor, t: int, l1: bool) -> np.ndarray:
    M, K = x.shape
    e = torch.empty(M, dtype=torch.int32, device=x.device)
    _ext.call("tbf16_row_exps", x.data_ptr(), M, K, x.stride(0), t, int(l1), e.data_ptr(), None, _ext.stream())
    return e.cpu().numpy()


def linear_ws(M, K, N, cfg, dev):
    """tbf16_linear's workspace (bytes) and the int32 view of its row exponents."""
    b = int(_ext.lib().tbf16_linear_ws_bytes(M, K, N, cfg))
    w = torch.full((b,), 0xAB, dtype=torch.uint8, device=dev)
    return w, w[: 4 * M].view(torch.int32)


def test_native_library_is_the_one_loaded(dev):
    assert _ext.available()
    p = _ext.lib_path()
    assert p.name == "libtbf16_hip.so" and "turing-bf16_amd" in str(p)
    assert tbf16.is_supported_gpu()


# ---- exponents and payloads, exhaustive over bf16 ---------------------------------

@pytest.mark.parametrize("t", [-1, 0, 15])
def test_row_exps_every_bf16_amax(dev, t):
    """Each row holds one bf16 pattern (and zeros): its max is that pattern.
    All 32,640 finite non-negative patterns plus +inf, both signs."""
    bits = np.arange(0, 0x7F81, dtype=np.uint32)  # 0 .. +inf
    x = torch.zeros(2 * len(bits), 8, dtype=torch.bfloat16)
    x[: len(bits), 3] = bf16_from_bits(bits)
    x[len(bits):, 5] = bf16_from_bits(bits | 0x8000)
    xd = x.to(dev)
    got = row_exps_gpu(xd, t, False)
    want = O.row_exps(x, t)
    assert np.array_equal(got, want)
    # the L1 variant on the same rows (sum of one value = the value)
    assert np.array_equal(row_exps_gpu(xd, t, True), O.row_exps(x, t, l1=True))


@pytest.mark.parametrize("t,l1", [(15, False), (0, False), (15, True), (-1, False)])
def test_quantize_rows_payload_every_bf16(dev, t, l1):
    """All 65,536 bf16 patterns as payload, with row maxima spread over 2^0..2^40 so
    scaled values fall into fp16's subnormal range (RNE there)."""
    bits = np.arange(0, 1 << 16, dtype=np.uint32)
    x = bf16_from_bits(bits).reshape(512, 128).clone()
    x = torch.where(torch.isnan(x), torch.zeros_like(x), x)
    g = torch.Generator().manual_seed(1)
    x[:, 0] = torch.ldexp(torch.ones(512), torch.randint(0, 41, (512,), generator=g).float()).bfloat16()
    y, s = ops.quantize_rows(x.to(dev), t, l1)
    y_o, s_o = O.quantize_rows(x, t, l1)
    assert np.array_equal(f16_bits(y), f16_bits(y_o))
    assert torch.equal(s.cpu(), s_o)


def test_quantize_rows_t_and_cols_t_bit_exact(dev):
    g = torch.Generator().manual_seed(2)
    x = (torch.randn(203, 264, generator=g) * torch.exp2(torch.randint(-30, 30, (203, 1), generator=g).float()))
    x = x.bfloat16()
    xd = x.to(dev)
    x16T, sx, exps = autograd._quantize_rows_t(xd, 0)
    y_o, s_o = O.quantize_rows(x, 0)
    assert x16T.shape == (264, 208)
    assert np.array_equal(f16_bits(x16T[:, :203].t()), f16_bits(y_o))
    assert (x16T[:, 203:] == 0).all()
    assert torch.equal(sx.cpu(), s_o)
    assert np.array_equal(exps.cpu().numpy(), O.row_exps(x, 0))
    rm = torch.ldexp(torch.ones(203), torch.randint(-9, 9, (203,), generator=g).float())
    for t, r in ((0, None), (-2, rm)):
        yc, sc = tbf16.autograd.quantize_cols(xd, t, None if r is None else r.to(dev))
        yo, so = O.quantize_cols(x, t, r)
        assert np.array_equal(f16_bits(yc), f16_bits(yo)) and torch.equal(sc.cpu(), so)


# ---- MFMA layout and epilogue: exact small-integer GEMMs -------------------------

# tiled configurations take any M; skinny ones (5-8, 13, 14) M <= 32 or 64; the
# decode ones (15-18, fp16 a) any M, in row tiles of 32 / 64 / 128 / 256
GEMM_CFG_M = {0: 300, 1: 300, 2: 300, 3: 300, 4: 300, 5: 29, 6: 29, 7: 61, 8: 61, 9: 300, 10: 300, 11: 300, 12: 300, 19: 300,
              13: 29, 14: 61, 15: 300, 16: 300, 17: 300, 18: 300}
STREAM_CFGS = (15, 16, 17, 18)


@pytest.mark.parametrize("K", [200, 1000, 3040])
@pytest.mark.parametrize("cfg", sorted(GEMM_CFG_M))
def test_gemm_small_integers_bit_exact(dev, cfg, K):
    """Entries in {-1, 0, 1}: every partial sum is an integer of at most K, so the
    fp32 accumulation is exact and the bf16 output must equal the integer product
    rounded once, bit for bit. Ragged M, N, K exercise every tile edge (and, for
    the skinny kernel, a K chunk that runs past K); K = 1000 (16 k tiles) and
    K = 3040 (48 chunks of 64, the last one partial) also run the steady-state
    loops, whose register sets must never carry the partial last chunk unmasked
    (K = 3040 puts it right at the steady-state bound of every skinny depth);
    K = 200 runs only the tails; pow2 scales and an integer bias exercise the
    epilogue."""
    g = torch.Generator().manual_seed(3)
    M, N = GEMM_CFG_M[cfg], 264
    a = torch.randint(-1, 2, (M, K), generator=g)
    b = torch.randint(-1, 2, (N, K), generator=g)
    bias = torch.randint(-8, 9, (N,), generator=g)
    sa = torch.ldexp(torch.ones(M), torch.randint(-3, 4, (M,), generator=g).float())
    sb = torch.ldexp(torch.ones(N), torch.randint(-3, 4, (N,), generator=g).float())
    want = ((a @ b.t()).double() * sa.double()[:, None] * sb.double()[None, :] + bias.double()).bfloat16()
    y = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
    a16, b16 = a.half().to(dev), b.half().to(dev)
    sad, sbd, bd = sa.to(dev), sb.to(dev), bias.bfloat16().to(dev)
    _ext.call("tbf16_gemm_f16", a16.data_ptr(), M, K, K, sad.data_ptr(), b16.data_ptr(), N, K, sbd.data_ptr(),
              bd.data_ptr(), y.data_ptr(), N, cfg, _ext.stream())
    assert torch.equal(y.cpu(), want)
    # bf16 activations through the fused path (the decode configurations: through the
    # workspace's fp16 copy): row max 1 -> scale 2^14, exact
    xb = a.bfloat16().to(dev)
    work, e = linear_ws(M, K, N, cfg, dev)
    ones = torch.ones(N, device=dev)
    _ext.call("tbf16_linear", xb.data_ptr(), M, K, K, b16.data_ptr(), N, K, ones.data_ptr(), None, y.data_ptr(), N, 15,
              0, cfg, work.data_ptr(), _ext.stream())
    assert torch.equal(y.cpu(), (a @ b.t()).double().bfloat16())
    assert np.array_equal(e.cpu().numpy(), O.row_exps(a.bfloat16(), 15))


@pytest.mark.parametrize("K", [8, 64, 128, 200, 1000, 3040])
@pytest.mark.parametrize("cfg", range(20, 31))
def test_gemm_pingpong_small_integers_bit_exact(dev, cfg, K):
    """The ping-pong configurations as above: exact integer products at one k tile (whole
    and partial), two, an odd and an even number of tiles with a partial last one (the
    group without a last tile reads zeros); rows and columns past whole tiles, and one
    row of tiles against few columns (fewer columns per block than the tile has)."""
    g = torch.Generator().manual_seed(11)
    for M, N in ((523, 264), (29, 1032), (1, 8)):
        a = torch.randint(-1, 2, (M, K), generator=g)
        b = torch.randint(-1, 2, (N, K), generator=g)
        bias = torch.randint(-8, 9, (N,), generator=g)
        sa = torch.ldexp(torch.ones(M), torch.randint(-3, 4, (M,), generator=g).float())
        sb = torch.ldexp(torch.ones(N), torch.randint(-3, 4, (N,), generator=g).float())
        want = ((a @ b.t()).double() * sa.double()[:, None] * sb.double()[None, :] + bias.double()).bfloat16()
        a16, b16, sad, sbd, bd = (t.to(dev) for t in (a.half(), b.half(), sa, sb, bias.bfloat16()))
        y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=dev)
        _ext.call("tbf16_gemm_f16", a16.data_ptr(), M, K, K, sad.data_ptr(), b16.data_ptr(), N, K, sbd.data_ptr(),
                  bd.data_ptr(), y.data_ptr(), N, cfg, _ext.stream())
        assert torch.equal(y.cpu(), want), (M, N)


@pytest.mark.parametrize("M,N,K", [(2, 8, 1000), (64, 256, 8200), (130, 72, 4096), (260, 8, 30000), (2, 264, 130000),
                                   (72, 264, 98312)])
def test_linear_dispatch_splits_bit_exact(dev, M, N, K):
    """The dispatcher's own choice where few tiles meet a long K (2, 4 or 8 splits, a K
    tail in the last one) and where x16 would not fit the no-allocation array (kernels
    that add over k in order): exact products, so any order gives the same bits; the
    no-allocation entry point gives them too."""
    g = torch.Generator().manual_seed(12)
    a, b = torch.randint(-1, 2, (M, K), generator=g), torch.randint(-1, 2, (N, K), generator=g)
    xb, b16, ones = a.bfloat16().to(dev), b.half().to(dev), torch.ones(N, device=dev)
    want = (a @ b.t()).double().bfloat16()
    work, _ = linear_ws(M, K, N, -1, dev)
    for name, tail in (("tbf16_linear", (work.data_ptr(), _ext.stream())), ("tbf16_linear_noalloc", (_ext.stream(),))):
        y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=dev)
        _ext.call(name, xb.data_ptr(), M, K, K, b16.data_ptr(), N, K, ones.data_ptr(), None, y.data_ptr(), N, 15, 0, -1,
                  *tail)
        assert torch.equal(y.cpu(), want), name


@pytest.mark.parametrize("M,K,N", [(17, 6528, 832), (32, 4104, 264), (33, 6528, 832), (2048, 3200, 640), (1999, 3400, 520),
                                   (640, 16384, 512), (16, 1000, 9000), (31, 1544, 8192), (32, 512, 8),
                                   (33, 256, 72), (64, 328, 264), (64, 256, 10248), (300, 320, 1032), (4100, 768, 136),
                                   (16390, 1032, 40)])
def test_linear_dispatch_few_rows_and_row_chunks(dev, M, K, N):
    """At most 32 rows whose tiles would split K (converted in the skinny kernel) and 33; a
    short K, or few columns for many rows (converted in the tiles); x16 beyond the no-allocation array, which that entry point then takes in chunks of
    rows (the last one short): exact products, and the same bits from both entry points."""
    g = torch.Generator().manual_seed(M)
    a, b = torch.randint(-1, 2, (M, K), generator=g), torch.randint(-1, 2, (N, K), generator=g)
    ones = torch.ones(N, device=dev)
    b16 = b.half().to(dev)
    work, _ = linear_ws(M, K, N, -1, dev)
    for x, exact in ((a.bfloat16().to(dev), True), (torch.randn(M, K, generator=g).bfloat16().to(dev), False)):
        ys = []
        for name, tail in (("tbf16_linear", (work.data_ptr(), _ext.stream())), ("tbf16_linear_noalloc", (_ext.stream(),))):
            y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=dev)
            _ext.call(name, x.data_ptr(), M, K, K, b16.data_ptr(), N, K, ones.data_ptr(), None, y.data_ptr(), N, 15, 0, -1,
                      *tail)
            ys.append(y.cpu())
        assert torch.equal(ys[0], ys[1])
        if exact:
            assert torch.equal(ys[0], (a.double() @ b.double().t()).bfloat16())


@pytest.mark.parametrize("N", [50, 64])
def test_linear_q_many_rows(dev, N):
    """More rows than 65535 of the tiles that a few columns would get otherwise (128 x 64): a
    taller tile takes them. Exact products."""
    M, K = 65536 * 128 + 5, 8
    g = torch.Generator(device=dev).manual_seed(N)
    a, b = (torch.randint(-4, 5, (r, K), generator=g, device=dev).half() for r in (M, N))
    y = ops.linear_q(a, torch.ones(M, device=dev), b, torch.ones(N, device=dev))
    assert y.shape == (M, N)
    for m in range(0, M, 1 << 21):
        assert torch.equal(y[m:m + (1 << 21)], (a[m:m + (1 << 21)].float() @ b.float().t()).bfloat16()), m


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("M,N,K", [(2, 1, 64), (17, 9, 4096), (100, 515, 200), (300, 2049, 520), (64, 32001, 64), (2, 257, 16392)])
def test_linear_any_n(dev, M, N, K, bias):
    """N that is no multiple of 8 without padding the weight, scale and bias views that
    start at any element, split and unsplit: exact products, and the same from
    already-quantised rows."""
    g = torch.Generator().manual_seed(N)
    a, b = torch.randint(-1, 2, (M, K), generator=g), torch.randint(-1, 2, (N, K), generator=g)
    sw = torch.ldexp(torch.ones(N + 1), torch.randint(-3, 4, (N + 1,), generator=g).float())[1:]
    bb = torch.randint(-8, 9, (N + 1,), generator=g).bfloat16()[1:] if bias else None
    want = (a @ b.t()).double() * sw.double() + (bb.double() if bias else 0.0)
    wide = lambda t: torch.cat([t[:1], t]).to(dev)[1:]  # noqa: E731  (a view one element into its storage)
    args = (b.half().to(dev), wide(sw), wide(bb) if bias else None)
    y = tbf16.scaled_linear(a.bfloat16().to(dev), *args)
    assert y.shape == (M, N) and torch.equal(y.cpu(), want.bfloat16())
    y = ops.linear_q(a.half().to(dev), torch.ones(M, device=dev), *args)
    assert y.shape == (M, N) and torch.equal(y.cpu(), want.bfloat16())


@pytest.mark.parametrize("M,N,K", [(256, 4096, 4096), (200, 768, 2560), (300, 264, 3040)])
def test_linear_split_k(dev, M, N, K):
    """K split over two blocks per tile (what tbf16_linear picks where the tiles leave
    half of the CUs idle: configs[0]'s shape, a ragged M and N, a K tail in the second
    half). Integer-valued products are exact in any summation order, so with an
    integer bias the output equals the integer product rounded once, bit for bit;
    on random rows the output stays within the fp64 bound."""
    assert int(_ext.lib().tbf16_linear_ws_bytes(M, K, N, -1)) >= 2 * M * N * 4  # the split's partial sums
    g = torch.Generator().manual_seed(7)
    a = torch.randint(-1, 2, (M, K), generator=g)
    b = torch.randint(-1, 2, (N, K), generator=g)
    bias = torch.randint(-8, 9, (N,), generator=g)
    w16, wsv = ops.prepare_weight(b.bfloat16().to(dev))
    y = ops.scaled_linear(a.bfloat16().to(dev), w16, wsv, bias.bfloat16().to(dev))
    assert torch.equal(y.cpu(), ((a @ b.t()).double() + bias.double()).bfloat16())
    x = torch.randn(M, K, generator=g).bfloat16()
    w = (torch.randn(N, K, generator=g) * 0.02).bfloat16()
    w16, wsv = ops.prepare_weight(w.to(dev))
    y = ops.scaled_linear(x.to(dev), w16, wsv)
    assert rel(y.cpu(), x.double() @ w.double().t()) <= TOL


def test_gemv_small_integers_bit_exact(dev):
    g = torch.Generator().manual_seed(4)
    K, N = 2560, 1000
    x = torch.randint(-1, 2, (1, K), generator=g).float()
    x[0, 200:] = 0  # keep |sum| < 256
    w = torch.randint(-1, 2, (N, K), generator=g).float()
    ws = torch.ldexp(torch.ones(N), torch.randint(-2, 3, (N,), generator=g).float())
    y = ops.small_m_linear(x.bfloat16().to(dev), w.half().to(dev), ws.to(dev))
    assert torch.equal(y.cpu(), ((x @ w.t()) * ws).bfloat16())


# ---- Config 1: CPU-path linear (256 x 4096 x 4096, 5 % rows x 2^17) --------------

def _linear_checks(x, w, dev, label):
    w16, ws = tbf16.prepare_weight(w.to(dev))
    w16_o, ws_o = O.prepare_weight(w)
    assert np.array_equal(f16_bits(w16), f16_bits(w16_o)), f"{label}: weight payload"
    assert torch.equal(ws.cpu(), ws_o), f"{label}: weight exponents"
    xd = x.to(dev)
    M = x.shape[0]
    y = tbf16.scaled_linear(xd, w16, ws)
    ref = xd.double() @ w.to(dev).double().t()
    err = rel(y, ref)
    if M == 1:
        own = O.gemv(x, w16_o, ws_o)
    elif M >= O.FUSED_MIN_M:
        t, l1 = 15, False
        assert np.array_equal(row_exps_gpu(xd, t, l1), O.row_exps(x, t, l1, fused=True)), f"{label}: x exponents"
        own = O.linear_fused(x, w16_o, ws_o)
    else:
        assert np.array_equal(row_exps_gpu(xd, 15, True), O.row_exps(x, 15, True)), f"{label}: x L1 exponents"
        own = O.linear_cublas_path(x, w16_o, ws_o)
    err_own = rel(own.to(dev), ref)
    print(f"{label}: rel err {err:.3e}  reference's own {err_own:.3e}")
    assert torch.isfinite(y).all()
    assert err <= TOL, (label, err)
    assert err <= err_own * REF_SLACK + 1e-6, (label, err, err_own)
    return err


def test_cfg1_cpu_path_linear(dev):
    x, w, _ = W.cfg1_cpu_linear()
    _linear_checks(x, w, dev, "cfg1 256x4096x4096")


def test_cfg2_square_gemm(dev):
    x, w, _ = W.cfg2_square_gemm()
    _linear_checks(x, w, dev, "cfg2 4096^3")


@pytest.mark.parametrize("M", W.CFG3_MS)
def test_cfg3_small_m(dev, M):
    w, xs = W.cfg3_small_m()
    _linear_checks(xs[M], w, dev, f"cfg3 M={M}")


@pytest.mark.parametrize("cfg,M", [(-1, 29), (-1, 61), (-1, 128), (-1, 255), (5, 29), (6, 29), (7, 61), (13, 29),
                                   (15, 29), (16, 61), (17, 100), (18, 255)])
@pytest.mark.parametrize("l1", [0, 1])
def test_decode_row_exponents_and_output(dev, cfg, M, l1):
    """Decode-sized tbf16_linear on the skinny and decode configurations and on the
    dispatcher's own choice: the row exponents it leaves in the caller's workspace
    equal the oracle's bit for bit (max and L1 rows, K not a multiple of 64, rows
    spanning 2^-30 .. 2^30, a zero row), and the output equals the same kernel run
    on those exponents (tbf16_linear_exps), or for the configurations that take fp16
    a, on quantize_rows' fp16 copy (tbf16_gemm_f16)."""
    g = torch.Generator().manual_seed(7 + l1 + M)
    N, K = 10240 if cfg in (-1, 18) else 264, 2504
    x = (torch.randn(M, K, generator=g) * torch.ldexp(torch.ones(M, 1), torch.randint(-30, 31, (M, 1), generator=g))
         ).bfloat16()
    x[3] = 0.0
    w = (torch.randn(N, K, generator=g) * 0.02).bfloat16()
    xd, wd = x.to(dev), w.to(dev)
    w16, ws = ops.prepare_weight(wd)
    y = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
    work, e = linear_ws(M, K, N, cfg, dev)
    e.fill_(-999)
    _ext.call("tbf16_linear", xd.data_ptr(), M, K, K, w16.data_ptr(), N, K, ws.data_ptr(), None, y.data_ptr(), N, 15,
              l1, cfg, work.data_ptr(), _ext.stream())
    torch.cuda.synchronize()
    assert np.array_equal(e.cpu().numpy(), O.row_exps(x, 15, bool(l1)))
    y2 = torch.empty_like(y)
    L = _ext.lib()
    # a configuration that takes fp16 a needs a larger workspace than skinny cfg 13
    if cfg in STREAM_CFGS or L.tbf16_linear_ws_bytes(M, K, N, cfg) != L.tbf16_linear_ws_bytes(M, K, N, 13):
        x16, sx = ops.quantize_rows(xd, 15, bool(l1))
        _ext.call("tbf16_gemm_f16", x16.data_ptr(), M, K, K, sx.data_ptr(), w16.data_ptr(), N, K, ws.data_ptr(),
                  None, y2.data_ptr(), N, cfg, _ext.stream())
    else:
        _ext.call("tbf16_linear_exps", xd.data_ptr(), M, K, K, e.data_ptr(), w16.data_ptr(), N, K, ws.data_ptr(),
                  None, y2.data_ptr(), N, cfg, _ext.stream())
    assert torch.equal(y, y2)
    ref = (x.double() @ (w16.cpu().double() * ws.cpu().double()[:, None]).t())
    assert rel(y.cpu(), ref) < TOL


# ---- Config 4: scaled attention forward ------------------------------------------

def _attn_checks(q, k, v, dev, rows=None, label=""):
    qd, kd, vd = q.to(dev), k.to(dev), v.to(dev)
    o, _, _, exps = attention.attn_forward(qd, kd, vd, None, True, None, v_exp=13)
    a_o, ev_o = O.attn_exponents(q, k, v, 13)
    ex = exps.cpu()
    assert int(ex[0]) == a_o, f"{label}: a"
    assert torch.equal(ex[2:].reshape(ev_o.shape), ev_o.int()), f"{label}: ev"
    ref = attn_fwd64(qd, kd, vd, True, rows=rows)
    got = o if rows is None else o[:, :, torch.as_tensor(rows, device=dev)]
    err = rel(got, ref)
    # the reference's own arithmetic (fp16 P, O / l rounded to fp16, then bf16),
    # emulated by the oracle on the same inputs and rows
    own = O.sdpa_reference_arith(qd, kd, vd, causal=True, v_exp=13, rows=rows)
    err_own = rel(own, ref)
    print(f"{label}: rel err {err:.3e}  reference's own {err_own:.3e}")
    assert torch.isfinite(got).all()
    assert err <= TOL, (label, err)
    assert err <= err_own * REF_SLACK + 1e-6, (label, err, err_own)
    return err, err_own


def test_cfg4_attention_4k(dev):
    q, k, v = W.cfg4_attention(4096)
    _attn_checks(q, k, v, dev, label="cfg4 S=4096")


@pytest.mark.parametrize("kform", ["bf16", "fp16"])
@pytest.mark.parametrize("split", ["0", "1"])
@pytest.mark.parametrize("B,H,S,D,layout", [(1, 3, 200, 128, "bhsd"), (2, 2, 328, 64, "bshd"),
                                            (1, 4, 1000, 128, "bshd"), (1, 2, 33, 64, "bhsd"),
                                            (2, 4, 2048, 128, "bhsd")])
def test_attention_causal_block_forms(dev, monkeypatch, B, H, S, D, layout, split, kform):
    """The causal forward's block forms on ragged lengths: split-key 8-wave blocks
    (waves w and w + 4 share 32 query rows and take alternate key tiles, merged
    through LDS) and the plain blocks, with the heavy/light pairing where the grid
    is small; S^T = K Q^T on the raw bf16 rows of q and k (bf16 MFMA, K tiles copied
    from k itself, also through (B, S, H, D) strides with a key tail) and on the
    fp16 k16 copy. Exponents bit-exact, output against fp64 and the reference's
    own error."""
    monkeypatch.setenv("TBF16_ATTN_SPLIT", split)
    if kform == "fp16":
        monkeypatch.setenv("TBF16_ATTN_KF16", "1")
    else:
        monkeypatch.delenv("TBF16_ATTN_KF16", raising=False)
    g = torch.Generator().manual_seed(S + D)
    shape = (B, H, S, D) if layout == "bhsd" else (B, S, H, D)
    q, k, v = ((torch.randn(*shape, generator=g) * m).bfloat16() for m in (8, 2, 300))
    if layout == "bshd":  # permuted views: row stride H * D
        q, k, v = (t.transpose(1, 2) for t in (q, k, v))
    _attn_checks(q, k, v, dev, label=f"split={split} k={kform} {layout} B={B} H={H} S={S} D={D}")


@pytest.mark.parametrize("H,S,D", [(1, 129, 128), (150, 200, 64), (170, 200, 64), (170, 300, 128), (280, 200, 64), (390, 200, 64),
                                   (3, 130, 192), (5, 577, 256)])
def test_attention_causal_grids(dev, H, S, D):
    """The causal grids on both sides of each line: single split-key tiles, pairs in one
    round, single tiles where the pairs are just more than a round, 256-row blocks."""
    g = torch.Generator().manual_seed(H)
    q, k, v = (torch.randn(1, H, S, D, generator=g).bfloat16() for _ in range(3))
    _attn_checks(q, k, v, dev, label=f"H={H} S={S} D={D}")


@pytest.mark.parametrize("split", ["0", "1"])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("Sq,Sk,D", [(33, 65, 64), (130, 257, 128), (200, 127, 96), (257, 64, 64), (16, 3, 128)])
def test_attention_bias_forms(dev, monkeypatch, Sq, Sk, D, causal, split):
    """Bias rows read four keys at a time at any alignment (odd row strides and a
    broadcast padding row), with whole and cut key tiles, in plain and split-key blocks
    (with fewer key tiles than groups too): within the bound of the unbiased forms of
    fp64 softmax(q k^T scale + bias) v."""
    monkeypatch.setenv("TBF16_ATTN_SPLIT", split)
    g = torch.Generator().manual_seed(Sq + Sk)
    q = torch.randn(2, 3, Sq, D, generator=g).bfloat16()
    k, v = (torch.randn(2, 3, Sk, D, generator=g).bfloat16() for _ in range(2))
    rows = torch.randn(2, 3, Sq, Sk, generator=g).half()
    pad = torch.arange(Sk).view(1, 1, 1, Sk) < torch.tensor([Sk, (Sk + 2) // 2]).view(2, 1, 1, 1)
    for mask in (rows, pad):
        got = tbf16.sdpa(q.to(dev), k.to(dev), v.to(dev), attn_mask=mask.to(dev), is_causal=causal)
        s = q.double() @ k.double().transpose(-1, -2) * D ** -0.5
        s = s + mask.double() if mask.dtype == torch.float16 else s.masked_fill(~mask, -math.inf)
        if causal:
            s = s.masked_fill(torch.ones(Sq, Sk, dtype=torch.bool).triu(1), -math.inf)
        assert rel(got.cpu(), torch.softmax(s, -1) @ v.double()) < TOL


@pytest.mark.parametrize("B,H,Sq,Sk,D", [(1, 8, 100, 64, 64), (1, 8, 200, 512, 128), (1, 8, 200, 513, 128),
                                         (2, 4, 130, 256, 64), (2, 4, 130, 257, 64), (9, 16, 128, 128, 64),
                                         (9, 16, 129, 70, 128), (33, 8, 33, 33, 64), (1, 3, 7, 1, 128)])
def test_attention_block_forms_of_short_calls(dev, B, H, Sq, Sk, D):
    """Few keys or few queries on both sides of the lines between 4-wave blocks, split-key
    blocks and 256-row blocks, with and without bias rows: fp64 softmax(q k^T scale + bias) v
    within the bound of the other forms."""
    g = torch.Generator().manual_seed(Sq + Sk)
    q = torch.randn(B, H, Sq, D, generator=g).bfloat16().to(dev)
    k, v = (torch.randn(B, H, Sk, D, generator=g).bfloat16().to(dev) for _ in range(2))
    s = (q.double() @ k.double().transpose(-1, -2).contiguous()) * D ** -0.5
    bias = torch.randn(B, 1, 1, Sk, generator=g).half().to(dev)
    tri = torch.ones(Sq, Sk, dtype=torch.bool, device=dev).triu(1)
    for mask, causal, ref in ((None, False, s), (bias, False, s + bias.double()), (None, True, s.masked_fill(tri, -math.inf))):
        got = tbf16.sdpa(q, k, v, attn_mask=mask, is_causal=causal)
        assert rel(got, torch.softmax(ref, -1) @ v.double()) < TOL


@pytest.mark.parametrize("split", ["0", "1"])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("D", [64, 128, 192])
def test_attention_running_maximum(dev, monkeypatch, D, causal, split):
    """The running maximum of a row: key tiles in which it sees no key before the first one
    that it sees (rows 0-15 and 16-31 of a wave's block at different tiles), rows that see
    none, and maxima that grow tile by tile by more and by less than the lazy bound, in
    only one of the two blocks or in both."""
    monkeypatch.setenv("TBF16_ATTN_SPLIT", split)
    g = torch.Generator().manual_seed(D)
    S = 330
    q, k, v = (torch.randn(1, 2, S, D, generator=g).bfloat16() for _ in range(3))
    row, key = torch.arange(S).view(S, 1), torch.arange(S).view(1, S)
    first = torch.where(row % 32 < 16, 70, 135) * (row // 32 % 2)  # every other wave block: keys from 70 / 135 on
    mask = (key >= first).expand(1, 1, S, S).clone()
    mask[..., 37, :] = False
    mask[..., 300:, :] = False
    grow = torch.where(row % 32 < 16, 4.0, 24.0) * (key // 64)     # in logits; the bound is 8 ln 2
    for m in (mask, mask & (key < 200), grow.half().expand(1, 1, S, S)):
        got = tbf16.sdpa(q.to(dev), k.to(dev), v.to(dev), attn_mask=m.to(dev), is_causal=causal)
        s = q.double() @ k.double().transpose(-1, -2) * D ** -0.5
        s = s + m.double() if m.dtype == torch.float16 else s.masked_fill(~m, -math.inf)
        if causal:
            s = s.masked_fill(key > row, -math.inf)
        want = torch.nan_to_num(torch.softmax(s, -1)) @ v.double()  # rows that see no key: zeros
        assert torch.isfinite(got).all() and rel(got.cpu(), want) < TOL


@pytest.mark.parametrize("kform", ["bf16", "fp16"])
@pytest.mark.parametrize("causal", [True, False])
def test_sdpa_gqa_key_forms(dev, monkeypatch, causal, kform):
    """Grouped-query attention (8 query heads on 2 key/value heads, a key tail)
    through tbf16.sdpa with K read as bf16 rows or as the fp16 k16 copy: within the
    fp64 bar, and the two forms within each other's rounding."""
    if kform == "fp16":
        monkeypatch.setenv("TBF16_ATTN_KF16", "1")
    else:
        monkeypatch.delenv("TBF16_ATTN_KF16", raising=False)
    g = torch.Generator().manual_seed(91)
    q = (torch.randn(2, 8, 333, 128, generator=g) * 6).bfloat16().to(dev)
    k = (torch.randn(2, 2, 333, 128, generator=g) * 3).bfloat16().to(dev)
    v = (torch.randn(2, 2, 333, 128, generator=g) * 50).bfloat16().to(dev)
    o = tbf16.sdpa(q, k, v, is_causal=causal, enable_gqa=True)
    assert rel(o, attn_fwd64(q, k, v, causal)) <= TOL


@pytest.mark.parametrize("causal", [True, False])
def test_sdpa_without_exponents_output(dev, causal):
    """tbf16.sdpa asks for no exponents: with bf16 K rows only V's maxima are taken.
    Its output equals attn_forward's with the exponents requested (same kernels,
    same V scale) and meets the fp64 bar."""
    g = torch.Generator().manual_seed(77)
    q, k, v = ((torch.randn(1, 4, 700, 128, generator=g) * m).bfloat16().to(dev) for m in (16, 4, 1e3))
    o = tbf16.sdpa(q, k, v, is_causal=causal)
    o2 = attention.attn_forward(q, k, v, None, causal, None, v_exp=13)[0]
    assert torch.equal(o, o2)
    assert rel(o, attn_fwd64(q, k, v, causal)) <= TOL


def test_cfg4_attention_16k_sampled_rows(dev):
    q, k, v = W.cfg4_attention(16384)
    g = torch.Generator().manual_seed(5)
    rows = torch.cat([torch.arange(0, 64), torch.randint(64, 16384, (192,), generator=g), torch.arange(16320, 16384)])
    _attn_checks(q, k, v, dev, rows=rows.sort().values, label="cfg4 S=16384")


# ---- Config 5: training step --------------------------------------------------------

def test_cfg5_linear_fwd_bwd(dev):
    x, w, dy = W.cfg5_train_linear()
    M, K = x.shape
    N = w.shape[0]
    xd = x.to(dev).requires_grad_()
    wd = w.to(dev).requires_grad_()
    y = autograd.linear(xd, wd)
    y.backward(dy.to(dev))
    # exponents of every quantisation the reference makes, bit-exact
    x16T, sx, exps = autograd._quantize_rows_t(x.to(dev), O.target_exp(K))
    assert np.array_equal(exps.cpu().numpy(), O.row_exps(x, O.target_exp(K)))
    _, sdy = ops.quantize_rows(dy.to(dev), 15, True)
    assert torch.equal(sdy.cpu(), O.quantize_rows(dy, 15, True)[1])
    _, swc = autograd._quantize_cols_t(w.to(dev), O.target_exp(N))
    assert torch.equal(swc.cpu(), O.quantize_cols(w, O.target_exp(N))[1])
    sx_o = O.quantize_rows(x, O.target_exp(K))[1]
    _, sdyc = autograd._quantize_cols_t(dy.to(dev), O.dw_target_exp(M), sx)
    assert torch.equal(sdyc.cpu(), O.quantize_cols(dy, O.dw_target_exp(M), sx_o)[1])
    # gradients vs fp64, and vs the reference's own (fp16-output) arithmetic
    xg, wg, dg = x.to(dev).double(), w.to(dev).double(), dy.to(dev).double()
    refs = {"y": xg @ wg.t(), "dx": dg @ wg, "dw": dg.t() @ xg}
    got = {"y": y, "dx": xd.grad, "dw": wd.grad}
    y_o, x16_o, sx_o2, _, _ = O.linear_train_fwd(x, w, double_round=True)
    dx_o, dw_o, _, _ = O.linear_train_bwd(dy, x16_o, sx_o2, w, double_round=True)
    own = {"y": y_o, "dx": dx_o, "dw": dw_o}
    for n in refs:
        e, eo = rel(got[n], refs[n]), rel(own[n].to(dev), refs[n])
        print(f"cfg5 linear {n}: rel err {e:.3e}  reference's own {eo:.3e}")
        assert torch.isfinite(got[n]).all() and e <= TOL and e <= eo * REF_SLACK + 1e-6, (n, e, eo)


def test_cfg5_attention_fwd_bwd(dev):
    q, k, v, do = W.cfg5_train_attention()
    from _ref64 import attn_bwd64
    qd, kd, vd = (t.to(dev).requires_grad_() for t in (q, k, v))
    o = autograd.sdpa(qd, kd, vd, is_causal=True)
    o.backward(do.to(dev))
    # exponents: forward a / ev (v_exp = 0), backward e / G
    a_o, ev_o = O.attn_exponents(q, k, v, 0)
    e_o, t_do, G_o = O.attn_bwd_exponents(do, O.expand_heads(ev_o, 16), 128)
    _, _, _, exps = attention.attn_forward(q.to(dev), k.to(dev), v.to(dev), None, True, None, 0, True, True)
    assert int(exps[0]) == a_o and torch.equal(exps[2:].cpu().reshape(ev_o.shape), ev_o.int())
    qv, kv, vv = q.to(dev), k.to(dev), v.to(dev)
    o2, lse, o16, exps2 = attention.attn_forward(qv, kv, vv, None, True, None, 0, True, True)
    dq, dk, dv, ex_b = autograd.attn_backward(qv, kv, vv, o16, lse, do.to(dev), exps2, None, 128 ** -0.5, True)
    assert (int(ex_b[0]), int(ex_b[1])) == (e_o, G_o)
    ro, rdq, rdk, rdv = attn_bwd64(qv, kv, vv, do.to(dev), True)
    # the reference's own training arithmetic (fp16 out16 / dq16 / dk16 / dv16 before
    # the bf16 scale-back), emulated by the oracle; its exponents are the closed forms
    own_o, own_dq, own_dk, own_dv, (a_r, _, e_r, G_r) = O.sdpa_bwd_reference_arith(qv, kv, vv, do.to(dev), True)
    assert (a_r, e_r, G_r) == (a_o, e_o, G_o)
    for n, g_, r_, w_ in (("o", o, ro, own_o), ("dq", qd.grad, rdq, own_dq), ("dk", kd.grad, rdk, own_dk),
                          ("dv", vd.grad, rdv, own_dv)):
        e, eo = rel(g_, r_), rel(w_, r_)
        print(f"cfg5 attention {n}: rel err {e:.3e}  reference's own {eo:.3e}")
        assert torch.isfinite(g_).all() and e <= TOL, (n, e)
        assert e <= eo * REF_SLACK + 1e-6, (n, e, eo)
