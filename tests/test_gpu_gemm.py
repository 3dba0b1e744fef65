"""hsl_gemm_f32 (fp32 MFMA GEMM) against an fp64 CPU product.

Tolerance: the fp32 result must lie within 2e-6 * sqrt(K) * (|A| |B|)_mn of the
fp64 product (|A||B| is the product of absolute values, the scale of the
rounding error of any fp32 summation order).
"""

import pytest
import torch

from prlstm_amd import _lib

pytestmark = pytest.mark.gpu


def _gemm(A, B, bias, M, N, K, ta, tb, split=True):
    dev = A.device
    C = torch.empty(M, N, device=dev)
    lda, ldb = max(A.shape[1], 1), max(B.shape[1], 1)
    nbytes = _lib.load().hsl_gemm_ws_bytes(M, N, K) if split else 0
    ws = torch.empty(max(nbytes, 1), dtype=torch.uint8, device=dev)
    P = _lib.ptr
    _lib.call("hsl_gemm_f32", P(A), P(B), P(bias), P(C), M, N, K, lda, ldb, N, int(ta), int(tb),
              P(ws), nbytes, _lib.stream_of(dev))
    return C


@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (5, 7, 3), (33, 65, 17), (128, 128, 32),
                                   (96, 48, 8192), (300, 200, 130), (2048, 512, 4096)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_matches_fp64(dev, M, N, K, ta, tb):
    print(f"gemm M={M} N={N} K={K} ta={ta} tb={tb}", flush=True)
    g = torch.Generator().manual_seed(M * 31 + N * 7 + K + ta * 2 + tb)
    a = torch.randn(M, K, generator=g)
    b = torch.randn(K, N, generator=g)
    bias = torch.randn(N, generator=g)
    A = (a.t().contiguous() if ta else a).to(dev)
    B = (b.t().contiguous() if tb else b).to(dev)
    C = _gemm(A, B, bias.to(dev), M, N, K, ta, tb).cpu().double()
    ref = a.double() @ b.double() + bias.double()
    scale = a.double().abs() @ b.double().abs() + bias.double().abs()
    err = (C - ref).abs()
    assert bool((err <= 2e-6 * max(K, 1) ** 0.5 * scale + 1e-30).all()), float((err / scale).max())


def test_gemm_split_and_unsplit_agree(dev):
    M, N, K = 256, 256, 16384
    g = torch.Generator().manual_seed(0)
    a = torch.randn(K, M, generator=g).to(dev)
    b = torch.randn(K, N, generator=g).to(dev)
    c1 = _gemm(a, b, None, M, N, K, 1, 0, split=True)
    c2 = _gemm(a, b, None, M, N, K, 1, 0, split=False)
    ref = a.cpu().double().t() @ b.cpu().double()
    e1 = (c1.cpu().double() - ref).abs().max().item()
    e2 = (c2.cpu().double() - ref).abs().max().item()
    print(f"split err {e1:.3e} unsplit err {e2:.3e}")
    assert e1 < 5e-3 and e2 < 5e-3


def test_gemm_empty_and_unaligned(dev):
    # K = 0 gives the bias; an offset (non 16-byte aligned) view takes the scalar path
    z = torch.zeros(3, 0, device=dev)
    bias = torch.arange(5.0, device=dev)
    C = _gemm(z, torch.zeros(0, 5, device=dev), bias, 3, 5, 0, 0, 0)
    assert torch.equal(C.cpu(), bias.cpu().expand(3, 5))
    base = torch.randn(1 + 37 * 19, device=dev)
    A = base[1:].view(37, 19)
    B = torch.randn(19, 23, device=dev)
    C = _gemm(A, B, None, 37, 23, 19, 0, 0)
    ref = A.cpu().double() @ B.cpu().double()
    assert (C.cpu().double() - ref).abs().max() < 1e-4


@pytest.fixture
def split_products():
    prev = _lib.set_split_products(1)
    yield
    _lib.set_split_products(prev)


SENTINEL = -12345.5


def _both(A, B, bias, M, N, K, lda=None, ldb=None, ta=0, tb=1, ldc=None):
    """C = op(A) op(B) (+bias) by the split-bf16 kernel and by the fp32 MFMA kernel
    (A B^T by default; ta=1, tb=0 for A^T B, with the workspace hsl_gemm_ws_bytes asks).
    C has a row before it, one after it and ldc - N columns beside it that must stay as they are."""
    dev = A.device
    out = []
    nbytes = _lib.load().hsl_gemm_ws_bytes(M, N, K)
    ws = torch.empty(max(nbytes, 1), dtype=torch.uint8, device=dev)
    for on in (1, 0):
        _lib.set_split_products(on)
        buf = torch.full((M + 2, ldc or N), SENTINEL, device=dev)
        C = buf[1:M + 1]
        P = _lib.ptr
        _lib.call("hsl_gemm_f32", P(A), P(B), P(bias), P(C), M, N, K, lda or A.shape[1], ldb or B.shape[1], ldc or N,
                  ta, tb, P(ws), nbytes, _lib.stream_of(dev))
        out.append(C[:, :N].cpu().double())
        C[:, :N] = SENTINEL
        assert bool((buf == SENTINEL).all())
    _lib.set_split_products(1)
    return out


@pytest.mark.parametrize("M,N,K,pad_a,pad_b", [(4096, 4096, 256, 0, 0), (4096 + 37, 4096 + 100, 207, 0, 0),
                                               (4352, 4096, 96, 3, 1), (2048, 8192, 1024, 0, 0),
                                               (2048, 4096, 512, 0, 0), (2048 + 5, 4096 - 64, 300, 1, 0)])
def test_split_products_as_accurate_as_fp32(dev, split_products, M, N, K, pad_a, pad_b):
    """Large A B^T products (>= 256 tiles of 256x256, or of 256x128: the last two shapes)
    take the split-bf16 kernel: every
    fp32 operand is split exactly into three bf16 pieces and the six largest piece
    products are accumulated in fp32.  Against the fp64 product it must meet the fp32
    bound, and its error statistics must match those of the fp32 MFMA kernel on the
    same operands (rows sampled for the fp64 reference)."""
    print(f"split products M={M} N={N} K={K} pad=({pad_a},{pad_b})", flush=True)
    g = torch.Generator().manual_seed(M + N + K)
    a = torch.randn(M, K + pad_a, generator=g)
    b = torch.randn(N, K + pad_b, generator=g) * 0.1
    bias = torch.randn(N, generator=g)
    cx6, c32 = _both(a.to(dev), b.to(dev), bias.to(dev), M, N, K, K + pad_a, K + pad_b)
    assert not torch.equal(cx6, c32)  # two different kernels ran
    rows = torch.arange(0, M, 97)
    av, bv = a[rows, :K].double(), b[:, :K].double()
    ref = av @ bv.t() + bias.double()
    scale = av.abs() @ bv.abs().t() + bias.double().abs()
    ex6 = (cx6[rows] - ref).abs() / scale
    e32 = (c32[rows] - ref).abs() / scale
    print(f"  rel err x6 max {ex6.max():.3e} rms {ex6.pow(2).mean().sqrt():.3e}; "
          f"fp32 max {e32.max():.3e} rms {e32.pow(2).mean().sqrt():.3e}", flush=True)
    assert float(ex6.max()) <= 2e-6 * K ** 0.5
    assert float(ex6.pow(2).mean().sqrt()) <= 1.25 * float(e32.pow(2).mean().sqrt()) + 1e-12
    assert float(ex6.max()) <= 2.0 * float(e32.max()) + 1e-12


def test_split_products_non_finite(dev, split_products):
    """A non-finite element of A makes its row of C NaN, one of B its column (piece
    products of an infinite piece with zero pieces are NaN); finite values beyond the
    bf16 range count as non-finite.  Everything else is unaffected, and the fp32 path
    (split products off) keeps the IEEE results."""
    M, N, K = 4096, 4096, 64
    g = torch.Generator().manual_seed(5)
    a = torch.randn(M, K, generator=g)
    b = torch.rand(N, K, generator=g) + 0.5
    a[3, 5] = float("inf")
    a[700, 0] = -float("inf")
    a[1200, 9] = float("nan")
    a[2000, 1] = 3.4e38  # finite in fp32, beyond bf16
    b[17, 2] = float("inf")
    cx6, c32 = _both(a.to(dev), b.to(dev), None, M, N, K)
    bad_rows = torch.tensor([3, 700, 1200, 2000])
    for r in bad_rows.tolist():
        assert bool(torch.isnan(cx6[r]).all()), r
    assert bool(torch.isnan(cx6[:, 17]).all())
    keep = torch.ones(M, dtype=torch.bool)
    keep[bad_rows] = False
    rest = cx6[keep][:, torch.arange(N) != 17]
    assert bool(torch.isfinite(rest).all())
    ref = c32[keep][:, torch.arange(N) != 17]
    assert float(((rest - ref).abs() / (ref.abs() + 1.0)).max()) < 1e-5
    # the fp32 instruction: IEEE infinities
    assert bool(torch.isposinf(c32[3, :17]).all()) and bool(torch.isneginf(c32[700, :17]).all())
    assert bool(torch.isnan(c32[1200]).all()) and bool(torch.isinf(c32[5:10, 17]).all())
    assert torch.equal(torch.sign(c32[5:10, 17]), torch.sign(a[5:10, 2]).double())


@pytest.mark.parametrize("M,N,K,pad,ta", [(4096, 256, 65536, 0, 1), (2048, 512, 8192, 0, 1), (1000, 300, 20000, 3, 1),
                                          (65536, 256, 4096, 0, 0), (2048, 1024, 8192, 0, 0), (3000, 300, 5000, 1, 0)])
def test_split_products_weight_gradient_layout(dev, split_products, M, N, K, pad, ta):
    """C = A^T B over a long K (the weight gradients dgates^T x, K = T*B) and C = A B
    (dx = dgates W_ih, K = 4H): the split-bf16 kernel sums fp32 runs of 64 k into a second
    fp32 accumulator and splits K into planes of at most 2048 k added in fp64; against the
    fp64 product it must meet the fp32 bound and match the fp32 kernel's error (rows
    sampled)."""
    print(f"split products {'A^T B' if ta else 'A B'} M={M} N={N} K={K} pad={pad}", flush=True)
    g = torch.Generator().manual_seed(M + 3 * N + K + ta)
    if ta:
        a = torch.randn(K, M + pad, generator=g) * 0.05   # dgates-like [K, M]
    else:
        a = torch.randn(M, K + pad, generator=g) * 0.05   # dgates-like [M, K]
    b = torch.randn(K, N + pad, generator=g)              # [K, N]
    cx6, c32 = _both(a.to(dev), b.to(dev), None, M, N, K, ta=ta, tb=0)
    assert not torch.equal(cx6, c32)
    rows = torch.arange(0, M, max(1, M // 100))
    av = (a[:, rows].t() if ta else a[rows, :K]).double()
    bv = b[:, :N].double()
    ref = av @ bv
    scale = av.abs() @ bv.abs()
    ex6 = (cx6[rows] - ref).abs() / scale
    e32 = (c32[rows] - ref).abs() / scale
    print(f"  rel err x6 max {ex6.max():.3e} rms {ex6.pow(2).mean().sqrt():.3e}; "
          f"fp32 max {e32.max():.3e} rms {e32.pow(2).mean().sqrt():.3e}", flush=True)
    assert float(ex6.max()) <= 2e-6 * K ** 0.5
    assert float(ex6.pow(2).mean().sqrt()) <= 1.25 * float(e32.pow(2).mean().sqrt()) + 1e-12
    assert float(ex6.max()) <= 2.0 * float(e32.max()) + 1e-12


@pytest.mark.parametrize("layout", ["abt", "abt_narrow", "atb", "ab"])
@pytest.mark.parametrize("three_piece", ["a", "b"])
def test_split_products_exact_on_representable_sums(dev, split_products, layout, three_piece):
    """Pins the piece bookkeeping of the split-bf16 kernels by exact arithmetic.  One
    operand holds values m * 2^-16 with |m| < 2^18 (three non-zero bf16 pieces in
    general), the other +-1 (one piece), and only 32 k-values are non-zero.  Every piece
    product that is kept then enters exactly, every partial sum is a multiple of 2^-16
    below 2^7 in magnitude, which fp32 represents exactly, so the result must equal the
    exact sum bit for bit: a wrong, swapped or missing piece changes it.  The long-K
    layouts (A^T B, A B) run over K = 8192 (their size rule) with the 32 non-zero k in one
    band, which also exercises their k-splits and the fp64 sum of the planes."""
    g = torch.Generator().manual_seed(len(layout) * 7 + (three_piece == "a"))

    def fine(*shape):
        return torch.randint(-(1 << 18) + 1, 1 << 18, shape, generator=g).double() * 2.0 ** -16

    def sign(*shape):
        return torch.randint(0, 2, shape, generator=g).double() * 2 - 1

    def pair(shape_a, shape_b):
        return (fine(*shape_a), sign(*shape_b)) if three_piece == "a" else (sign(*shape_a), fine(*shape_b))

    if layout.startswith("abt"):  # C = A B^T, A [M,K], B [N,K]; narrow: 256 tiles of 256x128
        M, N, K = (4096, 4096, 32) if layout == "abt" else (2048, 4096, 32)
        a, b = pair((M, K), (N, K))
        exact, ta = a @ b.t(), 0
    else:
        M, N, K = 4096, 256, 8192
        band = torch.zeros(K, dtype=torch.double)
        band[1024:1056] = 1.0
        if layout == "atb":  # C = A^T B, A [K,M], B [K,N]
            a, b = pair((K, M), (K, N))
            a, b = a * band[:, None], b * band[:, None]
            exact, ta = a.t() @ b, 1
        else:  # C = A B, A [M,K], B [K,N]
            a, b = pair((M, K), (K, N))
            a, b = a * band[None, :], b * band[:, None]
            exact, ta = a @ b, 0
    print(f"exact sums layout={layout} three-piece operand={three_piece} M={M} N={N} K={K}", flush=True)
    cx6, c32 = _both(a.float().to(dev), b.float().to(dev), None, M, N, K, ta=ta, tb=int(layout.startswith("abt")))
    assert torch.equal(cx6, exact)
    assert torch.equal(c32, exact)


MIDDLE = [(64, 96, 1024), (65, 1024, 95), (129, 1000, 65), (200, 64, 1931), (1000, 67, 203), (333, 65, 700),
          (131, 97, 1430), (700, 650, 2603), (1027, 130, 64),            # gemm_m6.hip: edges of tiles and slices
          (128, 128, 16384), (256, 384, 2560), (1024, 256, 1040)]          # whole 128 x 128 tiles
LAYOUTS = [(0, 0), (0, 1), (1, 0)]


@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("M,N,K", MIDDLE)
@pytest.mark.parametrize("pad", [0, 1])
def test_middle_split_products(dev, split_products, M, N, K, ta, tb, pad):
    """Middle-sized and ragged products on split pieces, with and without 16-byte aligned rows:
    the fp32 bound against fp64, an rms error not above the fp32 kernel's (5% for the sampling
    noise of the rms; the fp64-folded sums of the backward are compared below), and nothing
    written beside C, whose rows are also longer than N here."""
    print(f"middle split products M={M} N={N} K={K} ta={ta} tb={tb} pad={pad}", flush=True)
    g = torch.Generator().manual_seed(M + N + K)
    a = torch.randn(*((K, M + pad) if ta else (M, K + pad)), generator=g)
    b = torch.randn(*((N, K + pad) if tb else (K, N + pad)), generator=g) * 0.1
    bias = torch.randn(N, generator=g)
    c6, c32 = _both(a.to(dev), b.to(dev), bias.to(dev), M, N, K, ta=ta, tb=tb, ldc=N + 5 * pad)
    assert not torch.equal(c6, c32)  # two different kernels ran
    av = (a[:, :M].t() if ta else a[:, :K]).double()
    bv = (b[:, :K].t() if tb else b[:, :N]).double()
    ref = av @ bv + bias.double()
    scale = av.abs() @ bv.abs() + bias.double().abs()
    e6, e32 = (c6 - ref).abs() / scale, (c32 - ref).abs() / scale
    assert float(e6.max()) <= 2e-6 * K ** 0.5
    assert float(e6.pow(2).mean().sqrt()) <= 1.05 * float(e32.pow(2).mean().sqrt())


@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("M,N,K", [(200, 100, 700), (256, 256, 4096)])
def test_middle_split_products_non_finite(dev, split_products, M, N, K, ta, tb):
    """Non-finite and out-of-bf16-range operands give the fp32 instruction's results: the same
    NaN, +inf and -inf elements, and finite elements within the fp32 bound of each other."""
    print(f"non-finite M={M} N={N} K={K} ta={ta} tb={tb}", flush=True)
    g = torch.Generator().manual_seed(K)
    a = torch.randn(M, K, generator=g)
    b = torch.randn(N, K, generator=g)
    a[3, 5], a[40, 7], a[77, K - 1], a[199, 0] = float("inf"), float("-inf"), float("nan"), 3.4e38
    b[9, 2], b[99, K - 1] = float("inf"), float("nan")
    A = (a.t().contiguous() if ta else a).to(dev)
    B = (b if tb else b.t().contiguous()).to(dev)
    c6, c32 = _both(A, B, None, M, N, K, ta=ta, tb=tb)
    for what in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(what(c6), what(c32)), what
    ok = torch.isfinite(c32)
    scale = (a.double().abs() @ b.double().abs().t())[ok]
    assert bool(((c6 - c32)[ok].abs() <= 4e-6 * K ** 0.5 * scale).all())


@pytest.mark.parametrize("M,N,K", [(130, 200, 16384), (128, 256, 8192), (70, 1030, 4100)])
def test_deep_products_of_few_tiles_use_the_workspace(dev, split_products, M, N, K):
    """C = A B^T of few tiles and many k is cut along K into the workspace's planes, which are
    added in fp64: nearer the fp64 product than the one running sum without a workspace."""
    print(f"deep A B^T M={M} N={N} K={K}", flush=True)
    g = torch.Generator().manual_seed(K)
    a, b = torch.rand(M, K, generator=g), torch.rand(N, K, generator=g)
    ref = a.double() @ b.double().t()
    cut, whole = (_gemm(a.to(dev), b.to(dev), None, M, N, K, 0, 1, split=s).cpu().double() for s in (True, False))
    e_cut, e_whole = float((cut - ref).norm() / ref.norm()), float((whole - ref).norm() / ref.norm())
    print(f"  planes {e_cut:.3e} one sum {e_whole:.3e}")
    assert e_cut <= 0.6 * e_whole


@pytest.mark.parametrize("M,N,K,ta,tb,ws,fp32", [
    (256, 512, 64, 0, 1, 0, True), (1024, 2048, 256, 0, 1, 0, True), (2100, 128, 64, 0, 1, 0, True),
    (1024, 1024, 128, 1, 0, 1, True), (1024, 512, 256, 0, 0, 1, True),
    (1000, 63, 203, 0, 1, 0, True), (2048, 33, 9800, 1, 0, 1, True), (2048, 64, 9800, 1, 0, 1, False),
    (4096, 1024, 256, 0, 1, 0, False), (300, 704, 2048, 0, 1, 0, False), (1024, 512, 512, 1, 0, 1, False),
    (1024, 1024, 288, 0, 1, 0, False), (1024, 2048, 260, 0, 1, 0, False)])
def test_which_whole_products_stay_on_the_fp32_kernel(dev, split_products, M, N, K, ta, tb, ws, fp32):
    """Whole tiles of the fp32 kernel on at most one workgroup per CU, in one split of at most
    256 k, and products of fewer than 64 columns run there with split products on too (the results
    are the same bits); their neighbours do not."""
    g = torch.Generator().manual_seed(K)
    a = torch.randn(*((K, M) if ta else (M, K)), generator=g).to(dev)
    b = torch.randn(*((N, K) if tb else (K, N)), generator=g).to(dev)
    out = []
    for on in (1, 0):
        _lib.set_split_products(on)
        out.append(_gemm(a, b, None, M, N, K, ta, tb, split=bool(ws)))
    assert torch.equal(*out) == fp32


@pytest.mark.parametrize("mean", [0.0, 0.5, 2.0])
@pytest.mark.parametrize("T,B,D,H", [(256, 8, 128, 512),    # K = 2048 either way, whole tiles
                                     (256, 7, 100, 333),    # ragged
                                     (35, 20, 650, 650),    # dx over K = 2600
                                     (128, 32, 50, 300),    # fewer than 64 columns: the fp32 kernel either way
                                     (128, 32, 256, 256)])  # dW_ih over K = 4096
def test_middle_gradients_as_accurate_as_fp64_folded_sums(dev, split_products, T, B, D, H, mean):
    """The weight gradient and dx products of the backward: with split products off their fp32
    kernel folds every 128 k into fp64.  The split pieces' fp32 sums are no further from the
    64-bit products of the same operands, of zero mean and not (5% for the noise of the rms)."""
    print(f"gradients T={T} B={B} D={D} H={H} mean={mean}", flush=True)
    lib, P, s = _lib.load(), _lib.ptr, _lib.stream_of(dev)
    g = torch.Generator(device=dev).manual_seed(T + H)
    rand = lambda *shape: torch.randn(*shape, device=dev, generator=g)  # noqa: E731
    gates, x, w, dout, c0 = rand(T, B, 4 * H), rand(T, B, D) + mean, rand(4 * H, D) + mean, rand(T, B, H) + mean, \
        rand(B, H).abs()
    out, ck = torch.empty(T, B, H, device=dev), torch.empty(lib.hsl_scan_ck_rows(T), B, H, device=dev)
    _lib.call("hsl_scan_fwd", P(gates), P(c0), 1e-6, P(out), P(ck), T, B, H, s)
    dg = torch.empty_like(gates)  # (T is short enough that the backward's scan is this one, uncut)
    _lib.call("hsl_scan_bwd", P(gates), P(c0), P(ck), P(dout), None, None, 1e-6, P(dg), None, None, T, B, H, s)
    dg, x2 = dg.double().view(T * B, 4 * H), x.double().view(T * B, D)
    want = {"dw": dg.t() @ x2, "dx": dg @ w.double()}
    err = {}
    for on in (1, 0):
        _lib.set_split_products(on)
        n = lib.hsl_par_bwd_ws_bytes(T, B, D, H)
        ws = torch.empty(n, dtype=torch.uint8, device=dev)
        got = {"dw": torch.empty(4 * H, D, device=dev), "dx": torch.empty(T * B, D, device=dev)}
        _lib.call("hsl_par_bwd", P(dout), None, None, P(x), P(c0), P(gates), P(ck), P(w), 1e-6, P(got["dx"]),
                  P(got["dw"]), P(torch.empty(4 * H, device=dev)), None, P(ws), n, T, B, D, H, s)
        err[on] = {k: float((got[k].double() - v).norm() / v.norm()) for k, v in want.items()}
    print(err)
    for k in want:
        assert err[1][k] <= 1.05 * err[0][k] <= 1e-6, k
