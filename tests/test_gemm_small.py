"""Few-row GEMMs (sx8_gemm_small.hip): sx8_linear_f16 and the packed form behind the prefill
entry points at up to 128 rows.  Sizes at the edges of the kernel's tiles: 16-row fragments,
16 / 32 / 48-column tiles (every pair of row and column fragments that a plan picks), four-block groups, K tails inside a block and odd rows (whose last
element shares a word with the next row).  W16 is the oracle's R64 dequant; the bar against its
float64 product is the other GEMM tests' 1e-3 of max |Y| (weights rounded to fp16), and the
tiled kernels, forced by SX8_GEMM_TILE, multiply the same fp16 operands, so the two differ by
the order of float32 sums: at most K 2^-24 sum |x w| / max |Y|, below 1e-5 here."""
import ctypes

import numpy as np
import pytest


def _quantized(N, K, seed, cuda):
    import torch
    from quantize_sx8 import quantize_tensor
    g = torch.Generator(device="cpu").manual_seed(seed)
    W = (torch.randn(N, K, generator=g) * 0.02).half()
    return quantize_tensor(W, device=cuda, degenerate_frac=0.01, seed=seed + 1)


def _rel(a, b):
    return (a.double() - b.double()).abs().max().item() / b.double().abs().max().item()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,hb,bias", [
    (2, 64, 32, 6, False), (3, 80, 31, 8, True), (15, 1000, 1333, 6, True), (16, 2560, 4096, 8, False),
    (17, 1024, 2560, 6, True), (31, 9728, 515, 6, False), (32, 305, 2081, 8, True), (1, 129, 97, 6, False),
    (8, 4099, 640, 6, True), (8, 9728, 515, 6, True), (12, 6000, 99, 8, False), (32, 6001, 160, 8, True),
])
def test_linear_f16(hiplib, oracle, cuda, M, N, K, hb, bias):
    """fp16 outputs against the oracle (fp16 rounding on top of the GEMM bar), the bias as an
    fp16 sum on top, a row stride past K, and the module that calls it."""
    import torch
    import _sx8lib as L
    from integrate_fused_v44 import SX8LinearV44
    from sx8_decode1_v3 import make_tensors_v44
    print("linear", M, N, K, hb, flush=True)
    qt, bi = _quantized(N, K, 31 * M + N, cuda)
    t = make_tensors_v44(qt, bi, hdr_aligned=(hb == 8))
    g = torch.Generator(device="cpu").manual_seed(M)
    wide = torch.randn(M, K + 5, generator=g).half().to(cuda)
    wide[:, K:] = float("nan")                       # outside the rows: never part of a product
    X = wide[:, :K].contiguous()
    b = torch.randn(N, generator=g).half().to(cuda) if bias else None
    P = L.ptr

    def call(x, ld, bb):
        Y = torch.full((M, N), 7.0, dtype=torch.float16, device=cuda)
        L.call("sx8_linear_f16", P(x), M, ld, K, P(t[0]), P(t[1]), hb, P(t[2]), P(t[3]), P(bb), N, qt["n_cb"], P(Y),
               L.stream(cuda))
        return Y

    Y = call(X, K, None)
    ref = oracle.gemm_f64(X.cpu().numpy(), oracle.dequant_r64(qt, bi))
    err = np.abs(Y.cpu().numpy().astype(np.float64) - ref)
    assert (err <= 1e-3 * np.abs(ref).max() + 2.0 ** -11 * np.abs(ref)).all()
    assert torch.equal(call(wide, K + 5, None), Y)
    if bias:
        assert torch.equal(call(X, K, b), Y + b)
    lin = SX8LinearV44(qt, bi, b, hdr_bytes=hb)
    lin._t44 = t
    y = lin(X.reshape(1, M, K))
    assert y.shape == (1, M, N)
    if M > 1:
        assert torch.equal(y[0], Y + b if bias else Y)
        fp32_bias = torch.zeros(N, device=cuda)      # promotes the sum: the unfused path
        assert SX8LinearV44(qt, bi, fp32_bias, hdr_bytes=hb)(X).dtype == torch.float32


@pytest.mark.gpu
@pytest.mark.parametrize("M", [2, 16, 31])
@pytest.mark.parametrize("K", [31, 96, 128, 129, 510, 512, 2047])
def test_linear_f16_row_starts(hiplib, cuda, M, K):
    """Rows that begin anywhere in their 4-byte words, with NaN before, between and after them, give
    bit for bit what the same rows at 16 bytes give."""
    import torch
    import _sx8lib as L
    from sx8_decode1_v3 import make_tensors_v44
    print("row starts", M, K, flush=True)
    N = 70
    qt, bi = _quantized(N, K, M + K, cuda)
    t = make_tensors_v44(qt, bi)
    X = torch.randn(M, K, generator=torch.Generator().manual_seed(M + K)).half().to(cuda)
    P = L.ptr

    def call(x, ld):
        Y = torch.full((M, N), 7.0, dtype=torch.float16, device=cuda)
        L.call("sx8_linear_f16", P(x), M, ld, K, P(t[0]), P(t[1]), 6, P(t[2]), P(t[3]), None, N, qt["n_cb"], P(Y),
               L.stream(cuda))
        return Y
    pad = (K + 7) // 8 * 8
    even = torch.full((M, pad), float("nan"), dtype=torch.float16, device=cuda)
    even[:, :K] = X
    want = call(even, pad)
    assert want.isfinite().all()
    for ld in (K, K + 1, K + 2):
        for off in (0, 1, 2, 3):
            for tail in (0, 1):                       # X ends where its buffer ends, and before
                buf = torch.full((off + (M - 1) * ld + K + tail,), float("nan"), dtype=torch.float16, device=cuda)
                x = buf[off:].as_strided((M, K), (ld, 1))
                x.copy_(X)
                assert torch.equal(call(x, ld), want), (ld, off, tail)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [2, 17, 32])
def test_linear_f16_basis_range(hiplib, cuda, M):
    """Bases of any length with their scales the other way: Z keeps its 22 bits, and powers of two
    past the unscaled range change no bit between them (nothing is rounded where both are undone)."""
    import torch
    from sx8_decode1_v3 import make_tensors_v44
    from sx8_gemm_compact import linear_sx8
    print("basis range", M, flush=True)
    N, K = 130, 640 + 35
    qt, bi = _quantized(N, K, M, cuda)
    hdr, lv, bas, sca = make_tensors_v44(qt, bi)
    sca = sca * 64                                    # a PCA part as large as the core weights'
    X = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).half().to(cuda)
    want = linear_sx8(X, qt, hdr, lv, bas, sca)
    assert want.isfinite().all() and (want - linear_sx8(X, qt, hdr, lv, bas * 0, sca)).abs().max() > 0.1
    def scaled(f0, f1):
        f = torch.tensor([f0, f1], dtype=torch.float64, device=cuda)
        b = (bas.view(-1, 2, 32).double() * f[:, None]).float().view(-1, 64).contiguous()
        return linear_sx8(X, qt, hdr, lv, b, (sca.double() / f).float().contiguous())
    # the PCA part, about as large as Y, to 2^-22 and two float32 factors, and one fp16 rounding of
    # the output that may fall either way
    near = lambda y: ((y - want).abs() <= 2.0 ** -10 * want.abs() + 4e-6 * want.abs().max()).all()
    small = scaled(2.0 ** -12, 2.0 ** -12)
    assert near(small)
    for e0, e1 in ((17, 17), (-40, 30), (60, -60), (-100, 0)):
        assert torch.equal(scaled(2.0 ** e0, 2.0 ** e1), small), (e0, e1)
    for f in (1e-3, 3e-5, 0.2, 300.0, 7e4):
        assert near(scaled(f, f)), f
    # a power of two of its own for every block and vector
    e = torch.randint(-30, 30, (bas.shape[0], 2), generator=torch.Generator().manual_seed(M)).double().to(cuda)
    b = (bas.view(-1, 2, 32).double() * 2.0 ** e[..., None]).float().view(-1, 64).contiguous()
    assert near(linear_sx8(X, qt, hdr, lv, b, (sca.double() * 2.0 ** -e).float().contiguous()))


@pytest.mark.gpu
@pytest.mark.parametrize("M", [4, 32])
def test_linear_f16_not_finite(hiplib, cuda, M):
    """Infinities and NaN of X stay in their rows, which are NaN as the tiled kernels give them
    (Z's second fp16 part of an infinity is NaN)."""
    import torch
    from sx8_decode1_v3 import make_tensors_v44
    from sx8_gemm_compact import gemm_sx8_compact, linear_sx8
    print("not finite", M, flush=True)
    N, K = 200, 515
    qt, bi = _quantized(N, K, M, cuda)
    t = make_tensors_v44(qt, bi)
    X = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).half().to(cuda)
    want = linear_sx8(X, qt, *t)
    X[1, 70], X[M - 1, K - 1] = float("inf"), float("nan")
    got = linear_sx8(X, qt, *t)
    rows = [i for i in range(M) if i not in (1, M - 1)]
    assert torch.equal(got[rows], want[rows]) and got[[1, M - 1]].isnan().all()
    assert torch.equal(got.isnan(), gemm_sx8_compact(X, qt, bi, *t).isnan())


@pytest.mark.gpu
@pytest.mark.parametrize("N,K,hb,bias", [
    (1024, 2560, 6, False), (2560, 9728, 8, True), (33, 31, 6, True), (300, 97, 8, False), (777, 1333, 6, True),
    (4097, 4095, 8, True), (129, 4098, 6, False), (100, 16390, 6, True), (70001, 64, 6, True),
])
def test_one_row_equals_gemv(hiplib, cuda, N, K, hb, bias):
    """One row through sx8_linear_f16 is bit for bit decode1_v44's float32 result converted
    (and the bias added): widths at the panel forms' edges, K tails inside a block and odd K,
    table passes past the up-front ones, a row 2 bytes off 16-byte alignment."""
    import torch
    from sx8_decode1_v3 import decode1_v44, make_tensors_v44
    from sx8_gemm_compact import linear_sx8
    print("one row", N, K, hb, flush=True)
    qt, bi = _quantized(N, K, N + K, cuda)
    t = make_tensors_v44(qt, bi, hdr_aligned=(hb == 8))
    g = torch.Generator(device="cpu").manual_seed(K)
    buf = torch.full((K + 1,), float("nan"), dtype=torch.float16, device=cuda)
    buf[1:] = torch.randn(K, generator=g).half().to(cuda)
    x = buf[1:]
    b = torch.randn(N, generator=g).half().to(cuda) if bias else None
    y = decode1_v44(x.clone(), qt, bi, *t, hdr_bytes=hb)[0].half()
    assert torch.equal(linear_sx8(x[None], qt, *t, hb, b)[0], y + b if bias else y)
    assert torch.equal(linear_sx8(x.clone()[None], qt, *t, hb, None)[0], y)
    assert linear_sx8(buf[None], qt, *t, hb, None) is None          # not in_f long: decode1_v44's rules


@pytest.mark.gpu
@pytest.mark.parametrize("M,Ns,K,hb", [
    (1, [64], 96, 6), (16, [1000], 2560, 8), (17, [129, 300, 64, 700], 80, 6), (33, [4096, 1024, 1024], 2560, 6),
    (48, [777], 1000, 6), (49, [513], 4096, 8), (64, [9728], 640, 6), (65, [640], 1333, 6), (80, [1001], 515, 8),
    (96, [300, 500], 2081, 6), (97, [256], 129, 6), (128, [2560], 2560, 6), (16, [9729], 515, 6), (32, [9728], 640, 8),
    (27, [4001, 3000, 1000, 900], 259, 6), (31, [6001], 320, 8), (45, [5003], 640, 6), (64, [4100, 2000], 515, 8),
    (80, [5001], 320, 6),
])
def test_packed_forms_match_tiles(hiplib, oracle, cuda, gemm_tuning, M, Ns, K, hb):
    """sx8_gemm_prefill_group against the oracle, against the tiled kernels, and against the
    split-array and caller-Z contracts of the same product."""
    import torch
    import _sx8lib as L
    from sx8_decode1_v3 import make_tensors_v44
    from sx8_fused_wmma import gemm_sx8_wmma_cached, make_tensors, to_kbmajor
    from sx8_gemm_compact import _ext
    print("packed", M, Ns, K, hb, flush=True)
    mats = [_quantized(N, K, 900 + 7 * i + M, cuda) for i, N in enumerate(Ns)]
    ts = [make_tensors_v44(qt, bi, hdr_aligned=(hb == 8)) for qt, bi in mats]
    n, n_cb = len(Ns), mats[0][0]["n_cb"]
    X = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).half().to(cuda)
    arr = lambda i: (ctypes.c_void_p * n)(*[t[i].data_ptr() for t in ts])

    def group():
        ys = [torch.full((M, N), float("nan"), device=cuda) for N in Ns]
        ws, nb = L.gemm_workspace(M, Ns, n_cb, cuda)
        L.call("sx8_gemm_prefill_group", L.ptr(X), M, K, K, n, arr(0), arr(1), hb, arr(2), arr(3),
               (ctypes.c_int64 * n)(*Ns), n_cb, (ctypes.c_void_p * n)(*[y.data_ptr() for y in ys]), L.ptr(ws), nb,
               L.stream(cuda))
        return ys

    ys = group()
    assert all(torch.equal(a, b) for a, b in zip(ys, group()))      # deterministic
    gemm_tuning(TILE="256")
    tiles = group()
    gemm_tuning(TILE=None)
    for (qt, bi), y, yt in zip(mats, ys, tiles):
        ref = oracle.gemm_f64(X.cpu().numpy(), oracle.dequant_r64(qt, bi))
        assert oracle.rel_err(y.cpu().numpy(), ref) <= 1e-3
        assert _rel(y, yt) <= 1e-5
    if n == 1:
        qt, bi = mats[0]
        assert torch.equal(gemm_sx8_wmma_cached(X, make_tensors(to_kbmajor(qt, bi)[0], bi, cuda), n_cb), ys[0])
        Xp = torch.zeros(M, n_cb * 32, dtype=torch.float16, device=cuda)
        Xp[:, :K] = X
        Z = _ext().compute_z44_batch(Xp, ts[0][2], ts[0][3], n_cb)
        assert torch.equal(_ext().gemm_compact(Xp, ts[0][0], ts[0][1], Z, n_cb, hb), ys[0])


def test_linear_f16_refusals(hiplib):
    """Bad arguments and sizes past the kernel's are turned into errors on the host."""
    L, p = hiplib, ctypes.c_void_p(4096)
    N0 = ctypes.c_void_p(None)
    ok = [p, 4, 64, 64, p, p, 6, p, p, N0, 128, 2, p, N0]

    def call(**kw):
        a = list(ok)
        for k, v in kw.items():
            a[int(k[1:])] = v
        return L.sx8_linear_f16(*a)

    assert call(a0=N0) == 1 and call(a12=N0) == 1 and call(a7=N0) == 1
    assert call(a6=7) == 1                            # header width
    assert call(a2=63) == 1 and call(a11=3) == 1      # row stride below K; n_cb != ceil(K / 32)
    assert call(a1=0) == 1 and call(a10=0) == 1
    assert call(a5=ctypes.c_void_p(4100)) == 1        # levels misaligned
    assert call(a1=33) == 3                           # rows
    assert call(a10=1 << 27) == 3                     # levels past 2 GiB
    assert b"at most 32 rows" in L.sx8_last_error()
