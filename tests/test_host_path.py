"""The native per-call path of the wrappers (sx8_py.cpp) against their general path: the same
bits, shapes and types for every form of input, whichever of the two takes it."""
import ctypes

import numpy as np
import pytest
import torch


class _Decline:
    """A host module that takes no call."""

    def __getattr__(self, name):
        return lambda *a: None


@pytest.fixture
def both(hiplib, monkeypatch):
    """Run f through the native path, then through the general one; the native calls taken."""
    import _sx8lib

    def run(f):
        real, taken = _sx8lib.py(), []

        class Watch:
            def __getattr__(self, name):
                def g(*a):
                    r = getattr(real, name)(*a)
                    taken.append((name, r is not None))
                    return r
                return g
        monkeypatch.setattr(_sx8lib, "_py", Watch())
        def result():
            try:
                return f().clone()
            except (RuntimeError, ValueError) as e:
                return type(e)
        a = result()
        monkeypatch.setattr(_sx8lib, "_py", _Decline())
        b = result()
        monkeypatch.setattr(_sx8lib, "_py", real)
        return a, b, [n for n, t in taken if t]
    return run


def _same(a, b):
    if isinstance(b, type):                              # refused
        assert a is b
        return
    assert a.shape == b.shape and a.dtype == b.dtype and a.device == b.device and a.stride() == b.stride()
    a, b = a.detach(), b.detach()
    assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))


def _weight(N, K, seed=3):
    from quantize_sx8 import quantize_tensor
    g = torch.Generator().manual_seed(seed)
    return quantize_tensor((torch.randn(N, K, generator=g) * 0.02).half(), device="cpu", degenerate_frac=0.01, seed=1)


def test_host_tensors_are_left_to_the_general_path(hiplib):
    import _sx8lib
    py = _sx8lib.py()
    h, f = torch.zeros(1, 64, dtype=torch.float16), torch.zeros(64)
    u = torch.zeros(128, 6, dtype=torch.uint8)
    assert py.linear(h, (u, u, f, f), 6, None, 64, 64, 64, 2) is None
    assert py.gemv(h[0], u, u, f, f, 6, 64, 2, f) is None
    assert py.gemm(h, u, u, f, f, 6, 64, 64, 2) is None
    assert py.gemm_split(h, f, f, u, u, u, u, f, f, 2) is None
    assert py.dequant(h, h, u, u, u, u, f, f, 64, 64, 2) is None
    assert py.dequant(*[np.zeros(4)] * 8, 64, 64, 2) is None
    assert py.embed(torch.zeros(1, dtype=torch.long), u, u, f, f, 64, 64, 2, h) is None
    assert py.to_host(u) is None
    assert py.gemm(h, u, u, f, f, 6, 64, 64.0, 2) is None          # not an integer: no error here either
    assert py.gemv(h[0], u, u, f, f, 6, 64, None, f) is None
    with pytest.raises(TypeError):
        py.linear(h)
    with pytest.raises(KeyError):
        py.bind({})
    py.bind({n: ctypes.cast(getattr(hiplib, n), ctypes.c_void_p).value for n, _, _ in _sx8lib.SIGNATURES})


@pytest.mark.gpu
@pytest.mark.parametrize("hdr", [6, 8])
@pytest.mark.parametrize("N,K", [(96, 100), (40, 64)])
def test_linear_forms(both, cuda, N, K, hdr):
    from integrate_fused_v44 import SX8LinearV44
    qt, bi = _weight(N, K)
    g = torch.Generator().manual_seed(5)
    X = torch.randn(80, K + 3, generator=g).half().to(cuda)
    bias = torch.nn.Parameter(torch.randn(N, generator=g).half().to(cuda))
    forms = {"rows1": X[:1, :K].contiguous(), "vec": X[3, :K].contiguous(), "offset": X.reshape(-1)[1:1 + K],
             "strided": X[:7, :K], "transposed": X[:5, :K].t().contiguous().t(),
             "batch": X[:6, :K].reshape(2, 3, K), "rows32": X[:32, :K].contiguous(), "rows33": X[:33, :K].contiguous(),
             "empty_batch_dims": X[:1, :K].reshape(1, 1, 1, K), "float": X[:2, :K].float(), "longer": X[:2].contiguous()}
    for b, grad in ((None, False), (bias, False), (bias, True), (bias.detach().float(), False)):
        m = SX8LinearV44(qt, bi, b, hdr_bytes=hdr)
        m._load_t44()
        for name, x in forms.items():
            with torch.set_grad_enabled(grad):
                y, ref, taken = both(lambda: m(x))
            _same(y, ref)
            if isinstance(y, torch.Tensor):
                assert y.requires_grad == ref.requires_grad, name
            if name in ("rows1", "vec", "offset") and b is None:
                assert taken == ["linear"], name


@pytest.mark.gpu
def test_wrappers(both, cuda, monkeypatch):
    from kernel_sx8_v43 import decode_tensor_gpu_fast
    from sx8_decode1_v3 import decode1_v44, make_tensors_v44
    from sx8_embed_v44 import SX8EmbeddingV44
    from sx8_fused_wmma import gemm_sx8_wmma_cached, make_tensors, to_kbmajor
    from sx8_gemm_compact import gemm_sx8_compact
    N, K = 130, 96
    qt, bi = _weight(N, K)
    g = torch.Generator().manual_seed(6)
    X = torch.randn(140, K + 8, generator=g).half().to(cuda)
    t = make_tensors_v44(qt, bi)
    split = make_tensors(to_kbmajor(qt, bi)[0], bi, cuda)
    for x in (X[:1, :K].contiguous(), X[:77, :K].contiguous(), X[:3, :K], X[:5].contiguous(), X[:2, :K].float()):
        y, ref, taken = both(lambda: gemm_sx8_compact(x, qt, bi, *t))
        _same(y, ref)
        assert (taken == ["gemm"]) == (x.is_contiguous() and x.dtype == torch.float16)
        y, ref, _ = both(lambda: gemm_sx8_wmma_cached(x, split, qt["n_cb"]))
        _same(y, ref)
    with pytest.raises(ValueError):
        gemm_sx8_compact(X[:4, :K - 1].contiguous(), qt, bi, *t)
    y, ref, taken = both(lambda: gemm_sx8_compact(X[:4, :K].contiguous(), qt, bi, *t, in_f=float(K)))
    _same(y, ref)
    assert isinstance(y, torch.Tensor) and not taken
    for x in (X[0, :K].contiguous(), X[0, :K - 4], X.reshape(-1)[3:3 + K], X[:1, :K].float(), X[1]):
        y, ref, _ = both(lambda: decode1_v44(x, qt, bi, *t)[0])
        _same(y, ref)
    dq = {k: torch.as_tensor(np.ascontiguousarray(v).view(np.int16 if v.dtype == np.float16 else v.dtype)).to(cuda)
          if isinstance(v, np.ndarray) else v for k, v in qt.items()}
    db = dict(bi, data=torch.as_tensor(bi["data"]).to(cuda), scales=torch.as_tensor(bi["scales"]).to(cuda))
    for q, b, want in ((dq, db, ["dequant"]), (dict(dq, dmin=dq["dmin"].view(torch.float16)), db, ["dequant"]),
                       (qt, bi, []), (dict(dq, orig_shape=(N // 2, 2 * K)), db, ["dequant"]),
                       (dict(dq, config=dq["config"].int()), db, [])):
        y, ref, taken = both(lambda: decode_tensor_gpu_fast(q, b))
        _same(y, ref)
        assert taken == want
    with pytest.raises(ValueError):
        decode_tensor_gpu_fast(dict(dq, n_blocks=1), db)
    with pytest.raises(ValueError):
        decode_tensor_gpu_fast(dq, dict(db, scales=db["scales"][:1]))
    emb = SX8EmbeddingV44(qt, bi)
    ids = torch.randint(0, N, (4, 9), generator=g).to(cuda)
    for i in (ids, ids[0], ids[0, 0], ids[:, ::2], ids.int(), ids[:0]):
        y, ref, taken = both(lambda: emb(i))
        _same(y, ref)


@pytest.mark.gpu
def test_stream_and_capture(hiplib, cuda):
    """The native path launches on the current stream, and a graph that captured it replays."""
    from integrate_fused_v44 import SX8LinearV44
    qt, bi = _weight(128, 256)
    m = SX8LinearV44(qt, bi)
    x = torch.randn(4, 256, dtype=torch.float16, device=cuda)
    m(x)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        y = m(x)
    for i in range(3):
        x.normal_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, m(x))
        with torch.cuda.stream(s):
            z = m(x)
        s.synchronize()
        assert torch.equal(y, z)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 1 << 20, (1 << 20) + 1, (2 << 20) + 5, (7 << 20) - 3])
def test_to_host(hiplib, cuda, n):
    import _sx8lib
    x = torch.randint(0, 256, (n,), dtype=torch.uint8, device=cuda)
    for _ in range(2):
        y = _sx8lib.py().to_host(x)
        assert (y is None) == (n <= 1 << 20)
        assert y is None or (not y.is_cuda and torch.equal(y, x.cpu()))
        x.bitwise_not_()


def test_without_a_host_module(hiplib, monkeypatch, tmp_path):
    """Missing, built for something else or for another library: one warning, no call taken."""
    import _sx8lib
    real = _sx8lib.py()
    assert real.torch_version == torch.__version__ and not isinstance(real, _sx8lib._NoHostModule)
    for path, why in ((tmp_path / "none.so", "not found"), (tmp_path / "bad.so", "bad.so")):
        if why == "bad.so":
            path.write_bytes(b"not a module")
        monkeypatch.setattr(_sx8lib, "PY_PATH", str(path))
        monkeypatch.setattr(_sx8lib, "_py", None)
        with pytest.warns(RuntimeWarning, match=why):
            m = _sx8lib.py()
        assert m is _sx8lib.py() and m.linear(1, 2) is None and m.to_host(None) is None
    old = ctypes.CFUNCTYPE(ctypes.c_int32)(lambda: _sx8lib.ABI_VERSION - 1)
    names = {n: ctypes.cast(getattr(hiplib, n), ctypes.c_void_p).value for n, _, _ in _sx8lib.SIGNATURES}
    with pytest.raises(RuntimeError, match="ABI version"):
        real.bind(dict(names, sx8_abi_version=ctypes.cast(old, ctypes.c_void_p).value))
    real.bind(names)


def test_bias_left_to_torch():
    """Only a bias whose sum is the kernel's fp16 addition is fused."""
    import torch.autograd.forward_ad as fwd
    from sx8_gemm_compact import _fusable_bias

    class Sub(torch.Tensor):
        pass
    cpu = torch.device("cpu")
    b = torch.randn(8).half()
    assert _fusable_bias(b, 8, cpu) and _fusable_bias(torch.nn.Parameter(b, requires_grad=False), 8, cpu)
    for bad in (b.float(), b[::2], b[:4], b[None], torch.nn.Parameter(b), b.as_subclass(Sub), torch._neg_view(b), 1.0,
                b.to("meta")):
        assert not _fusable_bias(bad, 8, cpu)
    with torch.no_grad():
        assert _fusable_bias(torch.nn.Parameter(b), 8, cpu)
    seen = []
    with fwd.dual_level():
        assert not _fusable_bias(fwd.make_dual(b, b), 8, cpu) and _fusable_bias(b, 8, cpu)
    torch.func.vmap(lambda v: (seen.append(_fusable_bias(v, 8, cpu)), v)[1])(b.expand(2, 8).contiguous())
    torch.func.jvp(lambda v: (seen.append(_fusable_bias(v, 8, cpu)), v)[1], (b,), (b,))
    assert seen == [False, False]


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 4])
def test_bias_transforms(hiplib, cuda, M):
    """Tangents, vmap, subclasses and negating views of the bias reach torch's sum."""
    import torch.autograd.forward_ad as fwd
    from integrate_fused_v44 import SX8LinearV44
    from sx8_decode1_v3 import make_tensors_v44

    class Sub(torch.Tensor):
        pass
    N, K = 96, 100
    qt, bi = _weight(N, K)
    t = make_tensors_v44(qt, bi)
    g = torch.Generator().manual_seed(9)
    x = torch.randn(M, K, generator=g).half().to(cuda)
    b, db = (torch.randn(N, generator=g).half().to(cuda) for _ in range(2))

    def f(bias, x=x):
        m = SX8LinearV44(qt, bi, bias)
        m._t44 = t
        return m(x)
    y = f(b)
    for form in (x, x.t().contiguous().t(), x.float()):          # native path, copied rows, general path
        with fwd.dual_level():
            d = fwd.unpack_dual(f(fwd.make_dual(b, db), form))
            assert torch.equal(d.tangent, db.expand(M, N)) and torch.allclose(d.primal, y, atol=1e-2)
        out = torch.func.vmap(lambda v: f(v, form))(torch.stack([b, db]))
        assert out.shape == (2, M, N) and torch.allclose(out[0], y, atol=1e-2)
        assert type(f(b.as_subclass(Sub), form)) is Sub
        assert torch.allclose(f(torch._neg_view(b), form), f(-b, form), atol=1e-2)
        assert torch.allclose(f(0.5, form), f(torch.full_like(b, 0.5), form), atol=1e-2)


@pytest.mark.gpu
@pytest.mark.parametrize("K", [40, 100])
def test_k_blocks_of_another_length(both, cuda, K):
    """A weight of three K blocks used with shorter or longer rows: one row is padded or cut as
    decode1_v44 does it, more rows are refused."""
    from integrate_fused_v44 import SX8LinearV44
    from sx8_decode1_v3 import decode1_v44, make_tensors_v44
    qt, bi = _weight(80, 96)
    t = make_tensors_v44(qt, bi)
    m = SX8LinearV44(dict(qt, shape=(80, K)), bi)
    m._t44 = t
    x = torch.randn(4, K, generator=torch.Generator().manual_seed(K)).half().to(cuda)
    y, ref, taken = both(lambda: m(x[:1]))
    _same(y, ref)
    assert "linear" not in taken and torch.equal(y[0], decode1_v44(x[0], qt, bi, *t)[0].half())
    with pytest.raises(RuntimeError, match="bad shape"):
        m(x)


@pytest.mark.gpu
def test_to_host_parts(hiplib, cuda):
    """Parts that begin and end at, before and past the 1 MB pieces, empty and overlapping ones."""
    import _sx8lib
    M = 1 << 20
    n = 3 * M + 77
    x = torch.randint(0, 256, (n,), dtype=torch.uint8, device=cuda)
    at = ((0, n), (0, 1), (M - 1, 2), (M, M), (5, 2 * M), (n - 1, 1), (n, 0), (2 * M + 3, M + 74))
    for (off, nb), y in zip(at, _sx8lib.py().to_host(x, at)):
        assert torch.equal(y, x[off:off + nb].cpu())
    assert len(_sx8lib.py().to_host(x, at)) == len(at)
    small = x[:1000]
    assert [torch.equal(y, small[a:a + 10].cpu()) for a, y in zip((0, 990), _sx8lib.py().to_host(small, ((0, 10), (990, 10))))] == [True, True]
    for bad in ((-1, 2), (0, n + 1), (n, 1)):
        with pytest.raises(ValueError):
            _sx8lib.py().to_host(x, (bad,))


@pytest.mark.gpu
@pytest.mark.parametrize("n,k", [(16, 64), (1024, 2560)])
def test_quantizer_arrays_are_their_own(hiplib, cuda, n, k):
    """No array of a quantized tensor keeps another one's memory alive."""
    from quantize_sx8 import quantize_tensor
    qt, bi = quantize_tensor((torch.randn(n, k, device=cuda) * 0.02).half())
    sizes = {}
    for name, a in list(qt.items()) + list(bi.items()):
        if isinstance(a, np.ndarray):
            root = a
            while isinstance(root.base, np.ndarray):
                root = root.base
            sizes[name] = (root.nbytes, a.nbytes)
    assert all(r == own for r, own in sizes.values()), sizes
