"""The wave-per-four-rows dequant and row gather, on both sides of the rule that picks it: bit for
bit the oracle's R64 weights with a last quad of one to three rows, a last 16-block column group
that is not full, outputs whose rows are not a multiple of 8 values or off 16 bytes, both header
widths, rows in order from both layouts, and row numbers outside the table (their output rows stay
as they are)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _quantized(N, K, seed, cuda):
    import torch
    from quantize_sx8 import quantize_tensor
    g = torch.Generator(device="cpu").manual_seed(seed)
    W = (torch.randn(N, K, generator=g) * 0.02).half()
    return quantize_tensor(W, device=cuda, degenerate_frac=0.01, seed=seed + 1)


@pytest.mark.parametrize("N,K", [(3281, 2560), (3283, 2557), (8195, 1000), (16386, 512), (3683, 2560), (3731, 2504),
                                 (18402, 512), (9205, 1024), (5003, 1664)])
def test_whole_tensor(hiplib, oracle, cuda, N, K):
    from kernel_sx8_v43 import decode_tensor_gpu_fast
    print("dequant", N, K, flush=True)
    qt, bi = _quantized(N, K, N, cuda)
    got = decode_tensor_gpu_fast(qt, bi)
    assert np.array_equal(got.cpu().numpy().view(np.uint16), oracle.dequant_r64(qt, bi).view(np.uint16))


@pytest.mark.parametrize("T,N,K,hb", [(3301, 700, 2560, 6), (3302, 515, 2555, 8), (4100, 129, 2048, 6), (4097, 130, 2024, 8),
                                      (16402, 129, 2888, 8)])
def test_row_gather(hiplib, oracle, cuda, T, N, K, hb):
    import torch
    from sx8_decode1_v3 import make_tensors_v44
    from sx8_embed_v44 import ext
    print("gather", T, N, K, hb, flush=True)
    qt, bi = _quantized(N, K, T, cuda)
    t = make_tensors_v44(qt, bi, hdr_aligned=(hb == 8))
    ids = torch.randint(-3, N + 3, (T,), generator=torch.Generator().manual_seed(T))
    out = torch.full((T, K), 7.0, dtype=torch.float16, device=cuda)
    ext().sx8_embed_v44(ids.to(cuda), *t, K, N, qt["n_cb"], out)
    W = oracle.dequant_r64(qt, bi)
    ok = ((ids >= 0) & (ids < N)).numpy()
    got = out.cpu().numpy()
    assert ok.any() and not ok.all()
    assert np.array_equal(got[ok].view(np.uint16), W[ids.numpy()[ok]].view(np.uint16))
    assert (got[~ok] == 7.0).all()


@pytest.mark.parametrize("N,K,hb", [(3301, 2560, 6), (4098, 1664, 8), (3303, 2504, 8), (3303, 2501, 6)])
@pytest.mark.parametrize("off", [0, 1])
def test_rows_in_order_v44(hiplib, oracle, cuda, N, K, hb, off):
    import torch
    import _sx8lib as L
    from sx8_decode1_v3 import make_tensors_v44
    print("in order", N, K, hb, off, flush=True)
    qt, bi = _quantized(N, K, N, cuda)
    t = make_tensors_v44(qt, bi, hdr_aligned=(hb == 8))
    buf = torch.full((N * K + 8,), 7.0, dtype=torch.float16, device=cuda)
    out = buf[off:off + N * K]
    L.call("sx8_embed_gather", None, 0, L.ptr(t[0]), L.ptr(t[1]), hb, L.ptr(t[2]), L.ptr(t[3]), K, N, qt["n_cb"],
           L.ptr(out), L.stream(cuda))
    assert np.array_equal(out.view(N, K).cpu().numpy().view(np.uint16), oracle.dequant_r64(qt, bi).view(np.uint16))
    assert (buf[:off] == 7.0).all() and (buf[off + N * K:] == 7.0).all()
