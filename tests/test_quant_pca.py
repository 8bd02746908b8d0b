"""sx8_quant_pca (residuals, Gram matrices, eigenvectors, coefficients, medians) against
numpy on the same blocks: the residuals restated in float32 with the kernel's roundings, the
Gram matrix and its eigenvectors in float64, the coefficients from the float32 bases.  Row
counts at the edges of the Gram ranges and of the 256-row passes, K blocks at those of the
byte pass (four per thread)."""
import ctypes

import numpy as np
import pytest


def _reference(x, lv, mn, mx, cfg, n_rows, n_cb):
    f = np.float32
    r63 = f(1) / f(63)
    d = np.maximum(mx - mn, f(1e-10))
    q = d / f(4)
    w = np.maximum(d - f(2) * q, f(1e-10))
    lo = np.stack([mn, mn, mx - q, mn + q], 1)
    st = np.stack([d * r63, q * r63, q * r63, w * r63], 1)
    s = np.stack([(cfg >> (2 * i)) & 3 for i in range(4)], 1)
    lo, st = np.take_along_axis(lo, s, 1), np.take_along_axis(st, s, 1)
    rec = lo[:, :, None] + st[:, :, None] * lv.reshape(-1, 4, 8).astype(f)
    e = (x - rec.reshape(-1, 32)).reshape(n_rows, n_cb, 32).astype(np.float64)
    G = np.einsum("rci,rcj->cij", e, e)
    lam, vec = np.linalg.eigh(G)
    return e, G, lam, vec


@pytest.mark.gpu
@pytest.mark.parametrize("n_rows,n_cb,f16", [
    (4, 1, True), (5, 3, False), (32, 4, True), (63, 5, True), (64, 2, False), (65, 7, True), (255, 1, True),
    (256, 8, False), (257, 6, True), (1000, 9, True), (4099, 3, True),
])
def test_pca_against_numpy(hiplib, cuda, n_rows, n_cb, f16):
    import torch
    from quantize_sx8 import pca_correct, quantize_tensor, v6_encode_hip
    print("pca", n_rows, n_cb, f16, flush=True)
    g = torch.Generator().manual_seed(n_rows * 10 + n_cb)
    W = (torch.randn(n_rows, n_cb * 32, generator=g) * 0.02).half()
    W[1, :32] = W[1, 0]                                # a constant block
    blocks = W.reshape(-1, 32).to(cuda)
    lv, dmin, dmax, cfg, _, _ = v6_encode_hip(blocks)
    if f16:
        qt, bi = quantize_tensor(W, device=cuda)       # the fp16 form
        coeff, data, scales = qt["coeff"], bi["data"], bi["scales"]
        assert np.array_equal(qt["config"], cfg.cpu().numpy().astype(np.uint8))
    else:
        coeff, data, scales = pca_correct(lv, dmin.float(), dmax.float(), cfg, blocks.float(), n_cb, "gram")
    assert coeff.shape == (n_rows * n_cb, 1) and data.shape == (n_cb, 64) and scales.shape == (n_cb, 2)
    h = lambda t: t.cpu().numpy()
    e, G, lam, vec = _reference(h(blocks).astype(np.float32), h(lv), h(dmin).astype(np.float32),
                                h(dmax).astype(np.float32), h(cfg), n_rows, n_cb)
    for kb in range(n_cb):
        for k in range(2):
            v = data[kb, 32 * k:32 * k + 32].astype(np.float64)
            assert v[np.abs(v).argmax()] > 0
            # computed in float64, stored in float32: an eigenvector to a float32 rounding, of the
            # right eigenvalue, and numpy's vector up to sign where the gap resolves it
            assert abs(v @ v - 1) <= 1e-6
            assert np.abs(G[kb] @ v - lam[kb, -1 - k] * v).max() <= 1e-6 * lam[kb, -1]
            others = np.delete(lam[kb], 31 - k)
            gap = np.abs(others - lam[kb, -1 - k]).min() / lam[kb, -1]
            if gap > 1e-6:
                u = vec[kb][:, -1 - k]
                assert min(np.abs(v - u).max(), np.abs(v + u).max()) <= 1e-6 + 1e-12 / gap
            c = (e[:, kb] @ v).astype(np.float32)
            sc = max(np.sort(np.abs(c))[(n_rows - 1) // 2] / np.float32(3), np.float32(1e-10))
            assert abs(scales[kb, k] - sc) <= 1e-6 * sc
            ratio = c / scales[kb, k]
            want = np.clip(np.rint(ratio), -8, 7).astype(int)
            byte = coeff.reshape(n_rows, n_cb)[:, kb]
            got = ((byte >> (4 * k)) & 15).astype(int)
            got = np.where(got > 7, got - 16, got)
            tie = np.abs(np.abs(ratio - np.floor(ratio)) - 0.5) < 1e-4   # c differs in its last bit
            assert (got == want)[~tie].all()


@pytest.mark.gpu
def test_pca_not_finite_takes_general_path(hiplib, cuda):
    """Weights with an infinity keep the torch path's outcome (whatever it is), not zeros."""
    import torch
    from quantize_sx8 import _HostFields, _pca_hip, v6_encode_hip
    W = (torch.randn(64, 64, generator=torch.Generator().manual_seed(1)) * 0.02).half().to(cuda)
    W[3, 40] = float("inf")
    blocks = W.reshape(-1, 32)
    lv, dmin, dmax, cfg, _, _ = v6_encode_hip(blocks)
    out = _HostFields(128, 2, W.device)
    _pca_hip(lv, dmin, dmax, cfg, blocks, 64, 2, out)
    assert out.to_host() is None


def test_pca_refusals(hiplib):
    L, p, N0 = hiplib, ctypes.c_void_p(4096), ctypes.c_void_p(None)
    assert L.sx8_quant_pca_workspace_bytes(0, 4) == -1 and L.sx8_quant_pca_workspace_bytes(1 << 37, 4) == -1
    need = L.sx8_quant_pca_workspace_bytes(64, 4)
    call = lambda **k: L.sx8_quant_pca(k.get("x", p), p, p, 1, p, p, k.get("r", 64), 4, p, p, p, k.get("ws", p),
                                       k.get("nb", need), N0)
    assert call(x=N0) == 1 and call(ws=N0) == 1 and call(nb=need - 1) == 1 and call(r=0) == 1
    assert call(x=ctypes.c_void_p(4097)) == 1 and call(ws=ctypes.c_void_p(4104)) == 1
    assert b"misaligned" in L.sx8_last_error()
    big = L.sx8_quant_pca_workspace_bytes(4, 65536)               # one K block past the kernels' grids
    assert L.sx8_quant_pca(p, p, p, 1, p, p, 4, 65536, p, p, p, p, big, N0) == 3


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["zero", "rank1", "rank2_1e-5", "identity", "tiny_identity", "gap_2e-6", "gap_1e-7",
                                  "equal_pair", "large"])
def test_pca_spectra(hiplib, cuda, kind):
    """Residuals with chosen Gram spectra (levels and ranges of zero: the residual is the block):
    unit, orthogonal vectors, each an eigenvector of its eigenvalue, whatever the gaps; the
    subspace of the two where their common gap resolves it."""
    import torch
    from quantize_sx8 import pca_correct
    rng = np.random.default_rng(7)
    Q = np.linalg.qr(rng.standard_normal((32, 32)))[0]
    tail = np.linspace(0.5, 0.1, 30)
    s = {"zero": np.zeros(32), "rank1": np.r_[1, np.zeros(31)], "rank2_1e-5": np.r_[1, 1e-5, np.zeros(30)],
         "identity": np.ones(32), "tiny_identity": np.ones(32) * 1e-18, "gap_2e-6": np.r_[1, 1 - 1e-6, tail],
         "gap_1e-7": np.r_[1, 1 - 6e-8, tail], "equal_pair": np.r_[1, 1, tail], "large": np.r_[1, .9, tail] * 1e15}[kind]
    E = (s[:, None] * (np.eye(32) if "identity" in kind else Q)).astype(np.float32)
    z = torch.zeros(32, device=cuda)
    _, data, _ = pca_correct(torch.zeros(32, 32, dtype=torch.uint8, device=cuda), z, z, z.int(),
                             torch.from_numpy(E).to(cuda), 1, "gram")
    G = E.astype(np.float64).T @ E.astype(np.float64)
    lam, vec = np.linalg.eigh(G)
    v = data.reshape(2, 32).astype(np.float64)
    assert np.abs(v @ v.T - np.eye(2)).max() <= 1e-6           # float32 storage: 32 2^-24 at most
    for k in range(2):
        assert np.abs(G @ v[k] - lam[-1 - k] * v[k]).max() <= 1e-6 * lam[-1]
        assert v[k][np.abs(v[k]).argmax()] >= 0
    if (lam[-2] - lam[-3]) > 1e-3 * lam[-1]:
        U = vec[:, -2:]
        assert np.abs(v - v @ U @ U.T).max() <= 1e-6


def _fields(n_rows, n_cb, device):
    import torch
    from quantize_sx8 import v6_encode_6bit
    blocks = (torch.randn(n_rows * n_cb, 32, generator=torch.Generator().manual_seed(3)) * 0.02).half().float()
    return [t.to(device) for t in (*v6_encode_6bit(blocks), blocks)]


def test_pca_forms_left_to_torch():
    """The kernels read raw pointers: only the exact types, shapes and one device go there."""
    import torch
    from quantize_sx8 import _pca_plain
    lv, mn, mx, cfg, x = _fields(8, 3, "cpu")
    assert _pca_plain(lv, mn, mx, cfg, x, 3) and _pca_plain(lv, mn, mx, cfg.to(torch.uint8), x.half(), 3)
    for bad in ((lv.int(), mn, mx, cfg, x, 3), (lv.float(), mn, mx, cfg, x, 3), (lv.to("meta"), mn, mx, cfg, x, 3),
                (lv, mn.to("meta"), mx, cfg, x, 3), (lv, mn, mx, cfg.to("meta"), x, 3), (lv, mn.half(), mx.half(), cfg, x, 3),
                (lv, mn.double(), mx, cfg, x, 3), (lv, mn, mx, cfg.float(), x, 3), (lv, mn, mx, cfg, x.double(), 3),
                (lv, mn, mx, cfg, x, 5), (lv[:-1], mn, mx, cfg, x, 3), (lv.view(-1, 16), mn, mx, cfg, x, 3),
                (lv, mn[:-1], mx, cfg, x, 3), (lv, mn, mx, cfg[:-1], x, 3), (lv, mn, mx, cfg, x[:, :16], 3),
                (lv, mn[:, None], mx, cfg, x, 3), (lv, mn, mx, cfg, x.clone().requires_grad_(), 3)):
        assert not _pca_plain(*bad)


@pytest.mark.gpu
def test_pca_other_forms(hiplib, cuda):
    """Levels and fields of other types give what uint8 levels and float32 fields give; host
    levels, uneven block counts and short fields raise on the host."""
    import torch
    from quantize_sx8 import pca_correct
    n_rows, n_cb = 64, 3
    lv, mn, mx, cfg, x = _fields(n_rows, n_cb, cuda)
    want = pca_correct(lv, mn, mx, cfg, x, n_cb, "gram")
    for f in ((lv.int(), mn, mx, cfg, x), (lv.float(), mn, mx, cfg, x), (lv, mn, mx, cfg.cpu(), x),
              (lv, torch.cat([mn, mn]), torch.cat([mx, mx]), cfg, x)):
        got = pca_correct(*f, n_cb, "gram")
        # the same residuals, float64 Gram matrices on both sides; the coefficients are float32 sums of 32
        assert np.abs(got[1] - want[1]).max() <= 1e-6 and np.abs(got[2] / want[2] - 1).max() <= 1e-5
        assert (got[0] != want[0]).mean() <= 1e-2          # coefficients on a rounding tie
    with pytest.raises(RuntimeError):
        pca_correct(lv.cpu(), mn, mx, cfg, x, n_cb, "gram")
    with pytest.raises(RuntimeError):
        pca_correct(lv, mn.cpu(), mx.cpu(), cfg, x, n_cb, "gram")
    with pytest.raises(RuntimeError):
        pca_correct(lv, mn, mx, cfg, x, 5, "gram")
    with pytest.raises(IndexError):
        pca_correct(lv, mn[:-1], mx, cfg, x, n_cb, "gram")
    with pytest.raises((RuntimeError, IndexError)):
        pca_correct(lv, mn, mx, cfg[:-1], x, n_cb, "gram")
    with pytest.raises(RuntimeError):
        pca_correct(lv[:-1], mn, mx, cfg, x, n_cb, "gram")


@pytest.mark.gpu
def test_pca_past_the_kernels_sizes(hiplib, cuda, monkeypatch):
    """Where sx8_quant_pca reports a tensor too large, both callers take torch's path."""
    import torch
    import _sx8lib
    from quantize_sx8 import pca_correct, quantize_tensor
    W = (torch.randn(64, 96, generator=torch.Generator().manual_seed(2)) * 0.02).half().to(cuda)
    qt, bi = quantize_tensor(W)
    f = _fields(64, 3, cuda)
    want = pca_correct(*f, 3, "gram")

    class Small:
        def __getattr__(self, name):
            return (lambda *a: _sx8lib.ERR_UNSUPPORTED) if name == "sx8_quant_pca" else getattr(hiplib, name)
    monkeypatch.setattr(_sx8lib, "_lib", Small())
    q2, b2 = quantize_tensor(W)
    got = pca_correct(*f, 3, "gram")
    for k in ("dmin", "dmax", "config", "levels_hi", "levels_lo"):
        assert np.array_equal(qt[k], q2[k])
    for a, b in ((bi["data"], b2["data"]), (want[1], got[1])):
        assert np.abs(a - b).max() <= 1e-6
    assert (qt["coeff"] != q2["coeff"]).mean() <= 1e-2 and (want[0] != got[0]).mean() <= 1e-2
