"""Decode attention over caches longer than 2048 positions, where the position range is split
into more chunks (16, 32 or 64 by the number of KV heads): positions at the edges of the 64-
position passes and chunks, the first and last of the cache, against float32 attention, and
with a workspace that only holds 16 chunks' partials."""
import math

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh,nk,hd,L", [
    (32, 8, 128, 2049),      # 32 chunks
    (32, 4, 128, 5000),      # 64 chunks, G = 8
    (8, 2, 128, 2500),       # 64 chunks
    (16, 16, 64, 2600),      # 16 chunks, G = 1
    (4, 4, 64, 4500),        # 64 chunks, G = 1
])
def test_long_cache_chunks(hiplib, cuda, nh, nk, hd, L):
    import torch
    import _sx8lib as _L
    P = _L.ptr
    g = torch.Generator().manual_seed(L)
    q, kc, vc = (torch.randn(*s, generator=g).half().to(cuda) for s in ((nh, hd), (nk, L, hd), (nk, L, hd)))
    scale = 1.0 / math.sqrt(hd)
    full = int(_L.lib().sx8_dec_attn_workspace_bytes(nh, hd))
    small = nh * 16 * (hd + 2) * 4
    assert full >= small
    for pos in [0, 63, 64, 127, 640, 2047, 2048, L - 2, L - 1]:
        print("long attention", nh, nk, hd, L, pos, flush=True)
        pt = torch.tensor([pos], dtype=torch.int64, device=cuda)
        s = torch.einsum("hd,hnd->hn", q.float().cpu(), kc[:, :pos + 1].float().cpu().repeat_interleave(nh // nk, 0))
        ref = torch.einsum("hn,hnd->hd", torch.softmax(s * scale, 1),
                           vc[:, :pos + 1].float().cpu().repeat_interleave(nh // nk, 0))
        for nb in (full, small):
            ws = torch.full((nb // 4,), float("nan"), device=cuda)       # needs no clearing
            out = torch.empty(nh, hd, dtype=torch.float16, device=cuda)
            _L.call("sx8_dec_attn_split", P(q), P(kc), P(vc), P(pt), P(out), nh, nk, hd, L, scale, P(ws), nb,
                    _L.stream(cuda))
            # fp16 output and probabilities' float32 sums: the bar of the shorter caches' test
            err = (out.cpu().float() - ref).abs().max().item()
            assert err <= 2e-3 * max(1.0, ref.abs().max().item()), (pos, nb, err)
    with pytest.raises(RuntimeError, match="workspace"):
        _L.call("sx8_dec_attn_split", P(q), P(kc), P(vc), P(pt), P(out), nh, nk, hd, L, scale, P(ws), small - 4,
                _L.stream(cuda))
