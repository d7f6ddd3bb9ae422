"""fp32-cache attention: several rows per workgroup give a decode row's bits.

Windows whose launch still fills the chip share each K/V tile among four queries
(rows x heads); every row must equal the same row run alone, at window widths
around the row blocks, MHA and GQA, at tile edges, with XSA and the gate, and in
the tail placement.  The rows themselves are checked against float64.
"""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tail", [False, True])
@pytest.mark.parametrize("H,Hkv,W", [(8, 8, 5), (8, 8, 8), (8, 4, 3), (8, 4, 6), (4, 1, 6)])
def test_window_rows_equal_rows_alone(H, Hkv, W, tail):
    from altxs_amd import ops

    print(f"[gpu-case] fp32 attention H={H} Hkv={Hkv} W={W} tail={tail}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(100 * H + 10 * W + Hkv)
    B, L = 64, 192
    k, v = (torch.randn(B, Hkv, L, 64, device="cuda", generator=g) for _ in range(2))
    q = torch.randn(B * W, H, 64, device="cuda", generator=g) * 2
    gate = torch.rand(B * W, H, device="cuda", generator=g)
    pos = torch.arange(B, dtype=torch.int32, device="cuda") * 2  # positions 0 .. 126: tile edges inside windows
    end = L if tail else 0
    y = ops.decode_attn(q, k, v, pos, W=W, gate=gate, use_xsa=True, kv_tail_end=end)
    kk, vv = k.clone(), v.clone()
    if tail:  # the logical cache: the window's rows moved to their positions
        for b in range(B):
            p = int(pos[b])
            kk[b, :, p:p + W] = k[b, :, L - W:]
            vv[b, :, p:p + W] = v[b, :, L - W:]
    for t in range(W):
        qt = q.view(B, W, H, 64)[:, t].contiguous()
        gt = gate.view(B, W, H)[:, t].contiguous()
        alone = ops.decode_attn(qt, kk, vv, pos + t, gate=gt, use_xsa=True)
        assert torch.equal(y.view(B, W, -1)[:, t], alone)
        if t == W - 1:
            G = H // Hkv
            s = torch.einsum("bhd,bhld->bhl", qt.double(), kk.double().repeat_interleave(G, 1)) / 8
            s.masked_fill_(torch.arange(L, device="cuda")[None, None] > (pos + t)[:, None, None], float("-inf"))
            ref = torch.einsum("bhl,bhld->bhd", s.softmax(-1), vv.double().repeat_interleave(G, 1))
            cur = torch.stack([vv[b, :, int(pos[b]) + t] for b in range(B)]).double().repeat_interleave(G, 1)
            cur = cur / cur.norm(dim=-1, keepdim=True)
            ref = (ref - (ref * cur).sum(-1, keepdim=True) * cur) * gt.double()[..., None]
            # scores up to ~60 in magnitude carry 64 roundings each: exponentials within 2^-24 * 64 * 60
            assert (alone.view(B, H, 64) - ref).abs().max() < 3e-4


@pytest.mark.parametrize("W", [1, 2, 3])
def test_rows_of_large_launches_equal_small_ones(W):
    """Launches of one workgroup per CU and more keep no loads ahead, and windows of
    two rows run a row per workgroup: the same bits as single segments, from one key to
    more tiles than waves, around tile edges."""
    from altxs_amd import ops

    print(f"[gpu-case] fp32 attention large launch W={W}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(W)
    B, H, L = 40, 8, 384
    k, v = (torch.randn(B, H, L, 64, device="cuda", generator=g) for _ in range(2))
    q = torch.randn(B * W, H, 64, device="cuda", generator=g) * 2
    gate = torch.rand(B * W, H, device="cuda", generator=g)
    edges = [0, 1, 61, 62, 63, 64, 65, 126, 127, 128, 191, 192, 253, 254, 255, 256, 257, 319, 320, L - W]
    pos = torch.tensor((edges * 2)[:B], dtype=torch.int32, device="cuda")
    y = ops.decode_attn(q, k, v, pos, W=W, gate=gate, use_xsa=True).view(B, W, -1)
    for b in range(B):
        one = ops.decode_attn(q.view(B, W, H, 64)[b].contiguous(), k[b:b + 1], v[b:b + 1], pos[b:b + 1], W=W,
                              gate=gate.view(B, W, H)[b].contiguous(), use_xsa=True)
        assert torch.equal(y[b].reshape(-1), one.reshape(-1)), b
