"""Edges of the coder's table and encode kernels.

* Softmax / count tables at vocabularies around the row exchange's bounds (1, 2,
  4, ... 64 elements per thread; remainders; rows whose start is not 16-byte
  aligned): probabilities against float64 within a few float32 roundings, the
  table exactly the count rule on them, neighbouring rows untouched.
* The renormalised row against numpy's own float32 division by numpy's sum, also at
  every length where its summation tree gets another level.
* The one-wave encoder against the oracle's bytes at window widths around its 64
  symbols, with intervals of one count (long bit runs), of a whole table but one
  (E3 runs) and totals from 2 to 2^30.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [1, 63, 1023, 1025, 2047, 2049, 4095, 4097, 8191, 8193, 16383, 16385, 32769, 65536])
def test_tables_at_exchange_bounds(V):
    from altxs_amd import ops
    from oracle import coder

    print(f"[gpu-case] tables V={V}", flush=True)
    rng = np.random.default_rng(V)
    lg = (rng.standard_normal((3, V)) * 4).astype(np.float32)
    probs, cum = ops.softmax_cdf(torch.from_numpy(lg).cuda())
    p = probs.cpu().numpy()
    x = lg.astype(np.float64)
    ref = np.exp(x - x.max(1, keepdims=True))
    ref /= ref.sum(1, keepdims=True)
    # exponential, sum of V terms in a tree over runs of <= 64, quotient
    assert np.all(np.abs(p - ref) <= 90 * 2.0 ** -24 * ref + 1e-38)
    assert np.array_equal(cum.cpu().numpy().astype(np.int64), coder.scale_cum(p))
    got = ops.scale_cum(probs)
    assert torch.equal(got, cum)
    if V <= 16384:
        pr, _ = ops.softmax_cdf(torch.from_numpy(lg).cuda(), renorm=True)
        want = np.stack([r / np.float32(float(r.sum())) for r in p])
        assert np.array_equal(pr.cpu().numpy(), want)


@pytest.mark.parametrize("lo,hi", [(1, 20), (121, 145), (249, 275), (505, 535), (1017, 1042), (2040, 2065),
                                   (4088, 4112), (8180, 8202)])
def test_renormalised_rows_at_tree_levels(lo, hi):
    """Every level of numpy's summation tree begins a few lengths past a power of two."""
    from altxs_amd import ops

    print(f"[gpu-case] renorm V={lo}..{hi}", flush=True)
    for V in range(lo, hi):
        lg = (np.random.default_rng(V).standard_normal((5, V)) * 3).astype(np.float32)
        x = torch.from_numpy(lg).cuda()
        p = ops.softmax_cdf(x)[0].cpu().numpy()
        want = np.stack([r / np.float32(float(r.sum())) for r in p])
        assert np.array_equal(ops.softmax_cdf(x, renorm=True)[0].cpu().numpy(), want), V


@pytest.mark.parametrize("W", [1, 5, 63, 64, 65, 130])
@pytest.mark.parametrize("V", [2, 300])
def test_encoder_matches_oracle_bytes(W, V):
    from altxs_amd.coder import RangeCoder
    from oracle import coder

    print(f"[gpu-case] encoder W={W} V={V}", flush=True)
    rng = np.random.default_rng(1000 * W + V)
    n, calls = 3, 3
    rc = RangeCoder(n, 64 + 5 * W * calls)
    cums, syms = [[] for _ in range(n)], [[] for _ in range(n)]
    for _ in range(calls):
        cum = np.zeros((n, W, V + 1), dtype=np.int64)
        sym = rng.integers(0, V, (n, W))
        for b in range(n):
            for t in range(W):
                f = np.ones(V, dtype=np.int64)
                kind = rng.integers(0, 4)
                if kind == 1:  # the symbol has all but V - 1 of the largest total
                    f[sym[b, t]] = (1 << 30) - V + 1
                elif kind == 2:  # one count of the largest total
                    f[(sym[b, t] + 1) % V] = (1 << 30) - V + 1
                elif kind == 3:
                    f = rng.integers(1, 4000, V)
                cum[b, t, 1:] = np.cumsum(f)
        rc.encode(torch.from_numpy(cum.reshape(n * W, V + 1).astype(np.int32)).cuda(),
                  torch.from_numpy(sym.astype(np.int32)).cuda())
        for b in range(n):
            cums[b] += list(cum[b])
            syms[b] += list(sym[b])
    got = rc.finish()
    for b in range(n):
        assert got[b] == coder.wnc_encode(np.array(syms[b]), np.stack(cums[b]))


@pytest.mark.parametrize("n", [8191, 8192, 8193, 8255])
def test_many_streams_equal_few(n):
    """From 8192 streams a lane codes each (before, a wave): the same states and bytes."""
    from altxs_amd.coder import RangeCoder

    print(f"[gpu-case] encoder streams={n}", flush=True)
    rng = np.random.default_rng(n)
    V, W, calls, k = 17, 3, 9, 64  # k of the streams, again a wave each
    many, few = RangeCoder(n, 40), RangeCoder(k, 40)  # (40 bytes: some streams run full)
    pick = torch.from_numpy(np.sort(rng.choice(n, k, replace=False))).cuda()
    pick[-1] = n - 1
    for c in range(calls):
        f = rng.integers(1, 3000, (n, W, V))
        f[:, 1, 3] = (1 << 30) - 60000  # (17 x 3000 at most beside it)
        f[::2, 2, 5] = 1 << 29
        cum = np.zeros((n, W, V + 1), dtype=np.int64)
        cum[..., 1:] = np.cumsum(f, axis=-1)
        sym = rng.integers(0, V, (n, W))
        sym[1::7, 0] = np.where(c == 4, V, sym[1::7, 0])  # a symbol out of range: flagged, not coded
        cum = torch.from_numpy(cum.astype(np.int32)).cuda()
        sym = torch.from_numpy(sym.astype(np.int32)).cuda()
        many.encode(cum.view(n * W, V + 1), sym)
        few.encode(cum[pick].reshape(k * W, V + 1).contiguous(), sym[pick].contiguous())
    assert torch.equal(many.state[pick], few.state) and torch.equal(many.buf[pick], few.buf)
