"""Large-row GEMMs (row bands, K-split) against the 16-row tasks, bit for bit.

A step of many rows takes the large-row kernels (from 576 rows at D = 512, 896 at
D = 256 where MLP down has four K-slices, 672 and 1024 (dense: 1152) elsewhere, 1024
without expanded copies); the same tokens in committed windows of at most 16 tokens
take the 16-row tasks.
Logits, probabilities, tables and the cache must be equal: packed weights with
and without their expanded copies and dense bf16 ones, K = 256 and 512, GQA,
parallel lanes, RoPE widths whose partner columns lie in the same lane, another
block or another lane group, natural-order caches, rows that end inside a tile,
and windows that start off a 4-key boundary.

The taller bands (64 rows), which only launches of thousands of rows take, and
window rows kept in the tail of a natural cache: every segment must equal the same
segment alone, whose window of a few hundred rows runs the 16-row tasks.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [
    # profile, overrides, dense, kv, expand, B, W, p0
    ("large", {}, True, "bf16", None, 3, 193, 0),
    ("large", {}, True, "bf16n", None, 2, 289, 0),
    ("tiny", {}, True, "bf16", None, 8, 117, 0),
    ("tiny", {"rope_dims": 32}, False, "bf16", None, 8, 117, 3),
    ("tiny", {"rope_dims": 64}, False, "bf16", False, 9, 117, 2),
    ("tiny", {"rope_dims": 24}, False, "bf16n", None, 8, 117, 0),
    ("tiny", {"rope_dims": 8, "model_dim": 512, "num_heads": 8, "num_kv_heads": 2}, False, "bf16", None, 2, 300, 1),
    ("cfg1", {}, False, "bf16", None, 15, 64, 7),
    ("cfg1", {"vocab_size": 6144}, False, "bf16", None, 14, 65, 0),
    ("cfg3", {"num_layers": 2, "xsa_last_n": 1}, False, "bf16", None, 3, 193, 5),
    # the rows from which models with other MLP-downs than K-splits take them
    ("tiny", {}, True, "bf16", None, 9, 128, 1),
    ("tiny", {"rope_dims": 32}, False, "bf16", None, 8, 128, 3),
    ("tiny", {"rope_dims": 24}, False, "bf16n", None, 9, 117, 2),
    ("cfg1", {"mlp_mult": 3.0}, False, "bf16", None, 8, 128, 0),
    ("cfg3", {"num_layers": 2, "xsa_last_n": 1, "mlp_mult": 1.5}, False, "bf16", None, 4, 168, 5),
    ("cfg3", {"num_layers": 2, "xsa_last_n": 1, "mlp_mult": 1.0}, False, "bf16", None, 4, 179, 2),
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_window_equals_short_windows(case):
    from altxs_amd import synth
    from altxs_amd.config import make_config
    from altxs_amd.model import StepModel

    prof, over, dense, kv, expand, B, W, p0 = CASES[case]
    print(f"[gpu-case] large rows {CASES[case]}", flush=True)
    cfg = make_config(prof, **over)
    model = StepModel(synth.make_model(cfg, std=0.03, softcap=(30.0, 24.0), dense=dense), act="bf16", kv=kv,
                      expand=expand)
    toks = np.random.default_rng(case).integers(0, cfg.vocab_size, (B, p0 + W)).astype(np.int32)
    L = 512

    def state(win):
        st = model.make_static_state(L, win=win, batch=B)
        for i in range(p0):  # the tokens before, one at a time
            st.tokens(1).copy_(torch.from_numpy(toks[:, i:i + 1]))
            model.step(st, commit=True, width=1)
        return st

    big = state(W)
    assert B * W >= (1024 if expand is False else 576 if cfg.model_dim == 512 else 896)
    big.tokens().copy_(torch.from_numpy(toks[:, p0:]))
    model.step(big, commit=True)
    small = state(16)
    for w0 in range(0, W, 16):
        w = min(16, W - w0)
        small.tokens(w).copy_(torch.from_numpy(toks[:, p0 + w0:p0 + w0 + w]))
        model.step(small, commit=True, width=w)
        for name in ("logits", "probs", "cum"):
            a = getattr(big, name).view(B, W, -1)[:, w0:w0 + w]
            b = getattr(small, name)[:B * w].view(B, w, -1)
            assert torch.equal(a, b), (name, w0)
    assert torch.equal(big.kv, small.kv) and torch.equal(big.prev_raw, small.prev_raw)
    big.check_errors()
    small.check_errors()


def _all(bits):
    return {f"l{i}.{k}": bits for i in range(2) for k in ("qkv", "o", "up", "down")} | {"emb": bits}


L2 = {"num_layers": 2, "xsa_last_n": 1}
TALL = [
    # profile, overrides, bits of every tensor (None: the mix, 16: dense), kv, expand, B, W, p0, kv_tail_end
    *[("cfg3", L2, b, "bf16", False, 9, 461, 3, 0) for b in (2, 3, 4, 6)],
    ("cfg3", L2, None, "bf16", None, 9, 461, 2, 0),
    ("cfg3", L2, None, "bf16", None, 18, 457, 0, 0),  # 8226 rows: 64 x 128 tiles for MLP down
    ("large", {}, 16, "bf16", None, 9, 461, 1, 0),
    ("large", {}, 16, "bf16", None, 18, 457, 0, 0),
    ("tiny", {}, 16, "bf16", None, 18, 457, 2, 0),
    *[("cfg1", {}, b, "bf16", False, 18, 457, 1, 0) for b in (2, 3, 4, 6)],
    ("cfg1", {}, None, "bf16", None, 18, 457, 0, 0),
    ("large", {}, 16, "bf16n", None, 3, 193, 5, 512),
    ("large", {}, None, "bf16n", None, 3, 195, 6, 500),
]


@pytest.mark.parametrize("case", range(len(TALL)))
def test_segments_equal_themselves_alone(case):
    from altxs_amd import synth
    from altxs_amd.config import make_config
    from altxs_amd.model import StepModel

    prof, over, bits, kv, expand, B, W, p0, tail = TALL[case]
    print(f"[gpu-case] tall bands {TALL[case]}", flush=True)
    cfg = make_config(prof, **over)
    dense = bits == 16
    model = StepModel(synth.make_model(cfg, std=0.03, softcap=(30.0, 24.0), dense=dense,
                                       bits=None if dense or bits is None else _all(bits)),
                      act="bf16", kv=kv, expand=expand)
    toks = torch.from_numpy(np.random.default_rng(case).integers(0, cfg.vocab_size, (B, W)).astype(np.int32))
    g = torch.Generator(device="cuda").manual_seed(case)
    before = torch.randn(model.n_slots, B, 2, cfg.num_kv_heads, 512, cfg.head_dim, device="cuda", generator=g).bfloat16()
    assert W < 576 <= B * W

    def run(b0, b1):
        st = model.make_static_state(512, win=W, batch=b1 - b0, kv_tail_end=tail)
        st.kv.copy_(before[:, b0:b1])
        st.pos.fill_(p0)
        st.tokens().copy_(toks[b0:b1])
        model.step(st)
        st.check_errors()
        return st

    big = run(0, B)
    for b in sorted({0, B // 2, B - 1}):
        one = run(b, b + 1)
        for name in ("logits", "probs", "cum"):
            x = getattr(big, name).view(B, W, -1)[b]
            assert torch.equal(x, getattr(one, name).view(W, -1)), (name, b)
        assert torch.equal(big.kv[:, b], one.kv[:, 0]), b
