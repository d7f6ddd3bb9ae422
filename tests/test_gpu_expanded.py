"""Expanded weight values (altxs_expand_codes, AltxsQTensor.expanded).

* The expanded buffer equals the numpy tiler's bits-16 layout of the values
  code - (2^b - 1)/2 (codec.PackedTensor.from_dense at bits 16 on those
  values) with each block's (lane, k-step) operands transposed to k-step
  order, byte for byte, for every packed width.
* Steps of many rows read the expanded values in their QKV, out-projection and
  MLP-up row bands and in the MLP-down K-split (F = 2048) or row band (F = 512);
  the LM head stays packed.  The same windows with and without the expanded
  copies give the same logits, probabilities and tables bit for bit (the
  row-count tests in tests/test_gpu_step.py compare them with the 16-row GEMMs
  as well).
* Copies are made for exactly the tensors that some step reads, from the row
  count at which one does: a step changes when any of its copies does.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _log(msg: str) -> None:
    print(f"[gpu-case] {msg}", flush=True)


@pytest.mark.parametrize("bits", [2, 3, 4, 6])
def test_expand_codes_matches_tiled_values(bits):
    from altxs_amd import _lib, ops
    from altxs_amd.codec import PackedTensor

    _log(f"expand codes bits={bits}")
    n, k = 48, 768
    rng = np.random.default_rng(bits)
    p = PackedTensor.from_dense("w", rng.standard_normal((n, k)).astype(np.float32) * 0.02, bits)
    w = ops.DeviceQTensor(p)
    out = torch.empty(n * k, dtype=torch.bfloat16, device="cuda")
    L = _lib.load()
    _lib.check(L.altxs_expand_codes(ctypes.byref(w.qt), out.data_ptr(),
                                    ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)),
               "altxs_expand_codes")
    vals = p.codes.astype(np.float32) - np.float32(((1 << bits) - 1) / 2)
    # bits-16 tiles hold lane l's eight 16-byte k-step operands together; the
    # expanded blocks hold k-step s's 64 lane operands together
    t16 = np.asarray(PackedTensor.from_dense("e", vals, 16).tiled).view(np.uint8).reshape(-1, 64, 8, 16)
    want = t16.transpose(0, 2, 1, 3).reshape(-1)
    got = out.cpu().view(torch.int16).numpy().view(np.uint8)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("profile", ["cfg4", "tiny512"])
def test_windows_expanded_equal_packed(profile):
    from altxs_amd import synth
    from altxs_amd.config import make_config
    from altxs_amd.model import StepModel

    _log(f"expanded vs packed large tiles: {profile}")
    cfg = (make_config("tiny", model_dim=512, num_heads=8, num_kv_heads=4) if profile == "tiny512"
           else make_config(profile))
    sm = synth.make_model(cfg, std=0.02, softcap=(30.0, 24.0))
    B, T, L = 3, 361, 512
    toks = torch.from_numpy(np.random.default_rng(13).integers(0, cfg.vocab_size, (B, T)).astype(np.int32))
    out = []
    for expand in (False, True):
        model = StepModel(sm, act="bf16", expand=expand)
        assert model._expanded == expand
        st = model.make_static_state(L, win=T, batch=B, want_probs=True)
        st.token.copy_(toks)
        model.step(st)
        torch.cuda.synchronize()
        st.check_errors()
        out.append((st.logits.cpu(), st.probs.cpu(), st.cum.cpu()))
    for a, b in zip(*out):
        assert torch.equal(a, b)


@pytest.mark.parametrize("d,F,rows,down", [(512, 512, 672, True), (256, 512, 1024, True), (256, 256, 1024, True),
                                           (512, 2048, 576, True), (256, 1024, 896, True),
                                           (512, 768, 672, False), (256, 1536, 1024, False)])
def test_every_copy_is_read(d, F, rows, down):
    from altxs_amd import synth
    from altxs_amd.config import make_config
    from altxs_amd.model import StepModel

    _log(f"copies read: d={d} F={F} rows={rows}")
    cfg = make_config("cfg1", model_dim=d, num_heads=d // 64, num_kv_heads=d // 64, mlp_mult=F / d)
    model = StepModel(synth.make_model(cfg, std=0.02, softcap=(30.0, 24.0)), act="bf16")
    W = 16
    model.make_static_state(256, win=W, batch=rows // W - 1)
    assert not any(qt.expanded for qt in model.qt.values())  # a window below the line: none made
    st = model.make_static_state(256, win=W, batch=rows // W)
    names = {n for n, qt in model.qt.items() if qt.expanded}
    stages = ("qkv", "o", "up") + (("down",) if down else ())
    assert names == {f"l{i}.{k}" for i in range(cfg.num_layers) for k in stages}
    st.token.copy_(torch.arange(rows, dtype=torch.int32).view(-1, W) % cfg.vocab_size)

    def logits():
        st._descs.clear()  # (a descriptor holds the tensors' pointers)
        model.step(st)
        st.check_errors()
        return st.logits.clone()

    want = logits()
    for n in sorted(names):
        qt = model.qt[n]
        kept = qt.expanded
        other = torch.ones(qt.N * qt.K, dtype=torch.bfloat16, device="cuda")
        qt.expanded = other.data_ptr()
        assert not torch.equal(logits(), want), n
        qt.expanded = kept
    assert torch.equal(logits(), want)
