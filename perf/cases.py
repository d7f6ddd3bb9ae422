"""The work this framework is timed on: what a user of it has it do.

* Model steps (``kind = "step"``): one call of ``StepModel.static_extend`` on a
  state with a filled KV cache -- decode rows (W = 1), teacher-forced encode
  windows (W > 1), and chunk scoring (a window from position 0).  The mixed-bit
  "cfg3" model (10 layers, d = 512, V = 16384) is the production-scale
  configuration of the benchmark; "large" with dense bf16 weights is the
  shipped student (17 slots, GQA, parallel lanes, V = 256), whose cache keeps
  the reference's natural order; "cfg5" adds the rank-16 q/v adapters.
* ``softmax_cdf``: the coder's integer tables from logits a caller holds.
* ``qgemm`` / ``qgemv`` streams: products with packed 2/3/4/6-bit matrices.
* ``compress``: the engine's whole call -- context prefill, windows and range
  coder for a batch of segments, to payload bytes.

Whole numbers (CDF tables, payload bytes) have to stay the same: an encoder and
a decoder of different builds must form the same tables.
"""

from __future__ import annotations

import functools
import math

import numpy as np
import torch

from altxs_amd import ops, synth
from altxs_amd.codec import tile_kv
from altxs_amd.config import make_config
from altxs_amd.engine import StaticACEngine, encode_segments_gpu
from altxs_amd.model import StepModel

DEV = "cuda"


def _step(name, profile, act, kv, B, W, ctx, graph=False):
    """ctx: tokens already in the cache of every segment."""
    return {"name": name, "kind": "step", "profile": profile, "act": act, "kv": kv, "B": B, "W": W,
            "ctx": ctx, "graph": graph}


def listed():
    return [
        # one segment decoding, the reference's production regime; the step is
        # replayed as a graph, as the reference captures it
        _step("decode_b1", "cfg3", "bf16", "bf16", 1, 1, 2047, graph=True),
        # the benchmark's decode step
        _step("decode_b64", "cfg3", "bf16", "bf16", 64, 1, 2047),
        # fp32 compute mode (logits within 2e-3 of the fp32 model), fp32 cache
        _step("decode_fp32_b16", "cfg3", "fp32", "fp32", 16, 1, 1000),
        # the shipped student's shape, a few segments, natural-order cache
        _step("student_b7", "large", "bf16", "bf16n", 7, 1, 1501),
        # steady-state encoding: 16-token windows at the end of the context
        _step("encode_w16_b64", "cfg3", "bf16", "bf16", 64, 16, 2032),
        # encoding with few segments and an odd window
        _step("encode_w37_b5", "cfg3", "bf16", "bf16", 5, 37, 777),
        # chunk scoring: whole 2048-token chunks from position 0
        _step("prefill_b16", "cfg3", "bf16", "bf16", 16, 2048, 0),
        # chunk scoring in the fp32 compute mode, a ragged length
        _step("prefill_fp32_b2", "cfg3", "fp32", "fp32", 2, 700, 0),
        # coder tables from logits, a full production vocabulary
        {"name": "softmax_cdf", "kind": "softmax_cdf", "rows": 1024, "V": 16384},
        # packed products, batch 1 (a stream of distinct matrices) and batch 64
        {"name": "qgemv_b1", "kind": "qgemm", "rows": 1, "N": 512, "K": 2048, "bits": 3, "count": 1024},
        {"name": "qgemm_b64", "kind": "qgemm", "rows": 64, "N": 2048, "K": 512, "bits": 4, "count": 256},
        # compressing a batch of segments: 512 tokens of context, 300 symbols
        {"name": "compress_b16", "kind": "compress", "profile": "cfg3", "B": 16, "win": 64, "ctx": 512, "n": 300},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "encode", "encode", "prefill", "prefill", "softmax_cdf", "qgemm",
                       "qgemm", "compress"])
    if kind in ("decode", "encode", "prefill"):
        profile = rng.choice(["cfg3", "cfg3", "cfg5", "large"])
        fp32 = rng.random() < 0.25
        if fp32:
            act, kv = "fp32", rng.choice(["fp32", "bf16"])
        else:
            act, kv = "bf16", "bf16n" if profile == "large" and rng.random() < 0.5 else "bf16"
        if kind == "decode":
            B, W, ctx = _log(rng, 1, 64), 1, _log(rng, 16, 2047)
        elif kind == "encode":
            B = _log(rng, 1, 64)
            W = _log(rng, 2, max(2, min(256, (512 if kv != "bf16" else 4096) // B)))
            ctx = _log(rng, 16, 2048 - W)
        else:
            W = _log(rng, 64, 700 if kv != "bf16" else 2048)
            B = _log(rng, 1, max(1, (1400 if fp32 or kv != "bf16" else 32768) // W))
            ctx = 0
        c = _step("", profile, act, kv, B, W, ctx, graph=kind == "decode" and rng.random() < 0.5)
    elif kind == "softmax_cdf":
        V = rng.choice([256, 4096, 16384, _log(rng, 200, 50000)])
        c = {"kind": kind, "rows": _log(rng, 1, max(1, (1 << 24) // V)), "V": V}
    elif kind == "qgemm":
        N, K = rng.choice([(512, 2048), (2048, 512), (1536, 512), (512, 512)])
        rows = rng.choice([1, 1, 64, _log(rng, 2, 512)])
        c = {"kind": kind, "rows": rows, "N": N, "K": K, "bits": rng.choice([2, 3, 4, 6]),
             "count": _log(rng, 1, max(1, 1024 // max(1, rows // 16)))}
    else:
        c = {"kind": kind, "profile": rng.choice(["cfg3", "cfg1"]), "B": _log(rng, 1, 24),
             "win": rng.choice([16, 64, _log(rng, 8, 96)]), "ctx": _log(rng, 32, 512), "n": _log(rng, 16, 200)}
    c.pop("name", None)
    return c


# ---- what a program keeps: packed weights, the model ---------------------------


@functools.lru_cache(maxsize=None)
def _weights(profile):
    return synth.make_model(make_config(profile), std=0.02, softcap=(30.0, 24.0), dense=profile == "large")


@functools.lru_cache(maxsize=None)
def _model(profile, act, kv):
    return StepModel(_weights(profile), act=act, kv=kv)


def _gen(seed, salt=0):
    return torch.Generator(device=DEV).manual_seed(1000003 * salt + seed)


def _max_len(case):
    return (case["ctx"] + case["W"] + 255) // 256 * 256


def _kv_rows(case, cfg, seed, slot):
    """K and V of the tokens already in one slot's cache, natural order:
    [B, 2, Hkv, ctx, 64].  Keys are RMS-normalised rows, so unit variance."""
    dt = torch.float32 if case["kv"] == "fp32" else torch.bfloat16
    return torch.randn(case["B"], 2, cfg.num_kv_heads, case["ctx"], cfg.head_dim, device=DEV,
                       generator=_gen(seed, slot + 1)).to(dt)


def _tokens(case, cfg, seed):
    """Zipf(1.1) token ids [B, W], and the previous tokens [B]."""
    t = synth.zipf_tokens(cfg.vocab_size, (case["B"], case["W"] + 1), seed=seed)
    return t[:, 1:], t[:, 0]


def _packed_stream(case, seed):
    """count matrices of uniform random codes (tiled byte order) and fp16 group scales, and x."""
    g = _gen(seed, 91)
    N, K, b, c = case["N"], case["K"], case["bits"], case["count"]
    codes = torch.randint(0, 1 << 62, (c * N * K * b // 64,), dtype=torch.int64, device=DEV, generator=g)
    codes = codes ^ (torch.randint(0, 4, codes.shape, dtype=torch.int64, device=DEV, generator=g) << 62)
    scales = (torch.rand(c * N * K // 64, device=DEV, generator=g) * 0.02 + 0.005).half()
    x = torch.randn(case["rows"], K, device=DEV, generator=g).half()
    return codes.view(torch.uint8), scales, x


def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        model = _model(case["profile"], case["act"], case["kv"])
        cfg, ctx = model.cfg, case["ctx"]
        st = model.make_static_state(_max_len(case), win=case["W"], batch=case["B"], want_probs=False)
        toks, prev = _tokens(case, cfg, seed)
        st.token.copy_(torch.from_numpy(toks.astype(np.int32)))
        st.pos.fill_(ctx)
        if ctx:
            emb = torch.from_numpy(_weights(case["profile"]).packed["emb"].dense()[prev])
            st.prev_raw.copy_(emb)
            pad = (ctx + 63) // 64 * 64  # whole cache tiles
            for s in range(model.n_slots):
                kv = _kv_rows(case, cfg, seed, s)
                dst = st.kv[s]
                if case["kv"] == "bf16":
                    kv = torch.nn.functional.pad(kv, (0, 0, 0, pad - ctx))
                    dst[:, 0, :, :pad] = tile_kv(kv[:, 0], "k")
                    dst[:, 1, :, :pad] = tile_kv(kv[:, 1], "v")
                else:
                    dst[:, :, :, :ctx] = kv
        graph = None
        if case["graph"]:
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                model.static_extend(st)
            torch.cuda.current_stream().wait_stream(side)
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                model.static_extend(st)
        return kind, model, st, graph
    if kind == "softmax_cdf":
        # logits of the softcapped head: a peaked row now and then
        g = _gen(seed, 92)
        x = torch.randn(case["rows"], case["V"], device=DEV, generator=g) * 2.5
        return kind, 30.0 * torch.tanh(x / 30.0)
    if kind == "qgemm":
        codes, scales, x = _packed_stream(case, seed)
        out = torch.empty(case["count"], case["rows"], case["N"], device=DEV)
        return kind, dict(case), codes, scales, x, out
    model = _model(case["profile"], "bf16", "bf16")
    eng = StaticACEngine(model, batch=case["B"], win=case["win"], block=case["ctx"], every=case["n"])
    t = synth.zipf_tokens(model.cfg.vocab_size, (case["B"], case["ctx"] + case["n"]), seed=seed)
    return kind, eng, [r[:case["ctx"]] for r in t], [r[case["ctx"]:] for r in t], [case["ctx"]] * case["B"]


def run(state):
    kind = state[0]
    if kind == "step":
        _, model, st, graph = state
        if graph is not None:
            graph.replay()
        else:
            model.static_extend(st)
        return {"logits": st.logits, "cum": st.cum, "raw": st.cand_prev_raw, "kv": st.kv}
    if kind == "softmax_cdf":
        probs, cum = ops.softmax_cdf(state[1])
        return {"probs": probs, "cum": cum}
    if kind == "qgemm":
        _, c, codes, scales, x, out = state
        n, k, b = c["N"], c["K"], c["bits"]
        f = ops.qgemv_stream if c["rows"] == 1 else ops.qgemm_stream
        return f(codes, scales, c["count"], n, k, b, n * k * b // 8, n * k // 64 * 2, x, out)
    _, eng, prefixes, segs, starts = state
    payloads = encode_segments_gpu(eng, prefixes, segs, starts)
    # one row per segment, zeros after its last byte, and the lengths
    rows = np.zeros((len(payloads), 64 + 4 * len(segs[0])), dtype=np.uint8)
    for r, p in zip(rows, payloads):
        r[:len(p)] = np.frombuffer(p, dtype=np.uint8)
    return {"payloads": rows, "lengths": np.array([len(p) for p in payloads]), "carry": eng.carry_row_dev()}


def _step_work(cfg, n_slots, weight_bytes, B, W, ctx, kv_size):
    """Bytes and operations of one W-token window of B segments after ctx tokens."""
    d, kvd, f, V = cfg.model_dim, cfg.kv_dim, cfg.hidden_dim, cfg.vocab_size
    rows = B * W
    nbytes = n_slots * B * 2 * (ctx + W) * kvd * kv_size + weight_bytes + rows * (2 * V + 1) * 4
    keys = W * ctx + W * (W + 1) / 2
    flops = (rows * 2 * (n_slots * (d * (d + 2 * kvd) + d * d + 2 * d * f) + V * d)
             + n_slots * B * cfg.num_heads * 4 * keys * cfg.head_dim)
    return nbytes, flops


def work(case):
    kind = case["kind"]
    if kind in ("step", "compress"):
        sm = _weights(case["profile"])
        cfg = sm.cfg
        enc, dec = synth.slot_itinerary(cfg)
        n_slots = len(enc) + len(dec)
        wb = sum(p.nbytes_codes + p.nbytes_scales for p in sm.packed.values())
        if kind == "step":
            b, f = _step_work(cfg, n_slots, wb, case["B"], case["W"], case["ctx"], 4 if case["kv"] == "fp32" else 2)
        else:  # every symbol's table once; each window reads the cache before it
            b = f = 0
            p, end = 0, case["ctx"] + case["n"] - 1
            while p < end:
                stop = case["ctx"] if p < case["ctx"] else end
                w = min(case["win"], stop - p)
                wb_, wf = _step_work(cfg, n_slots, wb, case["B"], w, p, 2)
                b, f, p = b + wb_, f + wf, p + w
        return {"bytes": b, "flops": f}
    if kind == "softmax_cdf":
        n = case["rows"] * case["V"]
        return {"bytes": 12 * n + 4 * case["rows"], "flops": 8 * n}
    nk = case["count"] * case["N"] * case["K"]
    return {"bytes": nk * case["bits"] / 8 + nk / 32 + case["rows"] * (2 * case["K"] + 4 * case["count"] * case["N"]),
            "flops": 2 * case["rows"] * nk}


def tolerance(case):
    kind = case["kind"]
    if kind == "compress":
        return "exact"
    # about four times the relative error measured against 64 bits; the tables
    # are whole numbers that both sides of a stream must share
    if kind == "step":
        if case["act"] == "bf16":  # logits 1.6e-3 to 2.3e-3, cache rows up to 2.5e-3
            return {"rel": 0.01, "differ": 0.0}
        # fp32 cache: 3.2e-6; a bf16 cache holds rounded rows, up to 1.7e-3
        return {"rel": 1.5e-5 if case["kv"] == "fp32" else 7e-3, "differ": 0.0}
    if kind == "softmax_cdf":  # 9.4e-8
        return {"rel": 4e-7, "differ": 0.0}
    # batch 1: 4.1e-5 (the group centre comes out of each group's sum); more rows: 1.0e-7
    return {"rel": 1.6e-4 if case["rows"] == 1 else 4e-7}


# ---- plain 64-bit results ------------------------------------------------------


def _rms(x):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + float(np.finfo(np.float32).eps))


def _rope(x, pos, cfg):
    """x [..., T, H, hd]: the first rope_dims dims rotated (halves paired)."""
    rd = cfg.rope_dims_eff
    inv = 1.0 / cfg.rope_base ** (torch.arange(0, rd, 2, dtype=torch.float64, device=x.device) / rd)
    a = pos.double()[:, None] * inv
    cos, sin = a.cos()[:, None], a.sin()[:, None]
    x1, x2, rest = x[..., :rd // 2], x[..., rd // 2:rd], x[..., rd:]
    return torch.cat([x1 * cos + x2 * sin, x2 * cos - x1 * sin, rest], -1)


def _exact_step(case, seed):
    sm = _weights(case["profile"])
    cfg = sm.cfg
    sd = {k: torch.as_tensor(np.asarray(v)).to(DEV).double() for k, v in sm.state_dict().items()}
    B, W, ctx, D, H, G = case["B"], case["W"], case["ctx"], cfg.model_dim, cfg.num_heads, cfg.num_kv_heads
    hd, L = cfg.head_dim, cfg.num_layers
    toks, prev = _tokens(case, cfg, seed)
    emb = sd["tok_emb.weight"]
    raw = emb[torch.from_numpy(toks).to(DEV)]  # [B, W, D]
    before = emb[torch.from_numpy(prev).to(DEV)] if ctx else torch.zeros(B, D, dtype=torch.float64, device=DEV)
    shifted = torch.cat([before[:, None], raw[:, :-1]], 1)
    g = sd["smear_lambda"] * torch.sigmoid(raw[..., :cfg.gate_window] @ sd["smear_gate.weight"].T)
    x0 = _rms(raw + g * shifted)
    pos = torch.arange(ctx, ctx + W, device=DEV)
    n_slots = sum(len(p) for p in synth.slot_itinerary(cfg))
    kv_out = torch.zeros(n_slots, B, 2, G, _max_len(case), hd, device=DEV, dtype=torch.float32)
    slot = [0]

    def attn(i, n):  # n [B, W, D]: the normalised attention input
        s = slot[0]
        slot[0] += 1
        q, k, v = n @ sd["qo_bank"][i].T, n @ sd["kv_bank"][i].T, n @ sd["kv_bank"][L + i].T
        if cfg.lora_rank:
            sc = cfg.lora_alpha / cfg.lora_rank
            q = q + sc * (n @ sd[f"q_loras.{s}.A"].T @ sd[f"q_loras.{s}.B"].T)
            v = v + sc * (n @ sd[f"v_loras.{s}.A"].T @ sd[f"v_loras.{s}.B"].T)
        q, k, v = q.view(B, W, H, hd), k.view(B, W, G, hd), v.view(B, W, G, hd)
        q = _rope(_rms(q), pos, cfg) * sd[f"blocks.{i}.attn.q_gain"][:, None]
        k = _rope(_rms(k), pos, cfg)
        old = _kv_rows(case, cfg, seed, s) if ctx else None
        if ctx:
            kv_out[s][:, :, :, :ctx] = old.float()
        kv_out[s][:, 0, :, ctx:ctx + W] = k.transpose(1, 2).float()
        kv_out[s][:, 1, :, ctx:ctx + W] = v.transpose(1, 2).float()
        mask = torch.arange(ctx + W, device=DEV)[None] > pos[:, None]
        y = torch.empty(B, W, H, hd, dtype=torch.float64, device=DEV)
        for b in range(B):
            kb, vb = k[b].transpose(0, 1), v[b].transpose(0, 1)  # [G, W, hd]
            if ctx:
                kb = torch.cat([old[b, 0].double(), kb], 1)
                vb = torch.cat([old[b, 1].double(), vb], 1)
            qb = q[b].view(W, G, H // G, hd).permute(1, 2, 0, 3)
            a = (qb @ kb[:, None].transpose(-1, -2)) / math.sqrt(hd)
            a = torch.softmax(a.masked_fill(mask, float("-inf")), -1)
            y[b] = (a @ vb[:, None]).permute(2, 0, 1, 3).reshape(W, H, hd)
        if i >= L - cfg.xsa_last_n:
            vn = torch.nn.functional.normalize(v, dim=-1).repeat_interleave(H // G, 2)
            y = y - (y * vn).sum(-1, keepdim=True) * vn
        gate = torch.sigmoid(cfg.sparse_attn_gate_scale
                             * (n[..., :cfg.gate_window] @ sd[f"blocks.{i}.attn.attn_gate_w"].T))
        return (y * gate[..., None]).reshape(B, W, D) @ sd["qo_bank"][L + i].T

    def mlp(i, n):
        h = torch.nn.functional.leaky_relu(n @ sd["mlp_up_bank"][i].T, 0.5).square()
        return h @ sd["mlp_down_bank"][i].T

    def ln(i):
        return 1.0 / math.sqrt(i + 1) if cfg.ln_scale else 1.0

    def block(i, x):
        mix = sd[f"blocks.{i}.resid_mix"]
        x = mix[0] * x + mix[1] * x0
        x = x + sd[f"blocks.{i}.attn_scale"] * attn(i, _rms(x) * ln(i))
        return x + sd[f"blocks.{i}.mlp_scale"] * mlp(i, _rms(x) * ln(i))

    def skip(j, x, stack):
        if j >= len(sd["skip_weights"]) or not stack:
            return x
        s = sd["skip_weights"][j] * stack.pop()
        return s + torch.sigmoid(sd["skip_gates"][j]) * (x - s)

    enc, dec = synth.slot_itinerary(cfg)
    x, stack, lanes = x0, [], None
    for i in enc:
        x = block(i, x)
        stack.append(x)
    for j, i in enumerate(dec):
        if 0 < cfg.parallel_start_layer <= i:
            l0, l1 = lanes or (x, x)
            l0 = skip(j, l0, stack)
            mix = sd[f"blocks.{i}.resid_mix"]
            a = sd[f"blocks.{i}.attn_scale"] * attn(i, _rms(mix[0] * l0 + mix[1] * x0) * ln(i))
            m = sd[f"blocks.{i}.mlp_scale"] * mlp(i, _rms(l1) * ln(i))
            pr, pp = sd["parallel_resid_lambdas"][i], sd["parallel_post_lambdas"][i]
            lanes = (pr[0] * l0 + pp[0][0] * a + pp[1][0] * m, pr[1] * l1 + pp[0][1] * a + pp[1][1] * m)
        else:
            x = block(i, skip(j, x, stack))
    if lanes:
        x = 0.5 * (lanes[0] + lanes[1])
    lg = _rms(x).reshape(B * W, D) @ emb.T
    sp, sn = sd["softcap_pos"], sd["softcap_neg"]
    lg = torch.where(lg >= 0, sp * torch.tanh(lg / sp), sn * torch.tanh(lg / sn))
    if case["kv"] == "bf16":
        for s in range(n_slots):
            kv_out[s, :, 0], kv_out[s, :, 1] = tile_kv(kv_out[s, :, 0], "k"), tile_kv(kv_out[s, :, 1], "v")
    return {"logits": lg, "cum": None, "raw": raw[:, -1], "kv": kv_out}


def _exact_qgemm(case, seed):
    """Unpacks the tiled codes: blocks of 16 rows x 256 columns; per block one
    plane after the other, lane l's 64 codes (row l % 16, columns 32 s + 8 (l //
    16) + i at place 8 s + i) low bits first."""
    codes, scales, x = _packed_stream(case, seed)
    N, K, b, x = case["N"], case["K"], case["bits"], x.double()
    out = torch.empty(case["count"], case["rows"], N, dtype=torch.float64, device=DEV)
    planes = {2: (2,), 3: (2, 1), 4: (4,), 6: (4, 2)}[b]
    for c in range(case["count"]):
        raw = codes[c * N * K * b // 8:(c + 1) * N * K * b // 8].view(-1, 512 * b)
        v, off, sh = 0, 0, 0
        for pb in planes:
            p = raw[:, off:off + 512 * pb].reshape(-1, 64, 8 * pb, 1).int()
            bits = torch.arange(0, 8, pb, device=DEV, dtype=torch.int32)
            v = v + (((p >> bits) & ((1 << pb) - 1)) << sh).view(-1, 64, 64)
            off, sh = off + 512 * pb, sh + pb
        w = (v.double() - ((1 << b) - 1) / 2).view(N // 16, K // 256, 4, 16, 8, 8)  # n, k, lane group, row, s, i
        s = scales[c * N * K // 64:(c + 1) * N * K // 64].double().view(N // 16, K // 256, 16, 4)
        w = w.permute(0, 3, 1, 4, 2, 5).reshape(N // 16, 16, K // 256, 4, 64)
        w = (w * s.permute(0, 2, 1, 3)[..., None]).reshape(N, K)
        out[c] = x @ w.T
    return out


def exact(case, seed):
    if case["kind"] == "step":
        with torch.no_grad():
            return _exact_step(case, seed)
    if case["kind"] == "softmax_cdf":
        return {"probs": torch.softmax(prepare(case, seed)[1].double(), -1), "cum": None}
    if case["kind"] == "qgemm":
        return _exact_qgemm(case, seed)
    return None
