"""The work that performance is measured on: the framework's operators and whole calls.

Everything is at Qwen3.5-4B's per-layer sizes (``qwen3_5_4b_config``): hidden 2560,
intermediate 9216, vocabulary 248320, 16 key / 32 value Gated DeltaNet heads of 128, 16 query
/ 4 KV attention heads of 256, int4 group-128 weights. Whole-model calls run the first four
layers (three Gated DeltaNet, one attention) and the head.

``kind`` names a path:

- ``mlp_decode``        RMSNorm + gate|up + SwiGLU, down + residual for 1..16 rows;
- ``head_decode``       residual + RMSNorm + tied head for 1..16 rows;
- ``delta_step``        one Gated DeltaNet token (conv, norms, gates, delta rule) for 1..16 sequences;
- ``attention_decode``  one gated GQA token over a KV cache;
- ``mlp_prefill``       residual + RMSNorm, gate|up + SwiGLU, down over a prompt's rows;
- ``deltanet_prefill``  causal conv, chunked delta rule and gated RMSNorm over a prompt;
- ``attention_prefill`` q/k norm + RoPE + KV write and causal attention over a prompt (or over a
  later chunk of one, ``pos0`` > 0);
- ``model_prefill``     ``Prefiller.fill``: a prompt into a decoder's caches;
- ``model_decode``      persistent decode steps after a context, tokens given.

``exact`` is plain torch in 64 bits. It rounds to bf16 only what the model defines as bf16
inputs of a later stage: the dequantised weights and, ahead of the fp32 delta rule, the conv's
output and beta; so the fp32 recurrent states are held to fp32 accuracy.
"""

from __future__ import annotations

from dataclasses import replace

import torch
import torch.nn.functional as F

from deltaforge_amd import _native as N
from deltaforge_amd import ops, prefill
from deltaforge_amd.config import hybrid_layer_types, qwen3_5_4b_config
from deltaforge_amd.persistent import PersistentDecoder
from deltaforge_amd.prefill import Prefiller
from deltaforge_amd.synth import CanonicalInt4, SynthModel

DEV = "cuda"
BF16 = torch.bfloat16
HIDDEN, INTER, VOCAB = 2560, 9216, 248320
HK, HV, DK = 16, 32, 128
CONV = (2 * HK + HV) * DK  # q | k | v channels
HQ, HKV, HD, ROT = 16, 4, 256, 64
LAYERS = 4
EPS = 1e-6
SPARE = 64  # decode slots kept behind a prompt


def listed() -> list[dict]:
    return [
        # bs = 1 decode, one layer's MLP: two launches, latency counts
        {"name": "mlp_decode_1", "kind": "mlp_decode", "rows": 1},
        # the widest batched decode one GEMV launch takes
        {"name": "mlp_decode_16", "kind": "mlp_decode", "rows": 16},
        # the tied head of a bs = 1 step, the longest single stream of weights
        {"name": "head_decode_1", "kind": "head_decode", "rows": 1},
        # the smallest call: one token of one Gated DeltaNet layer
        {"name": "delta_step_1", "kind": "delta_step", "batch": 1},
        # attention of a bs = 1 step at the benchmark's context
        {"name": "attention_decode_1x4096", "kind": "attention_decode", "batch": 1, "context": 4096},
        # batched serving at a long context
        {"name": "attention_decode_8x32768", "kind": "attention_decode", "batch": 8, "context": 32768},
        # a chat turn: a short prompt's MLP
        {"name": "mlp_prefill_100", "kind": "mlp_prefill", "rows": 100},
        # the benchmark's prompt: its MLP, linear layers' middle, and attention
        {"name": "mlp_prefill_4096", "kind": "mlp_prefill", "rows": 4096},
        {"name": "deltanet_prefill_4096", "kind": "deltanet_prefill", "tokens": 4096},
        # a long document in one chunk
        {"name": "attention_prefill_8192", "kind": "attention_prefill", "tokens": 8192, "pos0": 0},
        # whole calls: a ragged prompt, and decode at the benchmark's context
        {"name": "model_prefill_717", "kind": "model_prefill", "tokens": 717},
        {"name": "model_decode_4096", "kind": "model_decode", "context": 4096, "steps": 4},
    ]


def draw(rng) -> dict:
    def log_int(lo: int, hi: int) -> int:
        return min(hi, max(lo, round(lo * (hi / lo) ** rng.random())))

    kind = rng.choice(["mlp_decode", "head_decode", "delta_step", "attention_decode", "mlp_prefill",
                       "deltanet_prefill", "attention_prefill", "attention_prefill", "mlp_prefill",
                       "model_prefill", "model_decode"])
    if kind in ("mlp_decode", "head_decode"):
        return {"kind": kind, "rows": rng.randint(2, 15)}
    if kind == "delta_step":
        return {"kind": kind, "batch": rng.randint(2, 16)}
    if kind == "attention_decode":
        batch = rng.randint(1, 8)
        return {"kind": kind, "batch": batch, "context": log_int(33, 262144 // batch)}
    if kind == "mlp_prefill":
        return {"kind": kind, "rows": log_int(17, 4095)}
    if kind == "deltanet_prefill":
        return {"kind": kind, "tokens": log_int(5, 4095)}
    if kind == "attention_prefill":
        tokens = log_int(17, 8000)
        pos0 = rng.choice([0, log_int(1, 32768)])
        while tokens * (pos0 + tokens // 2) > 8192 * 4096:
            pos0 //= 2
        return {"kind": kind, "tokens": tokens, "pos0": pos0}
    if kind == "model_prefill":
        return {"kind": kind, "tokens": log_int(9, 1500)}
    return {"kind": kind, "context": log_int(17, 8000), "steps": rng.randint(1, 4)}


# -- inputs -------------------------------------------------------------------------------


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(g, shape, std=1.0, mean=0.0, dtype=BF16):
    return (torch.randn(shape, generator=g, device=DEV) * std + mean).to(dtype)


def _int4(g, k: int, n: int) -> CanonicalInt4:
    """A symmetric quantiser's weight: nibbles 1..15 (-7..7), scales |N(0, 1)| * 0.02."""
    words = torch.randint(-(2**31), 2**31 - 1, (k // 2 * n // 4,), generator=g, dtype=torch.int32, device=DEV)
    packed = words.view(torch.uint8).reshape(k // 2, n)
    packed = packed + (packed & 0x0F == 0).to(torch.uint8) * 8 + (packed < 16).to(torch.uint8) * 128
    return CanonicalInt4(packed, (torch.randn((k // 128, n), generator=g, device=DEV).abs() * 0.02).to(BF16))


def _repack(w: CanonicalInt4) -> ops.Int4Weight:
    return ops.int4_repack(w.packed, w.scale)


def _gate_up(gate: CanonicalInt4, up: CanonicalInt4) -> ops.Int4Weight:
    return ops.int4_repack(*ops.interleave_gate_up(gate.packed, gate.scale, up.packed, up.scale))


def _inv_freq() -> torch.Tensor:
    """theta = 1e7 over 64 rotary dims, bf16-rounded as the model's buffer is; fp32."""
    f = 1.0 / (1e7 ** (torch.arange(0, ROT, 2, dtype=torch.float32) / ROT))
    return f.to(BF16).float().to(DEV)


def _mlp_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    return {"x": _normal(g, (case["rows"], HIDDEN)), "res": _normal(g, (case["rows"], HIDDEN)),
            "norm": _normal(g, (HIDDEN,), 0.02), "gate": _int4(g, HIDDEN, INTER), "up": _int4(g, HIDDEN, INTER),
            "down": _int4(g, INTER, HIDDEN)}


def _head_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    return {"x": _normal(g, (case["rows"], HIDDEN)), "res": _normal(g, (case["rows"], HIDDEN)),
            "norm": _normal(g, (HIDDEN,), 0.02), "head": _int4(g, HIDDEN, VOCAB)}


def _delta_params(g) -> dict:
    return {"conv_w": _normal(g, (CONV, 4), 0.3), "A_log": _normal(g, (HV,), 0.1), "dt_bias": _normal(g, (HV,), 0.1)}


def _delta_step_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    b = case["batch"]
    return {"qkv": _normal(g, (b, CONV)), "ab": _normal(g, (b, 2 * HV)), "ring": _normal(g, (b, CONV, 4)),
            "state": _normal(g, (b, HV, DK, DK), 0.1, dtype=torch.float32), **_delta_params(g)}


def _attention_decode_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    b, max_len = case["batch"], case["context"] + SPARE
    return {"q": _normal(g, (b, HQ * 2 * HD)), "k": _normal(g, (b, HKV * HD)), "v": _normal(g, (b, HKV * HD)),
            "q_norm": _normal(g, (HD,), 0.02), "k_norm": _normal(g, (HD,), 0.02),
            "k_cache": _normal(g, (b, HKV, max_len, HD)), "v_cache": _normal(g, (b, HKV, max_len, HD))}


def _deltanet_prefill_inputs(case: dict, seed: int) -> dict:
    """The input projection's rows ``q | k | v | z | a | b`` and a layer's small weights; a new
    sequence: empty history, zero state."""
    g = _gen(seed)
    return {"proj": _normal(g, (case["tokens"], CONV + HV * DK + 2 * HV)), "gnorm": _normal(g, (DK,), 0.02, 1.0),
            **_delta_params(g)}


def _attention_prefill_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    p, max_len = case["tokens"], case["pos0"] + case["tokens"] + SPARE
    return {"proj": _normal(g, (p, (2 * HQ + 2 * HKV) * HD)), "q_norm": _normal(g, (HD,), 0.02),
            "k_norm": _normal(g, (HD,), 0.02), "k_cache": _normal(g, (HKV, max_len, HD)),
            "v_cache": _normal(g, (HKV, max_len, HD))}


def _config():
    return replace(qwen3_5_4b_config(), num_hidden_layers=LAYERS, layer_types=hybrid_layer_types(LAYERS))


def _model(g) -> SynthModel:
    c = _config()
    m = SynthModel(c)
    lin, par = m.linears, m.params
    for i, kind in enumerate(c.layer_types):
        p = f"layers.{i}."
        if kind == "full_attention":
            a = p + "self_attn."
            shapes = {"q_proj": 2 * HQ * HD, "k_proj": HKV * HD, "v_proj": HKV * HD}
            lin[a + "o_proj.weight"] = _int4(g, HQ * HD, HIDDEN)
            par[a + "q_norm.weight"], par[a + "k_norm.weight"] = _normal(g, (HD,), 0.02), _normal(g, (HD,), 0.02)
        else:
            a = p + "linear_attn."
            shapes = {"in_proj_qkv": CONV, "in_proj_z": HV * DK, "in_proj_a": HV, "in_proj_b": HV}
            lin[a + "out_proj.weight"] = _int4(g, HV * DK, HIDDEN)
            d = _delta_params(g)
            par[a + "conv1d.weight"] = d["conv_w"].reshape(CONV, 1, 4)
            par[a + "A_log"], par[a + "dt_bias"] = d["A_log"], d["dt_bias"]
            par[a + "norm.weight"] = _normal(g, (DK,), 0.02, 1.0)
        for name, n in shapes.items():
            lin[a + name + ".weight"] = _int4(g, HIDDEN, n)
        lin[p + "mlp.gate_proj.weight"] = _int4(g, HIDDEN, INTER)
        lin[p + "mlp.up_proj.weight"] = _int4(g, HIDDEN, INTER)
        lin[p + "mlp.down_proj.weight"] = _int4(g, INTER, HIDDEN)
        par[p + "input_layernorm.weight"] = _normal(g, (HIDDEN,), 0.02)
        par[p + "post_attention_layernorm.weight"] = _normal(g, (HIDDEN,), 0.02)
    lin["lm_head"] = _int4(g, HIDDEN, VOCAB)
    par["norm.weight"] = _normal(g, (HIDDEN,), 0.02)
    return m


def _model_inputs(case: dict, seed: int) -> dict:
    """The model and a prompt; for decode also the caches that ``context`` tokens left."""
    g = _gen(seed)
    model = _model(g)
    n = case["tokens"] if case["kind"] == "model_prefill" else case["context"] + case["steps"]
    out = {"model": model, "ids": torch.randint(0, VOCAB, (1, n), generator=g, device=DEV), "max_len": n + SPARE}
    if case["kind"] == "model_decode":
        out["caches"] = []
        for kind in model.config.layer_types:
            if kind == "full_attention":
                out["caches"].append({"k_cache": _normal(g, (HKV, out["max_len"], HD)),
                                      "v_cache": _normal(g, (HKV, out["max_len"], HD))})
            else:
                out["caches"].append({"conv_ring": _normal(g, (CONV, 4)),
                                      "state": _normal(g, (HV, DK, DK), 0.1, dtype=torch.float32)})
    return out


_INPUTS = {"mlp_decode": _mlp_inputs, "mlp_prefill": _mlp_inputs, "head_decode": _head_inputs,
           "delta_step": _delta_step_inputs, "attention_decode": _attention_decode_inputs,
           "deltanet_prefill": _deltanet_prefill_inputs, "attention_prefill": _attention_prefill_inputs,
           "model_prefill": _model_inputs, "model_decode": _model_inputs}


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    t = _INPUTS[kind](case, seed)
    s = {"case": case, **{k: v for k, v in t.items() if isinstance(v, torch.Tensor)}}
    if kind in ("mlp_decode", "mlp_prefill"):
        s["gate_up"], s["down"] = _gate_up(t["gate"], t["up"]), _repack(t["down"])
    elif kind == "head_decode":
        s["head"] = _repack(t["head"])
        s["h_out"] = torch.empty_like(t["x"])
    elif kind == "delta_step":
        s["position"] = torch.full((1,), 5, dtype=torch.int32, device=DEV)
        s["out"] = torch.empty((case["batch"], HV, DK), dtype=BF16, device=DEV)
    elif kind == "attention_decode":
        s["position"] = torch.full((1,), case["context"], dtype=torch.int32, device=DEV)
        s["inv"] = _inv_freq()
    elif kind == "deltanet_prefill":
        s["ring"] = torch.zeros((CONV, 4), dtype=BF16, device=DEV)
        s["state"] = torch.zeros((HV, DK, DK), dtype=torch.float32, device=DEV)
    elif kind == "attention_prefill":
        s["inv"] = _inv_freq()
    else:
        s["decoder"] = PersistentDecoder(t["model"], max_seq_len=t["max_len"], max_new_tokens=SPARE)
        if kind == "model_prefill":
            s["prefiller"] = Prefiller(t["model"])
        else:
            for own, given in zip(s["decoder"].layer_state, t["caches"]):
                for name in own:
                    own[name].copy_(given[name])
            n = t["ids"].shape[1]
            s["decoder"].prompt[:n].copy_(t["ids"][0])
            s["decoder"].prompt_len = n
    return s


def run(s: dict):
    case = s["case"]
    kind = case["kind"]
    if kind == "mlp_decode":
        act = ops.int4_gemv(s["x"], s["gate_up"], prologue=N.PRO_RMSNORM, epilogue=N.EPI_SWIGLU, norm_w=s["norm"], eps=EPS)
        return ops.int4_gemv(act, s["down"], epilogue=N.EPI_RESIDUAL, res=s["x"])
    if kind == "head_decode":
        logits = ops.int4_gemv(s["x"], s["head"], prologue=N.PRO_ADD_RMSNORM, x2=s["res"], norm_w=s["norm"], eps=EPS,
                               h_out=s["h_out"])
        return logits, s["h_out"]
    if kind == "delta_step":
        out = ops.gated_delta_step(s["qkv"], s["ab"][:, :HV], s["ab"][:, HV:], s["A_log"], s["dt_bias"], s["conv_w"],
                                   s["state"], num_k_heads=HK, conv_ring=s["ring"], position=s["position"], out=s["out"])
        return out, s["state"], s["ring"]
    if kind == "attention_decode":
        out = ops.attention_decode(s["q"], s["k"], s["v"], s["q_norm"], s["k_norm"], s["inv"], s["k_cache"],
                                   s["v_cache"], s["position"], num_q_heads=HQ, eps=EPS)
        return out, s["k_cache"], s["v_cache"]
    if kind == "mlp_prefill":
        h, x = ops.add_rms_norm(s["x"], s["res"], s["norm"], EPS)
        act = prefill.int4_gemm(x, s["gate_up"], epilogue=N.EPI_SWIGLU)
        return h, prefill.int4_gemm(act, s["down"])
    if kind == "deltanet_prefill":
        proj, zc = s["proj"], CONV + HV * DK
        mixed = prefill.causal_conv_prefill(proj[:, :CONV], s["conv_w"], s["ring"])
        core = prefill.delta_rule_prefill(mixed, proj[:, zc:], proj[:, zc + HV:], s["A_log"], s["dt_bias"], s["state"],
                                          num_k_heads=HK)
        y = prefill.gated_rms_norm_rows(core, proj[:, CONV:zc], s["gnorm"], EPS)
        return mixed, core, y, s["state"], s["ring"]
    if kind == "attention_prefill":
        qd, kvd, pos0 = 2 * HQ * HD, HKV * HD, case["pos0"]
        q = prefill.qk_norm_rope_prefill(s["proj"], s["q_norm"], s["k_norm"], s["inv"], s["k_cache"], s["v_cache"],
                                         num_q_heads=HQ, k_col=qd, v_col=qd + kvd, pos0=pos0, eps=EPS)
        out = prefill.attention_prefill(q, s["k_cache"], s["v_cache"], s["proj"][:, HD:], gate_head_stride=2 * HD,
                                        pos0=pos0)
        return q, out, s["k_cache"], s["v_cache"]
    dec = s["decoder"]
    if kind == "model_prefill":
        s["prefiller"].fill(dec, s["ids"])
    else:
        dec.position.fill_(case["context"])
        dec.launch(case["steps"], teacher_forced=True)
    return {"logits": dec.logits, "caches": dec.layer_state}


# -- what a pass cannot do without -----------------------------------------------------------


def _w_bytes(k: int, n: int) -> int:
    return k * n // 2 + k // 128 * n * 2


def work(case: dict) -> dict:
    kind = case["kind"]
    mlp_w, mlp_flops = 3 * _w_bytes(HIDDEN, INTER), 6 * HIDDEN * INTER
    state = HV * DK * DK * 4
    if kind in ("mlp_decode", "mlp_prefill"):
        m = case["rows"]
        rows_moved = 2 if kind == "mlp_decode" else 4  # x in, y out; a prompt: x, res in, h, y out
        return {"bytes": mlp_w + HIDDEN * 2 + m * HIDDEN * 2 * rows_moved, "flops": m * mlp_flops}
    if kind == "head_decode":
        m = case["rows"]
        return {"bytes": _w_bytes(HIDDEN, VOCAB) + HIDDEN * 2 + m * (3 * HIDDEN + VOCAB) * 2,
                "flops": 2 * m * HIDDEN * VOCAB}
    if kind == "delta_step":
        b = case["batch"]
        return {"bytes": b * (2 * state + CONV * 2 + CONV * 8 + HV * DK * 2 + HV * 4) + CONV * 8,
                "flops": b * HV * DK * DK * 6}
    if kind == "attention_decode":
        b, n = case["batch"], case["context"] + 1
        return {"bytes": b * (n * HKV * HD * 4 + (3 * HQ + 4 * HKV) * HD * 2), "flops": b * HQ * n * HD * 4}
    if kind == "deltanet_prefill":
        p = case["tokens"]
        # token by token: decay, recall, write and read of the state
        return {"bytes": p * (CONV * 2 * 2 + 4 * HV * DK * 2 + HV * 4) + state + CONV * 16,
                "flops": p * HV * DK * DK * 6}
    if kind == "attention_prefill":
        p, pos0 = case["tokens"], case["pos0"]
        keys = p * pos0 + p * (p + 1) // 2
        return {"bytes": p * (2 * HQ + 2 * HKV) * HD * 2 + p * 2 * HQ * HD * 2 + (pos0 + 2 * p) * 2 * HKV * HD * 2,
                "flops": keys * HQ * HD * 4}
    mix_w = 3 * (_w_bytes(HIDDEN, CONV + HV * DK + 2 * HV) + _w_bytes(HV * DK, HIDDEN))
    mix_w += _w_bytes(HIDDEN, (2 * HQ + 2 * HKV) * HD) + _w_bytes(HQ * HD, HIDDEN)
    weights = mix_w + LAYERS * mlp_w + _w_bytes(HIDDEN, VOCAB)
    per_token = 3 * 2 * HIDDEN * (CONV + 2 * HV * DK + 2 * HV) + 2 * HIDDEN * (3 * HQ + 2 * HKV) * HD + LAYERS * mlp_flops
    per_token += 3 * HV * DK * DK * 6
    if kind == "model_prefill":
        p = case["tokens"]
        return {"bytes": weights + 3 * (state + CONV * 8) + p * 2 * HKV * HD * 2 + VOCAB * 2,
                "flops": p * per_token + p * (p + 1) // 2 * HQ * HD * 4 + 2 * HIDDEN * VOCAB}
    n, ctx = case["steps"], case["context"]
    keys = n * (ctx + 1) + n * (n - 1) // 2
    return {"bytes": n * (weights + 3 * (2 * state + CONV * 8)) + keys * HKV * HD * 4 + VOCAB * 2,
            "flops": n * (per_token + 2 * HIDDEN * VOCAB) + keys * HQ * HD * 4}


def tolerance(case: dict) -> dict:
    """Against 64 bits the blocks measured 1.6e-3 to 5e-3 (2-norm; one rounding of a bf16 result
    is 1.7e-3) and two orders of their sums differ by less; the four-layer model, which carries
    each stage's roundings through all that follow, 0.5e-2 to 2.5e-2."""
    kind = case["kind"]
    if kind in ("model_prefill", "model_decode"):
        return {"rel": 0.03, "max": 0.6}
    return {"rel": 0.01, "max": 0.1}


# -- the same results in 64 bits -------------------------------------------------------------


def _w64(w: CanonicalInt4) -> torch.Tensor:
    q = torch.cat((w.packed & 0x0F, w.packed >> 4), 0).to(torch.float32) - 8.0
    k, n = q.shape
    return (q.reshape(k // 128, 128, n) * w.scale.float().unsqueeze(1)).to(BF16).reshape(k, n).double()


def _mm(x: torch.Tensor, w: CanonicalInt4) -> torch.Tensor:
    """``x @ W`` in column panels, so that a wide weight's 64-bit form stays small."""
    n = w.packed.shape[1]
    return torch.cat([x @ _w64(CanonicalInt4(w.packed[:, c:c + 16384], w.scale[:, c:c + 16384]))
                      for c in range(0, n, 16384)], 1)


def _rms(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * (1.0 + w.double())


def _bf(x: torch.Tensor) -> torch.Tensor:
    return x.to(BF16).double()


def _mlp64(x, norm, gate, up, down):
    n = _rms(x, norm)
    return _mm(F.silu(_mm(n, gate)) * _mm(n, up), down)


def _conv64(x, ring, pos0, conv_w, kept):
    """``x [P, C]`` with the ring's last three inputs before it; the bf16 result and the ring with
    the last ``kept`` inputs (a prompt leaves the three that are read again, a step its own)."""
    hist = torch.stack([ring[:, (pos0 - 3 + j) % 4] for j in range(3)], 0).double()
    full = torch.cat((hist, x), 0)
    w, p = conv_w.double(), x.shape[0]
    acc = sum(full[j:j + p] * w[:, j] for j in range(4))
    ring = ring.clone()
    for t in range(max(0, p - kept), p):
        ring[:, (pos0 + t) % 4] = x[t].to(BF16)
    return _bf(F.silu(_bf(acc))), ring


def _delta64(mixed, a, b, A_log, dt_bias, state):
    """The token-by-token rule; ``mixed [P, q|k|v]``, ``state [..., HV, DK, DK]``."""
    p = mixed.shape[0]
    q, k, v = mixed.split([HK * DK, HK * DK, HV * DK], -1)
    q, k = (t.reshape(p, HK, DK) for t in (q, k))
    q, k = (t * torch.rsqrt(t.square().sum(-1, keepdim=True) + 1e-6) for t in (q, k))
    q, k = (t.repeat_interleave(HV // HK, 1) for t in (q / DK**0.5, k))
    v = v.reshape(p, HV, DK)
    decay = torch.exp(-A_log.double().exp() * F.softplus(a.double() + dt_bias.double()))
    beta = _bf(torch.sigmoid(b.double()))
    out = torch.empty((p, HV, DK), dtype=torch.float64, device=DEV)
    for t in range(p):
        state = state * decay[t][:, None, None]
        delta = (v[t] - (k[t].unsqueeze(1) @ state).squeeze(1)) * beta[t][:, None]
        state = state + k[t].unsqueeze(2) * delta.unsqueeze(1)
        out[t] = (q[t].unsqueeze(1) @ state).squeeze(1)
    return out, state


def _gated_norm64(core, z, w):
    x = core * torch.rsqrt(core.square().mean(-1, keepdim=True) + EPS) * w.double()
    return x * F.silu(z)


def _rope64(x, pos):
    """``x [P, H, HD]`` at positions ``pos [P]``, the first ROT dims rotated."""
    ang = pos.double()[:, None] * _inv_freq().double()[None]
    cos, sin = (t.repeat(1, 2)[:, None] for t in (ang.cos(), ang.sin()))
    r = x[..., :ROT]
    half = torch.cat((-r[..., ROT // 2:], r[..., :ROT // 2]), -1)
    return torch.cat((r * cos + half * sin, x[..., ROT:]), -1)


def _attention64(q, gate, k_cache, v_cache, pos0):
    """``q [P, HQ, HD]`` over ``[HKV, L, HD]`` caches up to each position, times sigmoid(gate)."""
    p = q.shape[0]
    out = torch.empty_like(q)
    cols = torch.arange(pos0 + p, device=DEV)
    for h in range(HQ):
        kc, vc = (t[h // (HQ // HKV), :pos0 + p].double() for t in (k_cache, v_cache))
        for r0 in range(0, p, 2048):
            r1 = min(r0 + 2048, p)
            s = q[r0:r1, h] @ kc.t() * HD**-0.5
            s.masked_fill_(cols[None] > pos0 + torch.arange(r0, r1, device=DEV)[:, None], float("-inf"))
            out[r0:r1, h] = s.softmax(-1) @ vc
    return (out * torch.sigmoid(gate)).reshape(p, HQ * HD)


def _attention_rows64(proj, q_norm, k_norm, k_cache, v_cache, pos0):
    """A projection's rows ``[per head query | gate] | k | v``: queries, output and 64-bit caches."""
    p = proj.shape[0]
    qg = proj[:, :2 * HQ * HD].reshape(p, HQ, 2, HD)
    kv = proj[:, 2 * HQ * HD:].reshape(p, 2, HKV, HD)
    pos = torch.arange(pos0, pos0 + p, device=DEV)
    q, k = _rope64(_rms(qg[:, :, 0], q_norm), pos), _rope64(_rms(kv[:, 0], k_norm), pos)
    k_cache, v_cache = k_cache.double(), v_cache.double()
    k_cache[:, pos0:pos0 + p], v_cache[:, pos0:pos0 + p] = k.transpose(0, 1), kv[:, 1].transpose(0, 1)
    return q, _attention64(q, qg[:, :, 1], k_cache, v_cache, pos0), k_cache, v_cache


def _forward64(model: SynthModel, ids: torch.Tensor, caches: list[dict], pos0: int, kept: int) -> tuple:
    lin, par = model.linears, model.params
    head = lin["lm_head"]
    cols = CanonicalInt4(head.packed[:, ids], head.scale[:, ids])
    h = _w64(cols).t()
    new = []
    for i, kind in enumerate(model.config.layer_types):
        p, cache = f"layers.{i}.", caches[i]
        x = _rms(h, par[p + "input_layernorm.weight"])
        if kind == "full_attention":
            a = p + "self_attn."
            proj = torch.cat([_mm(x, lin[a + f"{n}_proj.weight"]) for n in "qkv"], 1)
            _, o, kc, vc = _attention_rows64(proj, par[a + "q_norm.weight"], par[a + "k_norm.weight"],
                                             cache["k_cache"], cache["v_cache"], pos0)
            h = h + _mm(o, lin[a + "o_proj.weight"])
            new.append({"k_cache": kc, "v_cache": vc})
        else:
            a = p + "linear_attn."
            qkv, z, ga, gb = (_mm(x, lin[a + f"in_proj_{n}.weight"]) for n in ("qkv", "z", "a", "b"))
            mixed, ring = _conv64(qkv, cache["conv_ring"], pos0, par[a + "conv1d.weight"].reshape(CONV, 4), kept)
            core, state = _delta64(mixed, ga, gb, par[a + "A_log"], par[a + "dt_bias"], cache["state"].double())
            y = _gated_norm64(core, z.reshape(-1, HV, DK), par[a + "norm.weight"]).reshape(-1, HV * DK)
            h = h + _mm(y, lin[a + "out_proj.weight"])
            new.append({"conv_ring": ring, "state": state})
        h = h + _mlp64(h, par[p + "post_attention_layernorm.weight"], lin[p + "mlp.gate_proj.weight"],
                       lin[p + "mlp.up_proj.weight"], lin[p + "mlp.down_proj.weight"])
    return _mm(_rms(h[-1:], par["norm.weight"]), head), new


@torch.no_grad()
def exact(case: dict, seed: int):
    kind = case["kind"]
    t = _INPUTS[kind](case, seed)
    if kind == "mlp_decode":
        x = t["x"].double()
        return x + _mlp64(x, t["norm"], t["gate"], t["up"], t["down"])
    if kind == "mlp_prefill":
        h = t["x"].double() + t["res"].double()
        return h, _mlp64(h, t["norm"], t["gate"], t["up"], t["down"])
    if kind == "head_decode":
        h = t["x"].double() + t["res"].double()
        return _mm(_rms(h, t["norm"]), t["head"]), h
    if kind == "delta_step":
        outs, states, rings = [], [], []
        for i in range(case["batch"]):
            mixed, ring = _conv64(t["qkv"][i:i + 1].double(), t["ring"][i], 5, t["conv_w"], 1)
            o, st = _delta64(mixed, t["ab"][i:i + 1, :HV], t["ab"][i:i + 1, HV:], t["A_log"], t["dt_bias"],
                             t["state"][i].double())
            outs.append(o[0])
            states.append(st)
            rings.append(ring)
        return torch.stack(outs), torch.stack(states), torch.stack(rings).double()
    if kind == "attention_decode":
        outs, n = [], case["context"]
        kcs, vcs = t["k_cache"].double(), t["v_cache"].double()
        for i in range(case["batch"]):
            proj = torch.cat((t["q"][i:i + 1], t["k"][i:i + 1], t["v"][i:i + 1]), 1).double()
            _, o, kcs[i], vcs[i] = _attention_rows64(proj, t["q_norm"], t["k_norm"], t["k_cache"][i], t["v_cache"][i], n)
            outs.append(o[0])
        return torch.stack(outs), kcs, vcs
    if kind == "deltanet_prefill":
        proj = t["proj"].double()
        zc, p = CONV + HV * DK, case["tokens"]
        ring = torch.zeros((CONV, 4), dtype=BF16, device=DEV)
        mixed, ring = _conv64(proj[:, :CONV], ring, 0, t["conv_w"], 3)
        core, state = _delta64(mixed, proj[:, zc:zc + HV], proj[:, zc + HV:], t["A_log"], t["dt_bias"],
                               torch.zeros((HV, DK, DK), dtype=torch.float64, device=DEV))
        y = _gated_norm64(core, proj[:, CONV:zc].reshape(p, HV, DK), t["gnorm"])
        return mixed, core.reshape(p, HV * DK), y.reshape(p, HV * DK), state, ring.double()
    if kind == "attention_prefill":
        q, out, kc, vc = _attention_rows64(t["proj"].double(), t["q_norm"], t["k_norm"], t["k_cache"], t["v_cache"],
                                           case["pos0"])
        return q, out, kc, vc
    if kind == "model_prefill":
        caches = []
        for layer in t["model"].config.layer_types:
            if layer == "full_attention":
                kv = torch.zeros((HKV, t["max_len"], HD), dtype=BF16, device=DEV)
                caches.append({"k_cache": kv, "v_cache": kv})
            else:
                caches.append({"conv_ring": torch.zeros((CONV, 4), dtype=BF16, device=DEV),
                               "state": torch.zeros((HV, DK, DK), dtype=torch.float32, device=DEV)})
        logits, new = _forward64(t["model"], t["ids"][0], caches, 0, 3)
    else:
        n = case["context"]
        logits, new = _forward64(t["model"], t["ids"][0, n:], t["caches"], n, 4)
    # a ring's slots are what the model rounds to bf16; its 64-bit form is those values
    return {"logits": logits, "caches": [{k: v.double() for k, v in c.items()} for c in new]}
