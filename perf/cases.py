"""The work that programs built on this package give it, as measurable cases.

A case is one pass through public entry points: a layer's attention over a
prompt or a chunk of one, the attention over a few appended tokens, one decode
step of a layer's attention, the MLP of a decode step, or a whole token step of
a Qwen3 model through its graph runner.  Head counts and hidden sizes are those
of Qwen3-0.6B, Qwen3-4B and Qwen3-32B; everything is f16, as the package takes it.

``listed()`` holds the fixed cases, ``draw(rng)`` one more of the same ranges.
"""
from __future__ import annotations

import math

import torch

import grout_amd as ga

D = ga.HEAD_DIM
EPS = 1e-6
THETA = 1e6
#: f16(1/sqrt(128)), the scale that decode programs pass as f16 bits.
SCALE_F16 = 0.08837890625
SCALE_F16_BITS = 0x2DA8
VOCAB = 151936

#: name -> (query heads, KV heads, hidden, intermediate, layers, tied embeddings)
MODELS = {
    "0.6b": (16, 8, 1024, 3072, 28, True),
    "4b": (32, 8, 2560, 9728, 36, True),
    "32b": (64, 8, 5120, 25600, 64, False),
}
#: Weights of a drawn token step: no more than those of the whole 4B model.
STEP_MAX_BYTES = 8.1e9
#: Query-key pairs times query heads of a drawn prompt: no more than an
#: 8192-token prompt over 32 query heads.
PROMPT_MAX_PAIRS = 32 * 8192 * 8193 // 2
#: Longest cached prefix that a drawn prompt chunk or suffix follows.
MAX_START = 30000


def listed():
    return [
        # A one-line chat turn on the smallest model: latency and launches.
        {"name": "prompt_37_0.6b", "kind": "prompt", "model": "0.6b", "seq": 37, "start": 0, "cap": 512},
        # An ordinary prompt of about a thousand tokens.
        {"name": "prompt_1000_4b", "kind": "prompt", "model": "4b", "seq": 1000, "start": 0, "cap": 4096},
        # A document of a few thousand tokens on the largest model.
        {"name": "prompt_3001_32b", "kind": "prompt", "model": "32b", "seq": 3001, "start": 0, "cap": 4096},
        # The long prompt of the benchmark's headline (32 query heads, 8192 tokens).
        {"name": "prompt_8192_4b", "kind": "prompt", "model": "4b", "seq": 8192, "start": 0, "cap": 8192},
        # One chunk of a chunked prefill: 509 tokens behind 6003 cached ones.
        {"name": "chunk_509_at_6003_4b", "kind": "prompt", "model": "4b", "seq": 509, "start": 6003, "cap": 8192},
        # A few drafted tokens checked against a long context: the unfused
        # suffix writer, then attention of 7 rows over 12008 keys.
        {"name": "suffix_7_at_12001_4b", "kind": "suffix", "model": "4b", "seq": 7, "start": 12001, "cap": 16384},
        # Decode early in a conversation, in a cache laid out for 4096 tokens.
        {"name": "decode_700_0.6b", "kind": "decode", "model": "0.6b", "pos": 700, "cap": 4096},
        # Decode in the middle of a long conversation on the largest model.
        {"name": "decode_9001_32b", "kind": "decode", "model": "32b", "pos": 9001, "cap": 32768},
        # Decode at the end of a 32K context: the largest cache read.
        {"name": "decode_32701_4b", "kind": "decode", "model": "4b", "pos": 32701, "cap": 32768},
        # The MLP half of a decode step of the largest model, op by op.
        {"name": "mlp_32b", "kind": "mlp", "model": "32b"},
        # A whole token of the smallest model: many short kernels.
        {"name": "step_0.6b", "kind": "step", "model": "0.6b", "layers": 28, "pos": 611, "cap": 2048},
        # A whole token of the 4B model in a conversation of 4000 tokens.
        {"name": "step_4b", "kind": "step", "model": "4b", "layers": 36, "pos": 4001, "cap": 8192},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _layer_weights(model):
    hq, hkv, hidden, inter, _, _ = MODELS[model]
    return (hq + 2 * hkv) * D * hidden + hq * D * hidden + 3 * inter * hidden


def draw(rng):
    kind = rng.choice(["prompt", "prompt", "prompt", "suffix", "decode", "decode", "mlp", "step"])
    model = rng.choice(sorted(MODELS))
    hq = MODELS[model][0]
    if kind in ("prompt", "suffix"):
        seq = _log_int(rng, 1, 8192) if kind == "prompt" else _log_int(rng, 1, 16)
        start = _log_int(rng, 1, MAX_START) if kind == "suffix" or rng.random() < 0.5 else 0
        while hq * (seq * start + seq * (seq + 1) // 2) > PROMPT_MAX_PAIRS:
            start, seq = start // 2, max(1, seq * 3 // 4)
        return {"kind": kind, "model": model, "seq": seq, "start": start,
                "cap": start + seq + rng.choice([0, rng.randint(1, 2048)])}
    if kind == "decode":
        pos = _log_int(rng, 1, 32767)
        cap = rng.choice([c for c in (pos + 1, 2048, 4096, 8192, 16384, 32768, 40960) if c > pos])
        return {"kind": kind, "model": model, "pos": pos, "cap": cap}
    if kind == "mlp":
        return {"kind": kind, "model": model}
    most = MODELS[model][4]
    while 2 * (most * _layer_weights(model) + VOCAB * MODELS[model][2]) > STEP_MAX_BYTES:
        most -= 1
    pos = _log_int(rng, 1, 8191)
    return {"kind": kind, "model": model, "layers": _log_int(rng, 1, most), "pos": pos,
            "cap": rng.choice([c for c in (pos + 1, 2048, 4096, 8192) if c > pos])}


# ------------------------------------------------------------------ inputs --

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(0x67726F7574 + seed)
    return g


def _normal(g, *shape, scale=1.0):
    x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float16)
    return x.mul_(scale) if scale != 1.0 else x


def _norm_weight(g, n):
    return (1 + 0.1 * torch.randn((n,), generator=g, device="cuda")).half()


def _cache(g, hkv, cap, filled):
    c = torch.zeros((hkv, cap, D), dtype=torch.float16, device="cuda")
    c[:, :filled] = _normal(g, hkv, filled, D)
    return c


def _inputs_attention(case, g):
    hq, hkv = MODELS[case["model"]][:2]
    s = {"hq": hq, "hkv": hkv}
    if case["kind"] == "decode":
        s["qkv"] = _normal(g, (hq + 2 * hkv) * D)
        filled = case["pos"]
    else:
        s["q"] = _normal(g, case["seq"], hq, D)
        s["k"], s["v"] = (_normal(g, case["seq"], hkv, D) for _ in range(2))
        filled = case["start"]
    if case["kind"] != "suffix":
        s["q_weight"], s["k_weight"] = _norm_weight(g, D), _norm_weight(g, D)
        s["inv_freq"] = ga.build_inv_freq(THETA).cuda()
    s["k_cache"], s["v_cache"] = (_cache(g, hkv, case["cap"], filled) for _ in range(2))
    return s


def _inputs_mlp(case, g):
    _, _, hidden, inter, _, _ = MODELS[case["model"]]
    return {"residual": _normal(g, hidden), "x": _normal(g, hidden), "weight": _norm_weight(g, hidden),
            "gate_up": _normal(g, 2 * inter, hidden, scale=hidden ** -0.5),
            "down": _normal(g, hidden, inter, scale=inter ** -0.5)}


def _inputs_step(case, g):
    hq, hkv, hidden, inter, _, tied = MODELS[case["model"]]
    k_all, v_all = (torch.zeros((case["layers"], hkv, case["cap"], D), dtype=torch.float16, device="cuda")
                    for _ in range(2))
    layers = []
    for i in range(case["layers"]):
        k_all[i, :, :case["pos"]] = _normal(g, hkv, case["pos"], D)
        v_all[i, :, :case["pos"]] = _normal(g, hkv, case["pos"], D)
        layers.append({
            "input_norm": _norm_weight(g, hidden),
            "qkv_proj": _normal(g, (hq + 2 * hkv) * D, hidden, scale=hidden ** -0.5),
            "q_norm": _norm_weight(g, D), "k_norm": _norm_weight(g, D),
            "o_proj": _normal(g, hidden, hq * D, scale=(hq * D) ** -0.5),
            "post_attn_norm": _norm_weight(g, hidden),
            "gate_up_proj": _normal(g, 2 * inter, hidden, scale=hidden ** -0.5),
            "down_proj": _normal(g, hidden, inter, scale=inter ** -0.5),
            "k_cache": k_all[i], "v_cache": v_all[i]})
    lm_head = _normal(g, VOCAB, hidden, scale=4 * hidden ** -0.5)
    embed = lm_head if tied else _normal(g, VOCAB, hidden)
    token = int(torch.randint(VOCAB, (1,), generator=g, device="cuda").item())
    return {"layers": layers, "embed_tokens": embed, "final_norm": _norm_weight(g, hidden),
            "lm_head": lm_head, "inv_freq": ga.build_inv_freq(THETA).cuda(), "first": token,
            "k_all": k_all, "v_all": v_all, "hq": hq, "hkv": hkv}


def _inputs(case, seed):
    g = _gen(seed)
    if case["kind"] == "mlp":
        return _inputs_mlp(case, g)
    if case["kind"] == "step":
        return _inputs_step(case, g)
    return _inputs_attention(case, g)


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    kind = case["kind"]
    if kind in ("prompt", "suffix"):
        s["out"] = torch.empty_like(s["q"])
        if kind == "prompt":
            s["q_out"] = torch.empty_like(s["q"])
            s["counters"] = ga.prefill_sched_counters()
    elif kind == "decode":
        hq, hkv = s["hq"], s["hkv"]
        splits = ga.pick_num_splits(case["cap"], hkv, group=hq // hkv)
        s["att"], s["lse"] = ga.decode_scratch(hkv, hq // hkv, splits)
        s["counters"] = ga.decode_counters(hkv)
        s["q_out"] = torch.zeros((hq, D), dtype=torch.float16, device="cuda")
        s["out"] = torch.empty((hkv, hq // hkv, D), dtype=torch.float16, device="cuda")
        s["position"] = torch.tensor([case["pos"]], dtype=torch.int32, device="cuda")
    elif kind == "mlp":
        s["normed"], s["residual_out"], s["ff_down"] = (torch.empty_like(s["residual"]) for _ in range(3))
        s["ff"] = torch.empty((s["down"].shape[1],), dtype=torch.float16, device="cuda")
    else:
        s["token"] = torch.tensor([s["first"]], dtype=torch.int32, device="cuda")
        s["position"] = torch.zeros((1,), dtype=torch.int32, device="cuda")
        s["logits"] = torch.empty((VOCAB,), dtype=torch.float16, device="cuda")
        s["runner"] = ga.Qwen3DecodeRunner(
            layers=s["layers"], embed_tokens=s["embed_tokens"], final_norm=s["final_norm"],
            lm_head=s["lm_head"], inv_freq=s["inv_freq"], token=s["token"], position=s["position"],
            logits=s["logits"], num_q_heads=s["hq"], num_kv_heads=s["hkv"], eps=EPS,
            qk_scale_f16_bits=SCALE_F16_BITS, prime_position=case["pos"])
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "prompt":
        ga.qk_norm_rope_kv_prefill(s["q"], s["k"], s["v"], s["q_weight"], s["k_weight"], s["inv_freq"],
                                   s["q_out"], s["k_cache"], s["v_cache"], EPS, case["start"])
        ga.attend_prefill(s["q_out"], s["k_cache"], s["v_cache"], s["out"], case["start"],
                          sched_counters=s["counters"])
        return {"q_out": s["q_out"], "out": s["out"], "k_cache": s["k_cache"], "v_cache": s["v_cache"]}
    if kind == "suffix":
        ga.kv_cache_update_seq(s["k"], s["v"], s["k_cache"], s["v_cache"], case["start"])
        ga.attend_prefill(s["q"], s["k_cache"], s["v_cache"], s["out"], case["start"])
        return {"out": s["out"], "k_cache": s["k_cache"], "v_cache": s["v_cache"]}
    if kind == "decode":
        ga.decode_fused(s["qkv"], s["q_weight"], s["k_weight"], s["inv_freq"], s["q_out"], s["k_cache"],
                        s["v_cache"], s["att"], s["lse"], s["out"], s["counters"], s["position"], EPS,
                        SCALE_F16_BITS, s["hq"], s["hkv"])
        return {"q_out": s["q_out"], "out": s["out"], "k_cache": s["k_cache"], "v_cache": s["v_cache"]}
    if kind == "mlp":
        ga.add_rms_norm_decode(s["residual"], s["x"], s["weight"], s["normed"], s["residual_out"], EPS)
        ga.gemv_silu_mul(s["gate_up"], s["normed"], s["ff"])
        ga.gemv_f16(s["down"], s["ff"], s["ff_down"])
        return {"normed": s["normed"], "residual": s["residual_out"], "ff": s["ff"], "ff_down": s["ff_down"]}
    # The step waits for its token, as a program that streams text does.
    s["runner"].seed_token(s["first"])
    s["runner"].step(case["pos"])
    return {"logits": s["logits"], "k_all": s["k_all"], "v_all": s["v_all"]}


# ------------------------------------------------------------- what it needs --

def _work_decode(hq, hkv, keys):
    return {"bytes": 2 * 2 * hkv * keys * D + 2 * D * (2 * hq + 2 * hkv + hq), "flops": 4 * D * hq * keys}


def work(case):
    hq, hkv, hidden, inter, _, _ = MODELS[case["model"]]
    kind = case["kind"]
    if kind in ("prompt", "suffix"):
        seq, start = case["seq"], case["start"]
        pairs = seq * start + seq * (seq + 1) // 2
        # q, k, v in; out and the new K/V rows (and q_out) written; the prefix read.
        rows = seq * (2 * hq + 4 * hkv) + (seq * hq if kind == "prompt" else 0) + 2 * hkv * start
        return {"bytes": 2 * D * rows, "flops": 4 * D * hq * pairs}
    if kind == "decode":
        return _work_decode(hq, hkv, case["pos"] + 1)
    if kind == "mlp":
        return {"bytes": 2 * (3 * inter * hidden + 6 * hidden + inter), "flops": 6 * inter * hidden}
    att = _work_decode(hq, hkv, case["pos"] + 1)
    weights = case["layers"] * _layer_weights(case["model"]) + VOCAB * hidden
    return {"bytes": 2 * (weights + VOCAB) + case["layers"] * att["bytes"],
            "flops": 2 * weights + case["layers"] * att["flops"]}


def tolerance(case):
    # About four times what the outputs differ from the 64-bit results by.  A
    # f16 output alone is 2.1e-4 (2-norm) and 4.9e-4 (at most) off.
    if case["kind"] == "step":
        # Every layer's f16 roundings travel through all that follow: logits
        # measured 6e-4 off behind one layer, 1.7e-3 behind 9, 5.6e-3 behind 28.
        return {"rel": 2.5e-3 + 6e-4 * case["layers"], "max": 0.4}
    if case["kind"] == "mlp":
        # Three f16 roundings in a row (normed, ff, ff_down): 5.4e-4.
        return {"rel": 2.2e-3, "max": 1.3e-2}
    # Attention outputs measured 2.6e-4 to 4.1e-4.  The largest differences,
    # 2.4e-2 of the root mean square, are in the first rows of long prompts,
    # whose values are far larger than the rest.
    return {"rel": 1.6e-3, "max": 0.1}


# ------------------------------------------------------------- 64-bit results --

def _exact_rms(x, w):
    x = x.double()
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _exact_norm_rope(x, w, inv_freq, start):
    """x [seq, heads, D]: RMSNorm per head, then rotation by the f32 angles."""
    pos = torch.arange(start, start + x.shape[0], device="cuda", dtype=torch.float32)
    theta = (pos[:, None] * inv_freq[None, :]).double()[:, None, :]
    n = _exact_rms(x, w)
    lo, hi = n[..., :D // 2], n[..., D // 2:]
    return torch.cat([lo * theta.cos() - hi * theta.sin(), hi * theta.cos() + lo * theta.sin()], -1)


def _exact_attention(q, k_cache, v_cache, start, scale):
    """Causal attention of q [seq, hq, D] at positions start.. over the f64 caches."""
    seq, hq, _ = q.shape
    hkv = k_cache.shape[0]
    group = hq // hkv
    out = torch.empty_like(q)
    step = max(1, min(seq, (1 << 25) // (start + seq)))
    for r0 in range(0, seq, step):
        r1 = min(seq, r0 + step)
        keys = start + r1
        ahead = (torch.arange(keys, device="cuda")[None, :]
                 > torch.arange(start + r0, start + r1, device="cuda")[:, None])
        for h in range(hq):
            s = (q[r0:r1, h] @ k_cache[h // group, :keys].T) * scale
            out[r0:r1, h] = torch.softmax(s.masked_fill(ahead, -math.inf), -1) @ v_cache[h // group, :keys]
    return out


def _exact_decode(qkv, q_weight, k_weight, inv_freq, k_cache, v_cache, pos, hq, hkv):
    """(q_out, out [hkv, G, D]) of one decode step; writes the row at pos into the f64 caches."""
    x = qkv.reshape(1, hq + 2 * hkv, D)
    q = _exact_norm_rope(x[:, :hq], q_weight, inv_freq, pos)
    k_cache[:, pos] = _exact_norm_rope(x[:, hq:hq + hkv], k_weight, inv_freq, pos)[0]
    v_cache[:, pos] = x[0, hq + hkv:].double()
    out = _exact_attention(q, k_cache, v_cache, pos, SCALE_F16)
    return q[0], out[0].reshape(hkv, hq // hkv, D)


def _exact_silu_mul(gate, up):
    return gate / (1 + torch.exp(-gate)) * up


def _mv(w, x):
    """w [m, k] f16 times x [k] in 64 bits, a slice of rows at a time."""
    step = max(1, (1 << 27) // w.shape[1])
    return torch.cat([w[i:i + step].double() @ x for i in range(0, w.shape[0], step)])


def _exact_step(case, s):
    hq, hkv = s["hq"], s["hkv"]
    pos = case["pos"]
    k_all, v_all = s["k_all"].double(), s["v_all"].double()
    h = s["embed_tokens"][s["first"]].double()
    for i, layer in enumerate(s["layers"]):
        qkv = _mv(layer["qkv_proj"], _exact_rms(h, layer["input_norm"]))
        _, att = _exact_decode(qkv, layer["q_norm"], layer["k_norm"], s["inv_freq"], k_all[i], v_all[i],
                               pos, hq, hkv)
        h = h + _mv(layer["o_proj"], att.reshape(-1))
        gate, up = _mv(layer["gate_up_proj"], _exact_rms(h, layer["post_attn_norm"])).chunk(2)
        h = h + _mv(layer["down_proj"], _exact_silu_mul(gate, up))
    return {"logits": _mv(s["lm_head"], _exact_rms(h, s["final_norm"])), "k_all": k_all, "v_all": v_all}


def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "step":
        return _exact_step(case, s)
    if kind == "mlp":
        r = s["residual"].double() + s["x"].double()
        normed = _exact_rms(r, s["weight"])
        gate, up = _mv(s["gate_up"], normed).chunk(2)
        ff = _exact_silu_mul(gate, up)
        return {"normed": normed, "residual": r, "ff": ff, "ff_down": _mv(s["down"], ff)}
    k_cache, v_cache = s["k_cache"].double(), s["v_cache"].double()
    if kind == "decode":
        q_out, out = _exact_decode(s["qkv"], s["q_weight"], s["k_weight"], s["inv_freq"], k_cache, v_cache,
                                   case["pos"], s["hq"], s["hkv"])
        return {"q_out": q_out, "out": out, "k_cache": k_cache, "v_cache": v_cache}
    rows = slice(case["start"], case["start"] + case["seq"])
    v_cache[:, rows] = s["v"].double().transpose(0, 1)
    if kind == "suffix":
        k_cache[:, rows] = s["k"].double().transpose(0, 1)
        q = s["q"].double()
    else:
        k_cache[:, rows] = _exact_norm_rope(s["k"], s["k_weight"], s["inv_freq"], case["start"]).transpose(0, 1)
        q = _exact_norm_rope(s["q"], s["q_weight"], s["inv_freq"], case["start"])
    out = _exact_attention(q, k_cache, v_cache, case["start"], 1 / math.sqrt(D))
    got = {"out": out, "k_cache": k_cache, "v_cache": v_cache}
    if kind == "prompt":
        got["q_out"] = q
    return got
