"""What this engine is measured on: passes of whole requests through ``Engine.step``, as a serving program makes them.

A pass takes a batch of prompts in (cut into steps of at most 8,192 tokens), decodes ``new`` tokens for each of them one
step at a time, and ends the requests; it returns the fp32 logits of every step.  The decoded tokens are given (as in a
replay), so that a pass is the same work whatever the logits are.  The models are the ones of ``bench.py`` at its layer
sizes, with one layer of each kind that a design has (four of the Llama decoders') and random weights of the sizes that
the tests use, which keep every branch of order one.

``exact`` is each design in 64 bits, whole sequences without a cache, written down here on its own.
"""
from __future__ import annotations

import math
import zlib
from typing import Callable, Dict, List, Optional, Tuple

import torch

STEP_TOKENS = 8192
PAGE = 16
F64 = torch.float64

# ------------------------------------------------------------------------------------------------ configurations
LLAMA = {
    "1b": dict(model_type="llama", num_hidden_layers=4, hidden_size=2048, num_attention_heads=32, num_key_value_heads=8,
               head_dim=64, intermediate_size=8192, vocab_size=128256, rope_theta=500000.0, rms_norm_eps=1e-5,
               tie_word_embeddings=True, max_position_embeddings=131072,
               rope_scaling=dict(rope_type="llama3", factor=32.0, low_freq_factor=1.0, high_freq_factor=4.0,
                                 original_max_position_embeddings=8192)),
    "8b": dict(model_type="llama", num_hidden_layers=4, hidden_size=4096, num_attention_heads=32, num_key_value_heads=8,
               head_dim=128, intermediate_size=14336, vocab_size=128256, rope_theta=500000.0, rms_norm_eps=1e-5,
               tie_word_embeddings=False, max_position_embeddings=131072,
               rope_scaling=dict(rope_type="llama3", factor=8.0, low_freq_factor=1.0, high_freq_factor=4.0,
                                 original_max_position_embeddings=8192)),
}
# width, feed-forward, heads over key/value heads of 128, window or chunk, ...: bench.py's two sizes of every design
SIZES = {
    "2k": dict(width=2048, vocab=32000, ff=5504, heads=16, kv=4, window=1024, dense=8192, expert=1408, shared=2688,
               ssm_heads=64, q_rank=768, inner=4096, dt_rank=128),
    "4k": dict(width=4096, vocab=32000, ff=9600, heads=32, kv=8, window=2048, dense=14336, expert=2432, shared=4736,
               ssm_heads=128, q_rank=1536, inner=8192, dt_rank=256),
}


def configuration(case: dict) -> dict:
    """The model's config.json as a dict."""
    design, size = case["design"], case["size"]
    if design == "llama":
        return dict(LLAMA[size])
    z = SIZES[size]
    W, H, G, d, ff = z["width"], z["heads"], z["kv"], 128, z["ff"]
    out = {"architecture": design.capitalize(), "vocab": z["vocab"], "width": W}
    gated = {"kind": "dense", "ff": ff}
    if design == "nesilorn":            # latent attention over a window; a dense and a routed feed-forward
        mixer = {"heads": H, "dim": 64, "rot_dim": 32, "vdim": 64, "kv_rank": 224, "scale": 96 ** -0.5,
                 "rot": {"base": 10000.0, "dims": 32}, "mask": {"size": z["window"]}}
        moe = {"kind": "moe", "expert": {"ff": z["expert"], "limit": 7.0}, "router": {"experts": 32, "top": 4}}
        out.update(embedding={"scale": 1.0}, norm={"eps": 1e-6},
                   layers=[{"type": "latent_attention", "mixer": mixer, "mlp": m}
                           for m in ({"kind": "dense", "ff": z["dense"]}, moe)])
    elif design == "rogizen":           # a state-space layer, attention with convolved queries and keys
        attention = {"heads": H, "kv_heads": G, "dim": d, "vdim": d, "conv": 4, "scale": d ** -0.5,
                     "mask": {"size": z["window"]},
                     "rot": {"base": 10000.0, "dims": 64,
                             "scaling": {"factor": 4.0, "original": 4096, "fast": 32.0, "slow": 1.0}}}
        ssm = {"heads": z["ssm_heads"], "vdim": 64, "state": 128, "groups": 8, "norm_groups": 8, "conv": 4}
        out.update(embedding={"scale": 1.0}, norm={"eps": 1e-6}, logit_softcap=50.0,
                   loop={"start": 0, "stop": 2, "times": 1},
                   layers=[{"type": "mamba2", "mixer": ssm, "mlp": gated},
                           {"type": "attention", "mixer": attention, "mlp": gated}])
    elif design == "malinex":           # gated linear attention, attention with sigmoid weights
        attention = {"heads": H, "kv_heads": G, "dim": d, "vdim": d, "scale": d ** -0.5,
                     "q_temp": {"coef": 0.1, "every": 512}}
        gla = {"heads": H, "dim": d, "vdim": d, "tau": 16.0, "rank": 64}
        moe = {"kind": "moe", "router": {"experts": 8, "top": 2}, "expert": {"ff": ff // 2}, "shared": {"ff": ff // 2}}
        out.update(max_positions=8192, norm={"eps": 1e-6}, logit_scale=0.25,
                   layers=[{"type": "gla", "mixer": gla, "mlp": moe},
                           {"type": "attention", "mixer": attention, "mlp": {"kind": "dense", "ff": ff * 3 // 2}}])
    elif design == "sikazen":           # attention over a window and pooled blocks, latent attention, HGRN2
        attention = {"heads": H, "kv_heads": G, "dim": d, "vdim": d, "scale": d ** -0.5 * 4,
                     "mask": {"size": z["window"], "pool": 64}, "rot": {"base": 10000.0, "dims": d, "scaling": {"factor": 4.0}}}
        latent = {"heads": H, "dim": 64, "rot_dim": 32, "vdim": 64, "kv_rank": 224, "q_rank": z["q_rank"],
                  "scale": 96 ** -0.5, "rot": {"base": 10000.0, "dims": 32}}
        hgrn2 = {"heads": H, "dim": d, "vdim": d}
        out.update(embedding={"scale": 1.0}, norm={"eps": 1e-6}, token_side={"dim": 256},
                   loop={"start": 0, "stop": 3, "times": 1},
                   layers=[{"type": k, "mixer": m, "mlp": gated}
                           for k, m in (("attention", attention), ("latent_attention", latent), ("hgrn2", hgrn2))])
    elif design == "pamazen":           # four streams; window attention beside the delta rule, mixed values; grouped experts
        heads = {"heads": H, "kv_heads": G, "dim": d, "vdim": d, "scale": d ** -0.5}
        attention = dict(heads, v_mix=True, rot={"base": 10000.0, "dims": d // 2, "scaling": {"factor": 2.0}})
        side = {"left": dict(heads, softcap=30.0, mask={"size": z["window"], "keep_first": 8}),
                "right": {"heads": H, "dim": d, "rank": 64}, "left_scale": 1.0, "right_scale": 0.8}
        moe = {"kind": "moe", "expert": {"ff": z["expert"]}, "shared": {"ff": z["shared"]},
               "router": {"experts": 20, "identity": 4, "top": 2, "groups": {"count": 3, "keep": 2}}}
        out.update(norm={"eps": 1e-5}, streams=4, residual_mult=0.6, logit_softcap=25.0,
                   layers=[{"type": k, "mixer": m, "mlp": moe}
                           for k, m in (("parallel", side), ("attention", attention), ("attention", attention))])
    elif design == "mirovik":           # attention with a distance bias beside retention, the selective scan
        R = H // 2
        side = {"left": {"heads": H, "kv_heads": G, "dim": d, "vdim": d, "scale": d ** -0.5, "bias_max": 256, "buckets": 40},
                "right": {"heads": R, "dim": d, "vdim": d, "decay": [1.0 - 2.0 ** (-5 - 4 * i / R) for i in range(R)],
                          "rot": {"base": 10000.0, "dims": d}}, "left_scale": 1.0, "right_scale": 0.8}
        scan = {"inner": z["inner"], "state": 16, "dt_rank": z["dt_rank"], "conv": 4}
        moe = {"kind": "moe", "expert": {"ff": z["expert"]}, "shared": {"ff": z["shared"]},
               "router": {"experts": 16, "top": 2}}
        out.update(norm={"eps": 1e-5}, embedding={"scale": float(W) ** 0.5}, loop={"start": 0, "stop": 2, "times": 1},
                   layers=[{"type": "parallel", "mixer": side, "mlp": {"kind": "dense", "ff": ff * 3 // 2}},
                           {"type": "mamba1", "mixer": scan, "mlp": moe}])
    else:
        raise ValueError(design)
    return out


# ------------------------------------------------------------------------------------------------ cases
def _case(name: str, design: str, size: str, requests: int, prompt: int, new: int, dtype: str = "bfloat16") -> dict:
    return {"name": name, "design": design, "size": size, "requests": requests, "prompt": prompt, "new": new, "dtype": dtype}


def listed() -> List[dict]:
    return [
        # one person at a small model: a short prompt, then tokens one at a time; latency and launches
        _case("llama 1b - one request", "llama", "1b", 1, 24, 24),
        # the headline of bench.py: eight requests decode after prompts of about 512 tokens
        _case("llama 8b - 8 requests", "llama", "8b", 8, 512, 32),
        # a full serving batch: 64 requests with short prompts of uneven length
        _case("llama 8b - 64 requests", "llama", "8b", 64, 120, 32),
        # a prompt of ordinary length, and the first token (the prefill of bench.py)
        _case("llama 8b - prompt of 2048", "llama", "8b", 1, 2048, 0),
        # a long document in one step
        _case("llama 8b - prompt of 8192", "llama", "8b", 1, 8192, 0),
        # the 32-bit path, as a check of numbers is run: a few odd prompts and a few tokens
        _case("llama 1b in 32 bits", "llama", "1b", 3, 61, 4, "float32"),
        # the further designs, each with prompts and decoding: a long prompt and its answer, or a batch of requests
        _case("nesilorn 2k - prompt of 2047", "nesilorn", "2k", 1, 2047, 16),
        _case("rogizen 2k - 8 requests", "rogizen", "2k", 8, 256, 16),
        _case("malinex 2k - 2 requests", "malinex", "2k", 2, 1000, 8),
        _case("sikazen 2k - prompt of 3000", "sikazen", "2k", 1, 3000, 8),
        _case("pamazen 4k - 16 requests", "pamazen", "4k", 16, 128, 16),
        _case("mirovik 2k - 32 requests", "mirovik", "2k", 32, 64, 16),
    ]


def draw(rng) -> dict:
    def spread(lo: float, hi: float) -> int:
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    design = rng.choice(["llama", "llama", "nesilorn", "rogizen", "malinex", "sikazen", "pamazen", "mirovik"])
    size = rng.choice(["1b", "8b"] if design == "llama" else ["2k", "4k"])
    kind = rng.choice(["prompt", "decode", "both"])
    if kind == "prompt":                # one or a few prompts, nothing decoded
        requests = rng.choice([1, 1, 2, 3])
        prompt, new = spread(17, 4096 / requests), 0
    elif kind == "decode":              # short prompts, many tokens
        requests = spread(1, 64)
        prompt, new = spread(5, 96), rng.randint(12, 32)
    else:
        requests = spread(1, 24)
        prompt, new = spread(32, 4096 / requests), rng.randint(2, 16)
    dtype = "bfloat16"
    if size == "1b" and rng.random() < 0.25:
        dtype, requests, prompt, new = "float32", min(requests, 4), min(prompt, 96), min(new, 6)
    return {"design": design, "size": size, "requests": requests, "prompt": prompt, "new": new, "dtype": dtype}


def prompt_lengths(case: dict) -> List[int]:
    """One request has the prompt as stated; several have lengths from half to one and a half times it."""
    n, L = case["requests"], case["prompt"]
    if n == 1:
        return [L]
    return [max(1, int(L * (0.5 + (i * 0.6180339887) % 1.0))) for i in range(n)]


def prompt_steps(case: dict) -> List[List[int]]:
    """The requests whose prompts go in together: as many as fit into a step."""
    steps: List[List[int]] = []
    room = 0
    for i, n in enumerate(prompt_lengths(case)):
        if n > room:
            steps.append([])
            room = STEP_TOKENS
        steps[-1].append(i)
        room -= n
    return steps


def vocabulary(case: dict) -> int:
    return LLAMA[case["size"]]["vocab_size"] if case["design"] == "llama" else SIZES[case["size"]]["vocab"]


def tokens(case: dict, seed: int) -> Tuple[List[List[int]], List[List[int]]]:
    """(every request's prompt, the tokens it decodes)."""
    g = torch.Generator().manual_seed(seed * 7919 + 13)
    V = vocabulary(case)
    ids = [torch.randint(0, V, (n + case["new"],), generator=g).tolist() for n in prompt_lengths(case)]
    lens = prompt_lengths(case)
    return [t[:n] for t, n in zip(ids, lens)], [t[n:] for t, n in zip(ids, lens)]


# ------------------------------------------------------------------------------------------------ tensors
def tensor_shapes(cfg: dict) -> Dict[str, tuple]:
    """Name in the file -> shape, of every tensor of a model."""
    if "architecture" not in cfg:
        H, I, V = cfg["hidden_size"], cfg["intermediate_size"], cfg["vocab_size"]
        nq, nk = cfg["num_attention_heads"] * cfg["head_dim"], cfg["num_key_value_heads"] * cfg["head_dim"]
        out = {"model.embed_tokens.weight": (V, H), "model.norm.weight": (H,)}
        if not cfg["tie_word_embeddings"]:
            out["lm_head.weight"] = (V, H)
        for i in range(cfg["num_hidden_layers"]):
            p = f"model.layers.{i}."
            out.update({p + "input_layernorm.weight": (H,), p + "post_attention_layernorm.weight": (H,),
                        p + "self_attn.q_proj.weight": (nq, H), p + "self_attn.k_proj.weight": (nk, H),
                        p + "self_attn.v_proj.weight": (nk, H), p + "self_attn.o_proj.weight": (H, nq),
                        p + "mlp.gate_proj.weight": (I, H), p + "mlp.up_proj.weight": (I, H),
                        p + "mlp.down_proj.weight": (H, I)})
        return out
    arch, W, V = cfg["architecture"], cfg["width"], cfg["vocab"]
    scalar_norm = arch in ("Sikazen", "Pamazen")
    norm = () if scalar_norm else (W,)
    out = {"embed": (V, W), "final.norm": norm}
    if arch in ("Rogizen", "Malinex", "Sikazen", "Pamazen"):
        out["head"] = (V, W)
    if arch == "Rogizen":
        out["loop.in"] = (W, 2 * W)
    if arch == "Malinex":
        out["pos"] = (cfg["max_positions"], W)
    if arch == "Sikazen":
        out["side.embed"] = (V, cfg["token_side"]["dim"] * len(cfg["layers"]))
    if arch == "Mirovik":
        out["loop.step"] = (cfg["loop"]["times"], W)
    for i, layer in enumerate(cfg["layers"]):
        p, kind = f"l{i}.", layer["type"]
        m, f = layer["mixer"], layer["mlp"]
        q = p + "mix."
        out.update({p + "norm1": norm, p + "norm2": norm})
        if arch in ("Malinex", "Mirovik"):
            out.update({p + "norm1b": (W,), p + "norm2b": (W,)})
        if arch == "Malinex":
            out.update({p + "rg1": (W, W), p + "rg1.b": (W,), p + "rg2": (W, W), p + "rg2.b": (W,)})
        if arch == "Pamazen":
            S = cfg["streams"]
            for h in ("hc1.", "hc2."):
                out.update({p + h + "in": (S,), p + h + "out": (S,), p + h + "mix": (S, S)})
        if arch == "Sikazen":
            t = cfg["token_side"]["dim"]
            out.update({p + "side.gate": (t, W), p + "side.proj": (W, t), p + "side.norm": (W,)})
        # ---- mixers
        if kind == "latent_attention":
            H, dn, dr, dv, rk = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
            out.update({q + "dkv": (rk + dr, W), q + "dkv.norm": (rk,), q + "uk": (H * dn, rk), q + "uv": (H * dv, rk),
                        q + "o": (W, H * dv)})
            if arch == "Nesilorn":
                out.update({q + "q": (H * (dn + dr), W), q + "g": (H * dv, W)})
            else:
                out.update({q + "dq": (m["q_rank"], W), q + "dq.norm": (m["q_rank"],),
                            q + "uq": (H * (dn + dr), m["q_rank"]), q + "sink": (H,)})
        elif kind == "mamba2":
            inner, gn, n = m["heads"] * m["vdim"], m["groups"] * m["state"], m["heads"]
            out.update({q + "in": (2 * inner + 2 * gn + n, W), q + "conv": (inner + 2 * gn, m["conv"]),
                        q + "conv.b": (inner + 2 * gn,), q + "dt_bias": (n,), q + "A_log": (n,), q + "D": (n,),
                        q + "norm": (inner,), q + "o": (W, inner)})
        elif kind == "mamba1":
            I, R, n = m["inner"], m["dt_rank"], m["state"]
            out.update({q + "in": (2 * I, W), q + "conv": (I, m["conv"]), q + "conv.b": (I,), q + "x": (R + 2 * n, I),
                        q + "dt": (I, R), q + "dt.b": (I,), q + "A_log": (I, n), q + "D": (I,), q + "o": (W, I)})
        elif kind == "gla":
            nq, nv = m["heads"] * m["dim"], m["heads"] * m["vdim"]
            out.update({q + "q": (nq, W), q + "k": (nq, W), q + "v": (nv, W), q + "g": (nv, W), q + "o": (W, nv),
                        q + "norm": (m["vdim"],), q + "a1": (m["rank"], W), q + "a2": (nq, m["rank"]), q + "a2.b": (nq,)})
        elif kind == "hgrn2":
            H, d, dv = m["heads"], m["dim"], m["vdim"]
            out.update({q + "q": (H * d, W), q + "f": (H * d, W), q + "f.b": (H * d,), q + "lower": (H * d,),
                        q + "v": (H * dv, W), q + "norm": (dv,), q + "o": (W, H * dv)})
        elif kind == "attention":
            H, G, d, dv = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
            out.update({q + "q": (H * d, W), q + "k": (G * d, W), q + "o": (W, H * dv)})
            if arch != "Rogizen":
                out[q + "v"] = (G * dv, W)
            if arch == "Rogizen":
                out.update({q + "q.b": (H * d,), q + "k.b": (G * d,), q + "q.norm": (d,), q + "k.norm": (d,),
                            q + "q.conv": (H * d, m["conv"]), q + "k.conv": (G * d, m["conv"]), q + "o.b": (W,)})
            elif arch == "Pamazen":
                if any(x["type"] == "attention" for x in cfg["layers"][:i]):    # the first such layer has nothing to mix with
                    out[q + "vmix"] = ()
            else:
                out.update({q + "q.b": (H * d,), q + "k.b": (G * d,), q + "v.b": (G * dv,)})
            if arch == "Malinex":
                out.update({q + "q.norm": (H * d,), q + "k.norm": (G * d,), q + "r1": (H,), q + "r2": (H,), q + "pb": (H,),
                            q + "g": (H, W)})
        else:                           # two mixers side by side
            lt, rt = m["left"], m["right"]
            H, G, d, n = lt["heads"], lt["kv_heads"], lt["dim"], rt["heads"] * rt["dim"]
            a, b = q + "left.", q + "right."
            out.update({a + "q": (H * d, W), a + "k": (G * d, W), a + "o": (W, H * d), b + "k": (n, W), b + "v": (n, W),
                        b + "g": (n, W), b + "o": (W, n)})
            if arch == "Pamazen":
                out.update({a + "q.norm": (d,), a + "k.norm": (d,), a + "sink": (H,), b + "r": (n, W), b + "a": (n, W),
                            b + "a.b": (n,), b + "w1": (rt["rank"], W), b + "w2": (n, rt["rank"]), b + "w0": (n,),
                            b + "norm": (n,)})
            else:
                out.update({a + "v": (G * d, W), a + "g": (H * d, W), a + "q.norm": (H * d,), a + "k.norm": (G * d,),
                            a + "rel": (lt["buckets"], H), b + "q": (n, W)})
        # ---- feed-forwards
        q = p + "mlp."
        three = arch in ("Rogizen", "Sikazen")
        names = lambda three: ("gate", "up") if three else ("up",)                                  # noqa: E731
        if f["kind"] == "dense":
            out.update({q + x: (f["ff"], W) for x in names(three)})
            out[q + "down"] = (W, f["ff"])
        else:
            E, three = f["router"]["experts"], arch != "Malinex"
            blocks = [(f"e{e}.", f["expert"]["ff"]) for e in range(E)]
            blocks += [("shared.", f["shared"]["ff"])] if f.get("shared") else []
            for pre, ff in blocks:
                out.update({q + pre + x: (ff, W) for x in names(three)})
                out[q + pre + "down"] = (W, ff)
            total = E + f["router"].get("identity", 0)
            out[q + "router"] = (total, W)
            if arch in ("Malinex", "Pamazen"):
                out[q + "correction"] = (total,)
            if arch == "Nesilorn":
                out[q + "router.b"] = (total,)
            if arch == "Pamazen":
                out[q + "shared.sg"] = (1, W)
    return out


def specialities(cfg: dict, seed: int) -> Optional[Tuple[torch.Tensor, torch.Tensor]]:
    """What makes routers sure of their choice, as a trained one is (a near tie that two roundings decide differently
    would say nothing about either): as many directions [K, W] as experts, of which every token's embedding has one,
    and how strongly each expert [E, K] answers to each: ``top`` of them, the rest not at all."""
    routers = [x["mlp"]["router"] for x in cfg.get("layers", []) if x["mlp"]["kind"] == "moe"]
    if not routers:
        return None
    E, top, W = routers[0]["experts"] + routers[0].get("identity", 0), routers[0]["top"], cfg["width"]
    g = torch.Generator(device="cuda").manual_seed((seed * 1000003 + 11) & 0x7FFFFFFF)
    u = torch.empty((E, W), dtype=torch.float32, device="cuda").normal_(0.0, W ** -0.5, generator=g)
    strength = torch.zeros((E, E), device="cuda")
    for k in range(E):
        for j in range(top):
            strength[(5 * k + 3 * j) % E, k] = 3.6 - j * (1.2 / max(top - 1, 1))
    return u, strength


def tensor(cfg: dict, name: str, shape: tuple, seed: int) -> torch.Tensor:
    """One tensor in bfloat16 on the GPU, from (seed, name) alone."""
    g = torch.Generator(device="cuda").manual_seed((seed * 1000003 + zlib.crc32(name.encode())) & 0x7FFFFFFF)
    arch, last = cfg.get("architecture", "Llama"), name.rsplit(".", 1)[-1]

    def normal(std: float = 1.0, mean: float = 0.0) -> torch.Tensor:
        return torch.empty(shape, dtype=torch.float32 if len(shape) < 2 else torch.bfloat16, device="cuda").normal_(
            mean, std, generator=g)

    def uniform(lo: float, hi: float) -> torch.Tensor:
        return torch.empty(shape, dtype=torch.float32, device="cuda").uniform_(lo, hi, generator=g)

    if arch == "Llama":
        t = normal(0.2, 1.0) if len(shape) == 1 else normal(1.0 if "embed" in name else shape[-1] ** -0.5)
        if name == "model.embed_tokens.weight" and cfg["tie_word_embeddings"]:
            t = normal(shape[-1] ** -0.5 * 8)
    elif "norm" in last:
        offset = arch == "Nesilorn" and name.endswith("dkv.norm") or name.endswith((".q.norm", ".k.norm"))
        t = normal(0.2, 1.0 if offset or arch not in ("Nesilorn", "Mirovik") else 0.0)
    elif ".hc" in name:
        S = cfg["streams"]
        t = torch.eye(S, device="cuda") + normal(0.15).float() if last == "mix" else \
            (1.0 / S if last == "in" else 1.0) * normal(0.4, 1.0)
    elif last == "A_log" and len(shape) == 2:
        t = torch.log(torch.arange(1, shape[1] + 1, dtype=torch.float32, device="cuda"))[None, :] + normal(0.3)
    elif last == "A_log":
        t = torch.log(uniform(0.5, 3.5))
    elif last == "dt_bias":
        t = uniform(-2.0, 0.0)
    elif last == "D":
        t = uniform(0.5, 1.5)
    elif name.endswith("dt.b"):
        t = uniform(-4.0, 0.0)
    elif name.endswith("a2.b"):
        t = uniform(1.0, 4.0)
    elif name.endswith("f.b"):
        t = uniform(-1.0, 3.0)
    elif name.endswith("a.b"):
        t = normal()
    elif last == "b":
        t = normal(0.3)
    elif last in ("sink",):
        t = normal()
    elif last == "lower":
        t = uniform(0.0, 0.9)
    elif last == "r1":
        t = uniform(0.2, 1.0)
    elif last == "r2":
        t = uniform(0.05, 0.55)
    elif last == "pb":
        t = uniform(-3.0, -1.0)
    elif last == "w0":
        t = uniform(-4.0, 1.0)
    elif last == "vmix":
        t = uniform(0.2, 0.8)
    elif last == "rel":
        t = normal(1.5)
    elif last == "correction":
        t = normal(0.02)
    elif name == "loop.step":
        t = normal(0.5)
    elif last == "pos":
        t = normal(0.5)
    elif last == "embed":
        std = shape[-1] ** -0.5 if arch == "Mirovik" else 1.0
        t, special = normal(std), specialities(cfg, seed) if name == "embed" else None
        if special is not None:
            t *= 0.5 ** 0.5
            rows = (special[0] * (std * (0.5 * shape[-1]) ** 0.5)).to(t.dtype)
            t += rows[torch.arange(shape[0], device="cuda") % rows.shape[0]]
    elif name == "loop.in":
        t = normal((shape[1] / 2) ** -0.5)
    elif last == "router":
        u, strength = specialities(cfg, seed)
        t = strength @ u * (2.5 * shape[-1] ** -0.5) + normal(0.2 * shape[-1] ** -0.5).float()
    elif arch == "Nesilorn" and ".mlp.e" in name and last in ("gate", "up"):
        t = normal(2.0 * shape[-1] ** -0.5)
    elif arch == "Mirovik" and name.endswith(".right.k"):
        # a token's own key lies along its query, as what a retention head reads would otherwise be a difference of
        # nearly equal terms
        t = 0.7 * tensor(cfg, name[:-1] + "q", shape, seed).float() + normal(0.7 * shape[-1] ** -0.5)
    elif arch == "Pamazen" and name.endswith(".right.k"):
        t = normal(0.5 * shape[-1] ** -0.5)
    elif (arch == "Pamazen" and last in ("q", "k")) or (arch == "Sikazen" and last in ("q", "k", "uq", "uk")):
        t = normal(1.5 * shape[-1] ** -0.5)
    else:
        t = normal(shape[-1] ** -0.5)
    return t.to(torch.bfloat16)


# ------------------------------------------------------------------------------------------------ the engine's pass
def prepare(case: dict, seed: int) -> dict:
    """A loaded engine, the prompts and the tokens to decode."""
    from infernum_amd import CacheConfig, Engine
    from infernum_amd.config.registry import config_from_dict, model_spec_for
    from infernum_amd.engine import StepEntry
    from infernum_amd.kernels.api import load_library
    from infernum_amd.models.model import DecoderModel
    cfg = configuration(case)
    lens, new = prompt_lengths(case), case["new"]
    rt = Engine.runtime(case["dtype"], max_tokens_per_step=STEP_TOKENS)
    load_library("core")
    model = DecoderModel(model_spec_for(config_from_dict(cfg)), rt)
    weights = {name: tensor(cfg, name, shape, seed).to(rt.dtype) for name, shape in tensor_shapes(cfg).items()}
    if cfg.get("tie_word_embeddings"):
        weights["lm_head.weight"] = weights["model.embed_tokens.weight"]
    for name, spec in model.expected_weights().items():
        if name not in weights and spec.fallback is not None:
            weights[name] = weights[spec.fallback]
    model.load_weights(weights)
    pages = sum(-(-(n + new) // PAGE) + 1 for n in lens) + 4
    engine = Engine(model, CacheConfig(page_size=PAGE, num_pages=pages, num_state_slots=len(lens) + 1))
    prompts, more = tokens(case, seed)
    steps = [[StepEntry(i, prompts[i], [len(prompts[i]) - 1]) for i in group] for group in prompt_steps(case)]
    steps += [[StepEntry(i, [more[i][t]], [0]) for i in range(len(lens))] for t in range(new)]
    return {"engine": engine, "steps": steps, "requests": len(lens)}


def run(state: dict) -> List[torch.Tensor]:
    """The prompts in, ``new`` tokens of every request, the requests ended: the logits of every step."""
    engine = state["engine"]
    logits = [engine.step(entries) for entries in state["steps"]]
    for i in range(state["requests"]):
        engine.end(i)
    return logits


# ------------------------------------------------------------------------------------------------ what a pass needs
def work(case: dict) -> dict:
    """Every step reads the weights that its tokens multiply with once (of routed experts those that its tokens choose,
    as many as an even choice touches), the keys, values and states of its requests, and writes its logits; two
    operations a weight and token, four a query, key and head dimension."""
    cfg, lens, elem = configuration(case), prompt_lengths(case), 4 if case["dtype"] == "float32" else 2
    llama = case["design"] == "llama"
    V = vocabulary(case)
    W = cfg["hidden_size"] if llama else cfg["width"]
    dense = routed = 0.0
    experts, top = 1, 0
    for layer in ([] if llama else cfg["layers"]):
        if layer["mlp"]["kind"] == "moe":
            r = layer["mlp"]["router"]
            experts, top = r["experts"] + r.get("identity", 0), r["top"]
    for name, shape in tensor_shapes(cfg).items():
        if len(shape) < 2 or "embed" in name or name in ("head", "lm_head.weight", "pos"):
            continue
        n = float(shape[0] * shape[1])
        if ".mlp.e" in name:
            routed += n
        else:
            dense += n
    # per attention-like mixer: operations a pair, values cached a token, window; per recurrence: values of its state
    mixers = []
    if llama:
        mixers = [(4.0 * cfg["num_attention_heads"] * cfg["head_dim"], 2 * cfg["num_key_value_heads"] * cfg["head_dim"],
                   0)] * cfg["num_hidden_layers"]
    state = 0.0
    for layer in ([] if llama else cfg["layers"]):
        kind, m = layer["type"], layer["mixer"]
        if kind == "latent_attention":
            mixers.append((2.0 * m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"]), m["kv_rank"] + m["rot_dim"],
                           (m.get("mask") or {}).get("size", 0)))
        elif kind == "attention":
            mixers.append((4.0 * m["heads"] * m["dim"], 2 * m["kv_heads"] * m["dim"], (m.get("mask") or {}).get("size", 0)))
        elif kind == "parallel":
            lt, rt = m["left"], m["right"]
            mixers.append((4.0 * lt["heads"] * lt["dim"], 2 * lt["kv_heads"] * lt["dim"], (lt.get("mask") or {}).get("size", 0)))
            state += rt["heads"] * rt["dim"] * rt["dim"]
        elif kind == "mamba1":
            state += m["inner"] * m["state"]
        elif kind == "mamba2":
            state += m["heads"] * m["vdim"] * m["state"]
        else:
            state += m["heads"] * m["dim"] * m["vdim"]
    total_bytes = total_flops = 0.0

    def step(before: List[int], count: List[int]) -> None:
        nonlocal total_bytes, total_flops
        n, rows = sum(count), len(count)
        touched = 1.0 - (1.0 - top / experts) ** n if top else 0.0
        total_bytes += (dense + routed * touched + V * W + n * W) * elem + rows * V * 4
        total_flops += 2.0 * n * (dense + routed * top / experts) + 2.0 * rows * V * W + 6.0 * n * state
        total_bytes += 8.0 * rows * state
        for ops, cached, window in mixers:
            for b, c in zip(before, count):
                full = b + c if not window else min(b + c, window + c - 1)
                total_bytes += (full + c) * cached * elem
                pairs = sum(min(b + j + 1, window) for j in range(c)) if window else c * b + c * (c + 1) / 2.0
                total_flops += ops * pairs

    for group in prompt_steps(case):
        step([0] * len(group), [lens[i] for i in group])
    for t in range(case["new"]):
        step([n + t for n in lens], [1] * len(lens))
    return {"bytes": total_bytes, "flops": total_flops}


def tolerance(case: dict) -> dict:
    # the 32-bit path, 7e-7 from the exact logits here: sums of up to 8,192 products in another order
    if case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 1e-4}
    # every activation between two operations is rounded to bfloat16 (2^-9): over these layers that leaves the logits
    # 0.002 to 0.008 of their root mean square from the exact ones, and as far from another rounding's; the worst of
    # some millions of values is about six times that
    return {"rel": 0.02, "max": 0.2}


# ------------------------------------------------------------------------------------------------ 64 bits
Spans = List[Tuple[int, int]]


class _Exact:
    """A model in 64 bits over whole sequences that lie one after the other: x [N, W], ``spans`` their places."""

    def __init__(self, cfg: dict, seed: int, lens: List[int]):
        self.cfg, self.seed = cfg, seed
        self.shapes = tensor_shapes(cfg)
        self.spans: Spans = []
        for n in lens:
            at = self.spans[-1][1] if self.spans else 0
            self.spans.append((at, at + n))
        self.pos = torch.cat([torch.arange(n, device="cuda") for n in lens])
        self.shared: dict = {}
        self.eps = cfg["rms_norm_eps"] if "rms_norm_eps" in cfg else cfg["norm"]["eps"]

    def w(self, name: str) -> torch.Tensor:
        return tensor(self.cfg, name, self.shapes[name], self.seed).to(F64)

    def lin(self, x: torch.Tensor, name: str) -> torch.Tensor:
        return x @ self.w(name).T

    def unit(self, x: torch.Tensor) -> torch.Tensor:
        return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + self.eps)

    def each(self, fn: Callable, *xs: torch.Tensor) -> torch.Tensor:
        return torch.cat([fn(*(x[a:b] for x in xs)) for a, b in self.spans])

    # ---- pieces
    def rotate(self, x: torch.Tensor, freq: torch.Tensor, pairs: bool, mag: float = 1.0) -> torch.Tensor:
        """x [N, heads, n]: the first 2 len(freq) values of a head, neighbours (``pairs``) or halves together."""
        h = freq.numel()
        a = self.pos.to(F64)[:, None, None] * freq
        c, s = torch.cos(a) * mag, torch.sin(a) * mag
        out = x.clone()
        one, two = (slice(0, 2 * h, 2), slice(1, 2 * h, 2)) if pairs else (slice(0, h), slice(h, 2 * h))
        u, v = x[..., one], x[..., two]
        out[..., one], out[..., two] = u * c - v * s, v * c + u * s
        return out

    def attend(self, q, k, v, scale: float, seen: Optional[Callable] = None, sink=None, cap: float = 0.0,
               weigh: Optional[Callable] = None) -> torch.Tensor:
        """q [N, H, d], k [N, G, d], v [N, G, dv] -> [N, H dv], every sequence by itself, a block of queries and a head
        at a time.  ``seen(i, j)``: which keys beside j <= i; ``weigh(h, scores, i, j)``: scores -> weights."""
        H, G = q.shape[1], k.shape[1]

        def one(q, k, v):
            T = q.shape[0]
            out = torch.empty((T, H, v.shape[2]), dtype=F64, device="cuda")
            j = torch.arange(T, device="cuda")[None, :]
            for a in range(0, T, 2048):
                i = torch.arange(a, min(a + 2048, T), device="cuda")[:, None]
                ok = j <= i
                if seen is not None:
                    ok = ok & seen(i, j)
                for h in range(H):
                    s = q[a:a + 2048, h] @ k[:, h // (H // G)].T * scale
                    if weigh is not None:
                        p = weigh(h, s, i, j, ok)
                    else:
                        if cap:
                            s = cap * torch.tanh(s / cap)
                        s = s.masked_fill(~ok, -math.inf)
                        top = s.max(dim=1, keepdim=True).values
                        top = top if sink is None else torch.maximum(top, sink[h])
                        e = torch.exp(s - top)
                        p = e / (e.sum(dim=1, keepdim=True) + (0.0 if sink is None else torch.exp(sink[h] - top)))
                    out[a:a + 2048, h] = p @ v[:, h // (H // G)]
            return out.reshape(T, -1)
        return self.each(one, q, k, v)

    def conv(self, x: torch.Tensor, taps: torch.Tensor) -> torch.Tensor:
        K = taps.shape[1]

        def one(x):
            p = torch.cat([x.new_zeros((K - 1, x.shape[1])), x])
            return sum(p[j:j + x.shape[0]] * taps[:, j] for j in range(K))
        return self.each(one, x)

    def recur(self, q, k, v, decay: Callable, first: torch.Tensor) -> torch.Tensor:
        """S <- decay(t, S) + k_t v_t^T, o_t = S^T q_t for every head; q, k [N, H, d], v [N, H, dv]; ``decay(t, S)``
        with t the token's row."""
        out = torch.empty(q.shape[:2] + v.shape[2:], dtype=F64, device="cuda")
        for a, b in self.spans:
            S = first.clone()
            for t in range(a, b):
                S = decay(t, S) + k[t][:, :, None] * v[t][:, None, :]
                out[t] = (S * q[t][:, :, None]).sum(dim=1)
        return out

    def frequencies(self, rot: dict) -> torch.Tensor:
        f = float(rot["base"]) ** (-torch.arange(0, rot["dims"], 2, dtype=F64, device="cuda") / rot["dims"])
        sc = rot.get("scaling") or {}
        return f / float(sc.get("factor", 1.0)) if "original" not in sc else f

    # ---- mixers
    def llama_attention(self, a, p):
        c = self.cfg
        H, G, d = c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"]
        q, k, v = (self.lin(a, p + f"self_attn.{n}_proj.weight").view(-1, h, d) for n, h in (("q", H), ("k", G), ("v", G)))
        sc, freq = c["rope_scaling"], []
        for i in range(d // 2):
            f = c["rope_theta"] ** (-2.0 * i / d)
            turns = sc["original_max_position_embeddings"] * f / (2.0 * math.pi)
            r = min(max((turns - sc["low_freq_factor"]) / (sc["high_freq_factor"] - sc["low_freq_factor"]), 0.0), 1.0)
            freq.append(f * r + f / sc["factor"] * (1.0 - r))
        freq = torch.tensor(freq, dtype=F64, device="cuda")
        o = self.attend(self.rotate(q, freq, False), self.rotate(k, freq, False), v, d ** -0.5)
        return self.lin(o, p + "self_attn.o_proj.weight")

    def latent(self, a, p, m):
        H, dn, dr, dv, rk = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
        nes = self.cfg["architecture"] == "Nesilorn"
        q = self.lin(a, p + "q") if nes else self.lin(self.unit(self.lin(a, p + "dq")) * self.w(p + "dq.norm"), p + "uq")
        q = q.view(-1, H, dn + dr)
        low = self.lin(a, p + "dkv")
        c = self.unit(low[:, :rk]) * self.w(p + "dkv.norm")
        freq = self.frequencies(m["rot"])
        k_rot = self.rotate(low[:, None, rk:], freq, not nes).expand(-1, H, -1)
        q = torch.cat([q[..., :dn], self.rotate(q[..., dn:], freq, not nes)], dim=-1)
        k = torch.cat([self.lin(c, p + "uk").view(-1, H, dn), k_rot], dim=-1)
        size = (m.get("mask") or {}).get("size")
        o = self.attend(q, k, self.lin(c, p + "uv").view(-1, H, dv), m["scale"],
                        (lambda i, j: i - j < size) if size else None, None if nes else self.w(p + "sink"))
        if nes:
            o = o * torch.sigmoid(self.lin(a, p + "g"))
        return self.lin(o, p + "o")

    def conv_attention(self, a, p, m):
        H, G, d = m["heads"], m["kv_heads"], m["dim"]
        q = self.conv(self.lin(a, p + "q") + self.w(p + "q.b"), self.w(p + "q.conv")).view(-1, H, d)
        k = self.conv(self.lin(a, p + "k") + self.w(p + "k.b"), self.w(p + "k.conv")).view(-1, G, d)
        rot = m["rot"]
        sc, f, dims = rot["scaling"], self.frequencies(rot), rot["dims"]
        turn = lambda t: dims * math.log(sc["original"] / (2.0 * math.pi * t)) / (2.0 * math.log(rot["base"]))   # noqa: E731
        lo, hi = max(math.floor(turn(sc["fast"])), 0), min(math.ceil(turn(sc["slow"])), dims - 1)
        r = ((torch.arange(dims // 2, dtype=F64, device="cuda") - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
        f, mag = f / sc["factor"] * r + f * (1.0 - r), 0.1 * math.log(sc["factor"]) + 1.0
        size = m["mask"]["size"]
        o = self.attend(self.rotate(self.unit(q) * self.w(p + "q.norm"), f, True, mag),
                        self.rotate(self.unit(k) * self.w(p + "k.norm"), f, True, mag), k, m["scale"],
                        lambda i, j: i // size == j // size)
        return self.lin(o, p + "o") + self.w(p + "o.b")

    def mamba2(self, a, p, m):
        n, P, N, G, parts = m["heads"], m["vdim"], m["state"], m["groups"], m["norm_groups"]
        inner = n * P
        z, x, dt = torch.split(self.lin(a, p + "in"), [inner, inner + 2 * G * N, n], dim=1)
        x = torch.nn.functional.silu(self.conv(x, self.w(p + "conv")) + self.w(p + "conv.b"))
        x, B, C = x[:, :inner].view(-1, n, P), x[:, inner:inner + G * N].view(-1, G, N), x[:, inner + G * N:].view(-1, G, N)
        B, C = (t.repeat_interleave(n // G, dim=1) for t in (B, C))
        dt = torch.nn.functional.softplus(dt + self.w(p + "dt_bias"))
        decay = torch.exp(-torch.exp(self.w(p + "A_log")) * dt)
        y = self.recur(C, dt[:, :, None] * B, x, lambda t, S: decay[t][:, None, None] * S, x.new_zeros((n, N, P)))
        y = (y + self.w(p + "D")[:, None] * x).reshape(-1, inner) * torch.nn.functional.silu(z)
        y = self.unit(y.view(-1, parts, inner // parts)).reshape(-1, inner) * self.w(p + "norm")
        return self.lin(y, p + "o")

    def gla(self, a, p, m):
        H, d, dv = m["heads"], m["dim"], m["vdim"]
        q, k, v = (self.lin(a, p + n).view(-1, H, e) for n, e in (("q", d), ("k", d), ("v", dv)))
        log = torch.nn.functional.logsigmoid(self.lin(self.lin(a, p + "a1"), p + "a2") + self.w(p + "a2.b")) / m["tau"]
        alpha = torch.exp(log).view(-1, H, d)
        o = self.recur(q * d ** -0.5, k, v, lambda t, S: alpha[t][:, :, None] * S, q.new_zeros((H, d, dv)))
        o = (self.unit(o) * self.w(p + "norm")).reshape(-1, H * dv)
        return self.lin(o * torch.nn.functional.silu(self.lin(a, p + "g")), p + "o")

    def sigmoid_attention(self, a, p, m):
        H, G, d, dv = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        q, k, v = (self.lin(a, p + n) + self.w(p + n + ".b") for n in ("q", "k", "v"))
        every, coef = m["q_temp"]["every"], m["q_temp"]["coef"]
        temp = 1.0 + coef * torch.log(((self.pos + 1) // every).to(F64) + 1.0)
        q = (self.unit(q) * self.w(p + "q.norm") * temp[:, None]).view(-1, H, d)
        k = (self.unit(k) * self.w(p + "k.norm")).view(-1, G, d)
        r1, r2, pb = (self.w(p + n) for n in ("r1", "r2", "pb"))

        def weigh(h, s, i, j, ok):
            s = s - r1[h] * torch.log1p(r2[h] * (i - j).clamp(min=0)) + pb[h]
            return torch.where(ok, torch.sigmoid(s), torch.zeros((), dtype=F64, device="cuda"))
        o = self.attend(q, k, v.view(-1, G, dv), m["scale"], weigh=weigh).view(-1, H, dv)
        return self.lin((o * torch.sigmoid(self.lin(a, p + "g"))[:, :, None]).reshape(-1, H * dv), p + "o")

    def pooled_attention(self, a, p, m):
        H, G, d = m["heads"], m["kv_heads"], m["dim"]
        q, k, v = ((self.lin(a, p + n) + self.w(p + n + ".b")).view(-1, h, d) for n, h in (("q", H), ("k", G), ("v", G)))
        f = self.frequencies(m["rot"])
        q, k = self.unit(self.rotate(q, f, False)), self.unit(self.rotate(k, f, False))
        size, pool = m["mask"]["size"], m["mask"]["pool"]

        def one(q, k, v):
            T, B = q.shape[0], q.shape[0] // pool
            kp, vp = (x[:B * pool].view(B, pool, G, d).mean(dim=1) for x in (k, v))
            kk, vv = torch.cat([k, kp]), torch.cat([v, vp])
            out = torch.empty((T, H, d), dtype=F64, device="cuda")
            j, b = torch.arange(T, device="cuda")[None, :], torch.arange(B, device="cuda")[None, :]
            for at in range(0, T, 2048):
                i = torch.arange(at, min(at + 2048, T), device="cuda")[:, None]
                ok = torch.cat([(j <= i) & (i - j < size), b * pool + pool - 1 <= i - size], dim=1)
                for h in range(H):
                    s = q[at:at + 2048, h] @ kk[:, h // (H // G)].T * m["scale"]
                    out[at:at + 2048, h] = torch.softmax(s.masked_fill(~ok, -math.inf), dim=1) @ vv[:, h // (H // G)]
            return out.reshape(T, -1)
        return self.lin(self.each(one, q, k, v), p + "o")

    def hgrn2(self, a, p, m):
        H, d, dv = m["heads"], m["dim"], m["vdim"]
        low = self.w(p + "lower")
        f = (low + (1.0 - low) * torch.sigmoid(self.lin(a, p + "f") + self.w(p + "f.b"))).view(-1, H, d)
        q = torch.nn.functional.silu(self.lin(a, p + "q")).view(-1, H, d)
        o = self.recur(q, 1.0 - f, self.lin(a, p + "v").view(-1, H, dv), lambda t, S: f[t][:, :, None] * S,
                       q.new_zeros((H, d, dv)))
        return self.lin((self.unit(o) * self.w(p + "norm")).reshape(-1, H * dv), p + "o")

    def mixed_attention(self, a, p, m):
        H, G, d, dv = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        q, k, v = self.lin(a, p + "q").view(-1, H, d), self.lin(a, p + "k").view(-1, G, d), self.lin(a, p + "v")
        f = self.frequencies(m["rot"])
        if "first" in self.shared:
            lam = self.w(p + "vmix")
            v = (1.0 - lam) * v + lam * self.shared["first"]
        else:
            self.shared["first"] = v
        o = self.attend(self.rotate(q, f, True), self.rotate(k, f, True), v.view(-1, G, dv), m["scale"],
                        sink=torch.zeros(H, dtype=F64, device="cuda"))
        return self.lin(o, p + "o")

    def window_and_delta(self, a, p, m):
        lt, l = m["left"], p + "left."
        H, G, d = lt["heads"], lt["kv_heads"], lt["dim"]
        q, k = self.lin(a, l + "q").view(-1, H, d), self.lin(a, l + "k").view(-1, G, d)
        size, first = lt["mask"]["size"], lt["mask"]["keep_first"]
        o = self.attend(self.unit(q) * self.w(l + "q.norm"), self.unit(k) * self.w(l + "k.norm"), k * m["left_scale"],
                        lt["scale"], lambda i, j: (i - j < size) | (j < first), self.w(l + "sink"), lt["softcap"])
        left = self.lin(o, l + "o")
        H, d, r = m["right"]["heads"], m["right"]["dim"], p + "right."
        q, k, v, g, za = (self.lin(a, r + n) for n in ("r", "k", "v", "g", "a"))
        mid = torch.tanh(self.lin(a, r + "w1"))
        decay = torch.exp(-math.exp(-0.5) * torch.sigmoid(self.lin(mid, r + "w2") + self.w(r + "w0"))).view(-1, H, d)
        rate = torch.sigmoid(za + self.w(r + "a.b")).view(-1, H, d)
        q, k, v = (x.view(-1, H, d) for x in (q, k, v))
        u = k / torch.sqrt((k * k).sum(dim=-1, keepdim=True) + 1e-6)

        def step(t, S):
            return decay[t][:, :, None] * S - (rate[t] * u[t])[:, :, None] * (S * u[t][:, :, None]).sum(dim=1)[:, None, :]
        o = self.unit(self.recur(q, k, v, step, q.new_zeros((H, d, d)))).reshape(-1, H * d)
        return left + self.lin(o * self.w(r + "norm") * torch.sigmoid(g) * m["right_scale"], r + "o")

    def biased_and_retention(self, a, p, m):
        lt, l = m["left"], p + "left."
        H, G, d, nb, far = lt["heads"], lt["kv_heads"], lt["dim"], lt["buckets"], int(lt["bias_max"])
        q = (self.unit(self.lin(a, l + "q")) * self.w(l + "q.norm")).view(-1, H, d)
        k = (self.unit(self.lin(a, l + "k")) * self.w(l + "k.norm")).view(-1, G, d)
        rel, half = self.w(l + "rel"), nb // 2
        rows = list(range(half))        # distance -> row: one each, then row half + k from (n/half)^(nb-half) >= (far/half)^k on
        for n in range(half, max(b - a for a, b in self.spans)):
            e, row = nb - half, rows[-1]
            while row < nb - 1 and n ** e * half ** (row + 1 - half) >= far ** (row + 1 - half) * half ** e:
                row += 1
            rows.append(max(row, half))
        rows = torch.tensor(rows, device="cuda")

        def weigh(h, s, i, j, ok):
            s = s + rel[:, h][rows[(i - j).clamp(min=0)]]
            return torch.softmax(s.masked_fill(~ok, -math.inf), dim=1)
        o = self.attend(q, k, self.lin(a, l + "v").view(-1, G, d), lt["scale"], weigh=weigh)
        left = self.lin(o * torch.sigmoid(self.lin(a, l + "g")) * m["left_scale"], l + "o")
        rt, r = m["right"], p + "right."
        H, d = rt["heads"], rt["dim"]
        f = self.frequencies(rt["rot"])
        q, k, v = (self.lin(a, r + n).view(-1, H, d) for n in ("q", "k", "v"))
        decay = torch.tensor(rt["decay"], dtype=F64, device="cuda")[:, None, None]
        o = self.recur(self.rotate(q, f, False), self.rotate(k, f, False) * d ** -0.5, v, lambda t, S: decay * S,
                       q.new_zeros((H, d, d)))
        o = self.unit(o).reshape(-1, H * d) * torch.nn.functional.silu(self.lin(a, r + "g")) * m["right_scale"]
        return left + self.lin(o, r + "o")

    def mamba1(self, a, p, m):
        I, R, n = m["inner"], m["dt_rank"], m["state"]
        x, z = torch.split(self.lin(a, p + "in"), I, dim=1)
        x = torch.nn.functional.silu(self.conv(x, self.w(p + "conv")) + self.w(p + "conv.b"))
        low = self.lin(x, p + "x")
        dt = torch.nn.functional.softplus(self.lin(low[:, :R], p + "dt") + self.w(p + "dt.b"))
        A, B, C = -torch.exp(self.w(p + "A_log")), low[:, R:R + n], low[:, R + n:]
        y = torch.empty_like(x)
        for s, e in self.spans:
            S = x.new_zeros((I, n))
            for t in range(s, e):
                S = torch.exp(dt[t][:, None] * A) * S + (dt[t] * x[t])[:, None] * B[t][None, :]
                y[t] = S @ C[t]
        y = y + self.w(p + "D") * x
        return self.lin(y * torch.nn.functional.silu(z), p + "o")

    # ---- feed-forwards
    def gated(self, f, p):
        return self.lin(torch.nn.functional.silu(self.lin(f, p + "gate")) * self.lin(f, p + "up"), p + "down")

    def feed_forward(self, f, p, m):
        arch = self.cfg["architecture"]
        if m["kind"] == "dense":
            if arch in ("Rogizen", "Sikazen"):
                return self.gated(f, p)
            act = torch.nn.functional.gelu(self.lin(f, p + "up"), approximate="none" if arch == "Malinex" else "tanh")
            return self.lin(act, p + "down")
        r = m["router"]
        E, top = r["experts"], r["top"]
        z = self.lin(f, p + "router")
        if arch == "Nesilorn":
            val, ids = torch.topk(z + self.w(p + "router.b"), top, dim=1)
            wts = torch.softmax(val, dim=1)
        elif arch == "Mirovik":
            wts, ids = torch.topk(torch.sigmoid(z), top, dim=1)
        else:
            s = torch.softmax(z, dim=1)
            choice = s + self.w(p + "correction")
            if arch == "Pamazen":
                groups = choice.view(f.shape[0], r["groups"]["count"], -1)
                best = groups.max(dim=2).values.topk(r["groups"]["keep"], dim=1).indices
                kept = torch.zeros(groups.shape[:2], dtype=torch.bool, device="cuda").scatter_(1, best, True)
                choice = groups.masked_fill(~kept[:, :, None], -math.inf).view_as(choice)
            ids = torch.topk(choice, top, dim=1).indices
            wts = s.gather(1, ids)
            if arch == "Malinex":
                wts = wts / (wts.sum(dim=1, keepdim=True) + 1e-20)
        out = torch.zeros_like(f)
        for e in range(E + r.get("identity", 0)):
            rows, slot = (ids == e).nonzero(as_tuple=True)
            if rows.numel() == 0:
                continue
            x, wt, q = f[rows], wts[rows, slot][:, None], p + f"e{e}."
            if e >= E:
                y = x * wt
            elif arch == "Nesilorn":
                g = self.lin(x, q + "gate").clamp(max=m["expert"]["limit"])
                u = self.lin(x, q + "up").clamp(-m["expert"]["limit"], m["expert"]["limit"])
                y = self.lin(g * torch.sigmoid(1.702 * g) * (u + 1.0), q + "down") * wt
            elif arch == "Malinex":
                y = self.lin(self.lin(x, q + "up").clamp(min=0.0) ** 2, q + "down") * wt
            elif arch == "Mirovik":
                y = self.gated(x * wt, q)
            else:
                y = self.gated(x, q) * wt
            out.index_add_(0, rows, y)
        if arch == "Malinex":
            out += self.lin(self.lin(f, p + "shared.up").clamp(min=0.0) ** 2, p + "shared.down")
        elif arch == "Mirovik":
            out += self.gated(f, p + "shared.")
        elif arch == "Pamazen":
            out += torch.sigmoid(self.lin(f, p + "shared.sg")) * self.gated(f, p + "shared.")
        return out

    # ---- the model
    def logits(self, ids: torch.Tensor, rows: torch.Tensor) -> torch.Tensor:
        cfg = self.cfg
        arch = cfg.get("architecture", "Llama")
        if arch == "Llama":
            x = self.w("model.embed_tokens.weight")[ids]
            for i in range(cfg["num_hidden_layers"]):
                p = f"model.layers.{i}."
                x = x + self.llama_attention(self.unit(x) * self.w(p + "input_layernorm.weight"), p)
                f = self.unit(x) * self.w(p + "post_attention_layernorm.weight")
                act = torch.nn.functional.silu(self.lin(f, p + "mlp.gate_proj.weight")) * self.lin(f, p + "mlp.up_proj.weight")
                x = x + self.lin(act, p + "mlp.down_proj.weight")
            x = self.unit(x[rows]) * self.w("model.norm.weight")
            return self.lin(x, "model.embed_tokens.weight" if cfg["tie_word_embeddings"] else "lm_head.weight")
        mix = {"latent_attention": self.latent, "mamba2": self.mamba2, "mamba1": self.mamba1, "gla": self.gla,
               "hgrn2": self.hgrn2,
               "parallel": self.window_and_delta if arch == "Pamazen" else self.biased_and_retention,
               "attention": {"Rogizen": self.conv_attention, "Malinex": self.sigmoid_attention,
                             "Sikazen": self.pooled_attention, "Pamazen": self.mixed_attention}.get(arch)}
        x = self.w("embed")[ids] * (cfg.get("embedding") or {}).get("scale", 1.0)
        if arch == "Malinex":
            x = x + self.w("pos")[self.pos]
        if arch == "Rogizen":
            x = self.lin(torch.cat([x, x], dim=1), "loop.in")
        if arch == "Mirovik":
            x = x + self.w("loop.step")[0]
        if arch == "Pamazen":
            x = x[None].repeat(cfg["streams"], 1, 1)
        for i, layer in enumerate(cfg["layers"]):
            p, kind, m = f"l{i}.", layer["type"], layer["mixer"]
            subs = ((lambda a: mix[kind](a, p + "mix.", m)), (lambda f: self.feed_forward(f, p + "mlp.", layer["mlp"])))
            norms = [self.w(p + "norm1"), self.w(p + "norm2")]
            if arch == "Sikazen":
                u = self.unit(x)
                x = x + subs[0](u * norms[0]) + subs[1](u * norms[1])
                n = cfg["token_side"]["dim"]
                t = self.w("side.embed")[ids][:, i * n:(i + 1) * n]
                y = self.lin(torch.nn.functional.gelu(self.lin(x, p + "side.gate"), approximate="tanh") * t, p + "side.proj")
                x = x + self.unit(y) * self.w(p + "side.norm")
                continue
            for n, sub in enumerate(subs, 1):
                if arch == "Nesilorn":
                    x = x + self.unit(sub(x)) * (1.0 + norms[n - 1])
                elif arch == "Rogizen":
                    x = x + sub(self.unit(x) * norms[n - 1])
                elif arch == "Malinex":
                    a = self.unit(x) * norms[n - 1]
                    y = sub(a) * torch.sigmoid(self.lin(a, p + f"rg{n}") + self.w(p + f"rg{n}.b"))
                    x = x + self.unit(y) * self.w(p + f"norm{n}b")
                elif arch == "Pamazen":
                    h = p + f"hc{n}."
                    y = sub(self.unit(torch.einsum("s,stw->tw", self.w(h + "in"), x)) * norms[n - 1])
                    x = torch.einsum("st,snw->tnw", self.w(h + "mix"), x) + \
                        cfg["residual_mult"] * self.w(h + "out")[:, None, None] * y[None]
                else:
                    y = sub(self.unit(x) * (1.0 + norms[n - 1]))
                    x = x + self.unit(y) * (1.0 + self.w(p + f"norm{n}b"))
        if arch == "Pamazen":
            x = x.sum(dim=0)
        w = self.w("final.norm")
        x = self.unit(x[rows]) * (1.0 + w if arch in ("Nesilorn", "Mirovik") else w)
        z = self.lin(x, "embed" if arch in ("Nesilorn", "Mirovik") else "head") * cfg.get("logit_scale", 1.0)
        cap = cfg.get("logit_softcap")
        return cap * torch.tanh(z / cap) if cap else z


def exact(case: dict, seed: int) -> List[torch.Tensor]:
    """The logits of every step from whole sequences in 64 bits."""
    cfg, lens, new = configuration(case), prompt_lengths(case), case["new"]
    prompts, more = tokens(case, seed)
    model = _Exact(cfg, seed, [n + new for n in lens])
    ids = torch.tensor([t for p, m in zip(prompts, more) for t in p + m], device="cuda")
    first = [a for a, _ in model.spans]
    rows = [[first[i] + lens[i] - 1 for i in group] for group in prompt_steps(case)]
    rows += [[first[i] + lens[i] + t for i in range(len(lens))] for t in range(new)]
    with torch.no_grad():
        z = model.logits(ids, torch.tensor([r for step in rows for r in step], device="cuda"))
    return list(torch.split(z, [len(step) for step in rows]))
