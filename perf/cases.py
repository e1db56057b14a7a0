"""Performance cases of the quantized-linear path: the calls a user's program makes, at the sizes it makes them.

Each case goes through the public entry points (``blog_amd.qlin``, ``blog_amd.decoder``).  Decode steps
(one token, a few launches of some microseconds each) are captured into a HIP graph once and replayed,
as a serving loop does; prompt processing, whose sizes change from call to call, runs eagerly.

Weights are packed GGUF blocks whose scales and mins are those of quantized weights of standard
deviation 0.02 (real models' order of magnitude, so Q6_K block scales are f16 subnormals as they are
there); activations are N(0, 1), what follows a norm.

``exact`` evaluates the same inputs in float64 with plain torch, from its own decoders of the formats.
"""
from __future__ import annotations

import math

import torch

from blog_amd import qlin
from blog_amd.decoder import Qwen2Config, Qwen2Decoder

TYPES = {"q4_0": 2, "q5_0": 6, "q8_0": 8, "q4_k": 12, "q6_k": 14}
BLOCK = {"q4_0": (32, 18), "q5_0": (32, 22), "q8_0": (32, 34), "q4_k": (256, 144), "q6_k": (256, 210)}
DEV = "cuda"

# the largest listed product (Q4_K [14336, 4096] over 512 rows) and matrix (Q6_K [102400, 2048])
MAX_MACS = 512 * 14336 * 4096
MAX_WEIGHTS = 102400 * 2048


def listed():
    return [
        # one Qwen2-7B layer's linears for one decode token: q/k/v, o, gate/up SwiGLU, down
        {"name": "decode_layer_q4_k", "kind": "decode_layer", "type": "q4_k", "hidden": 3584, "kv": 512, "ffn": 18944},
        # one greedy decode step of a whole 0.5B model (hidden 896, 24 layers), the smallest launches
        {"name": "decoder_step_q8_0", "kind": "decoder_step", "pos": 159, "max_seq": 512},
        # the same model's prompt in one batched pass
        {"name": "decoder_prefill_q8_0", "kind": "decoder_prefill", "prompt": 384},
        # DeepSeek-V2-Lite's output head for one token
        {"name": "lm_head_q6_k", "kind": "linear", "type": "q6_k", "n": 102400, "k": 2048, "m": 1},
        # a Q4_K_M file's Q6_K ffn_down for a small batch of sequences (or a draft's tokens)
        {"name": "batch_down_q6_k", "kind": "linear", "type": "q6_k", "n": 3584, "k": 18944, "m": 12},
        # a ragged prompt through a Q4_0 gate matrix
        {"name": "prompt_gate_q4_0", "kind": "linear", "type": "q4_0", "n": 18944, "k": 3584, "m": 203},
        # a 512-token prompt through an 8B-class gate matrix, f32 activations
        {"name": "prefill_q4_k", "kind": "linear", "type": "q4_k", "n": 14336, "k": 4096, "m": 512},
        # the same with Q8_1 activations: the quantizer, then the product
        {"name": "prefill_q8_1_q4_k", "kind": "linear_q8_1", "type": "q4_k", "n": 14336, "k": 4096, "m": 512},
        # DeepSeek-V2-Lite's MoE FFN for one token and for a batch of 16
        {"name": "moe_token", "kind": "moe", "tokens": 1, "experts": 64, "k": 6, "ffn": 1408, "hidden": 2048,
         "down": "q5_0", "shared": 2},
        {"name": "moe_batch_16", "kind": "moe", "tokens": 16, "experts": 64, "k": 6, "ffn": 1408, "hidden": 2048,
         "down": "q5_0", "shared": 2},
        # DeepSeek-V2-Lite's MLA decode over the Q8_1 latent cache in mid conversation
        {"name": "mla_decode", "kind": "mla", "type": "q4_k", "heads": 16, "pos": 1500, "max_seq": 2048,
         "fused": False},
        # a weight matrix to f16, for a program that hands prompts to a library GEMM
        {"name": "dequant_q4_k_f16", "kind": "dequant", "type": "q4_k", "n": 14336, "k": 4096, "f16": True},
    ]


def log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode_layer", "decoder_step", "decoder_prefill", "linear", "linear", "linear", "linear_q8_1",
                       "linear_q8_1", "moe", "moe", "mla", "dequant"])
    if kind == "decode_layer":
        hidden = 256 * rng.randint(4, 20)
        return {"kind": kind, "type": rng.choice(["q4_k", "q8_0", "q4_0", "q6_k"]), "hidden": hidden,
                "kv": 64 * rng.randint(2, 16), "ffn": 256 * int(hidden / 256 * rng.uniform(2.0, 5.3))}
    if kind == "decoder_step":
        pos = log_int(rng, 1, 2000)
        return {"kind": kind, "pos": pos, "max_seq": max(512, 256 * ((pos + 256) // 256))}
    if kind == "decoder_prefill":
        return {"kind": kind, "prompt": log_int(rng, 16, 640)}
    if kind in ("linear", "linear_q8_1"):
        t = rng.choice(sorted(TYPES))
        unit = 256 if t.endswith("_k") else 64
        k = unit * (log_int(rng, 512, 16384) // unit)
        n = log_int(rng, 512, 32768)
        m = log_int(rng, 1, 768)
        while n * k < (1 << 21):
            n *= 2
        m = min(m, MAX_MACS // (n * k))
        n = min(n, MAX_WEIGHTS // k)
        return {"kind": kind, "type": t, "n": n, "k": k, "m": max(1, m)}
    if kind == "moe":
        ffn = rng.choice([512, 768, 1024, 1408, 1536])
        down = ["q5_0", "q8_0"] + (["q4_k", "q6_k"] if ffn % 256 == 0 else [])
        return {"kind": kind, "tokens": rng.choice([1, log_int(rng, 2, 40), log_int(rng, 2, 40)]),
                "experts": rng.choice([8, 16, 32, 60, 64, 96]), "k": rng.randint(2, 8), "ffn": ffn,
                "hidden": 256 * rng.randint(4, 10), "down": rng.choice(down), "shared": rng.randint(0, 2)}
    if kind == "mla":
        pos = log_int(rng, 8, 6000)
        return {"kind": kind, "type": rng.choice(["q4_k", "q8_0", "q6_k", "q5_0"]), "heads": rng.choice([16, 16, 32]),
                "pos": pos, "max_seq": max(256, 256 * ((pos + 256) // 256)), "fused": rng.random() < 0.3}
    t = rng.choice(sorted(TYPES))
    be = BLOCK[t][0]
    k = be * (log_int(rng, 512, 16384) // be)
    return {"kind": kind, "type": t, "n": min(log_int(rng, 256, 32768), (1 << 27) // k), "k": k,
            "f16": rng.random() < 0.6}


# ---- inputs ------------------------------------------------------------------------------------

def generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def packed(t, n, k, g):
    """A packed [n, k] matrix of format t (uint8, flat): uniform quants, scales of weights of deviation 0.02."""
    be, bb = BLOCK[t]
    nb = k // be
    w = torch.randint(0, 256, (n, nb, bb), dtype=torch.uint8, device=DEV, generator=g)
    base = {"q4_0": 0.02 / 4.6, "q5_0": 0.02 / 9.2, "q8_0": 0.02 / 73, "q4_k": 0.02 / (4.6 * 42),
            "q6_k": 0.02 / (18.5 * 74)}[t]
    d = ((0.75 + 0.5 * torch.rand((n, nb, 1), device=DEV, generator=g)) * base).to(torch.float16)
    if t == "q6_k":
        w[:, :, 208:210] = d.view(torch.uint8)
    else:
        w[:, :, 0:2] = d.view(torch.uint8)
    if t == "q4_k":
        # the min of a sub-block is about half its range: m near sc, dmin = 7.5 d
        w[:, :, 2:4] = (d.float() * 7.5).to(torch.float16).view(torch.uint8)
        sc = torch.randint(22, 62, (n, nb, 8), dtype=torch.uint8, device=DEV, generator=g)
        mn = sc + torch.randint(0, 2, (n, nb, 8), dtype=torch.uint8, device=DEV, generator=g)
        w[:, :, 4:8] = sc[:, :, :4] | ((sc[:, :, 4:] >> 4) << 6)
        w[:, :, 8:12] = mn[:, :, :4] | ((mn[:, :, 4:] >> 4) << 6)
        w[:, :, 12:16] = (sc[:, :, 4:] & 15) | ((mn[:, :, 4:] & 15) << 4)
    return w.view(-1)


def normal(g, *shape):
    return torch.randn(shape, device=DEV, generator=g)


def moe_inputs(c, seed):
    g = generator(seed)
    e, f, h, s = c["experts"], c["ffn"], c["hidden"], c["ffn"] * c["shared"]
    st = {"wg": packed("q4_k", e * f, h, g), "wu": packed("q4_k", e * f, h, g), "wd": packed(c["down"], e * h, f, g)}
    if s:
        t = shared_type(c)
        st.update(sg=packed(t, s, h, g), su=packed(t, s, h, g), sd=packed(t, h, s, g))
    st.update(x=normal(g, c["tokens"], h), logits=normal(g, c["tokens"], e))
    return st


def shared_type(c):
    """The shared experts' one format: Q4_K where their down projection's rows are whole super-blocks."""
    return "q4_k" if c["ffn"] * c["shared"] % 256 == 0 else "q8_0"


def mla_inputs(c, seed):
    g = generator(seed)
    h, qn, qr, vh, kl = c["heads"], 128, 64, 128, 512
    return {"w": packed(c["type"], h * (qn + vh), kl, g), "q": normal(g, h, qn + qr),
            "kv": normal(g, c["max_seq"], kl + qr)}


def decoder_config():
    return Qwen2Config()


def decoder_weights(seed):
    cfg, g = decoder_config(), generator(seed)
    h, f = cfg.hidden, cfg.ffn

    def norm():
        return (1.0 + 0.1 * normal(g, h)).to(torch.bfloat16).view(torch.int16)

    def layer():
        return {"wq": packed("q8_0", cfg.q_dim, h, g), "wk": packed("q8_0", cfg.kv_dim, h, g),
                "wv": packed("q8_0", cfg.kv_dim, h, g), "wo": packed("q8_0", h, cfg.q_dim, g),
                "wg": packed("q8_0", f, h, g), "wu": packed("q8_0", f, h, g), "wd": packed("q8_0", h, f, g),
                "attn_norm": norm(), "ffn_norm": norm()}

    return {"layers": [layer() for _ in range(cfg.layers)], "final_norm": norm(),
            "table": packed("q8_0", cfg.vocab, h, g)}


def decoder_inputs(c, seed):
    """Weights, the token ids and (a decode step) the cache rows of the positions before it."""
    cfg, g = decoder_config(), generator(seed + 1000003)
    n = c["prompt"] if c["kind"] == "decoder_prefill" else 1
    ids = torch.randint(0, cfg.vocab, (n,), dtype=torch.int32, device=DEV, generator=g)
    cache = None
    if c["kind"] == "decoder_step":
        cache = [(0.6 * normal(g, c["pos"], cfg.kv_dim), 0.6 * normal(g, c["pos"], cfg.kv_dim))
                 for _ in range(cfg.layers)]
    return decoder_weights(seed), ids, cache


def graph_of(fn):
    """fn captured into a HIP graph, after one eager pass (which loads the kernels)."""
    def bound():
        qlin.set_stream(torch.cuda.current_stream())
        fn()
    bound()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        bound()
    qlin.set_stream(torch.cuda.current_stream())
    return g


def prepare(case, seed):
    c, kind, st = case, case["kind"], {"case": case}
    if kind in ("linear", "linear_q8_1"):
        g = generator(seed)
        st.update(w=packed(c["type"], c["n"], c["k"], g), x=normal(g, c["m"], c["k"]),
                  y=torch.empty(c["m"], c["n"], device=DEV))
        if kind == "linear_q8_1":
            st["xq"] = torch.empty(c["m"], qlin.lib().qlin_q8_1_row_bytes(c["k"]), dtype=torch.uint8, device=DEV)
    elif kind == "decode_layer":
        g = generator(seed)
        h, kv, f, t = c["hidden"], c["kv"], c["ffn"], TYPES[c["type"]]
        w = {name: packed(c["type"], n, k, g) for name, n, k in
             (("q", h, h), ("k", kv, h), ("v", kv, h), ("o", h, h), ("g", f, h), ("u", f, h), ("d", h, f))}
        xs = [normal(g, h) for _ in range(3)]
        y = {name: torch.empty(n, device=DEV) for name, n in
             (("q", h), ("k", kv), ("v", kv), ("o", h), ("act", f), ("d", h))}
        rb, rbf = qlin.row_bytes(t, h), qlin.row_bytes(t, f)

        def layer():
            qlin.quant_gemv_multi(t, [w["q"], w["k"], w["v"]], rb, xs[0], [y["q"], y["k"], y["v"]], [h, kv, kv], h)
            qlin.quant_gemv(t, w["o"], rb, xs[1], y["o"], h, h, 1)
            qlin.quant_swiglu(t, w["g"], w["u"], rb, rb, xs[2], y["act"], f, h)
            qlin.quant_gemv(t, w["d"], rbf, y["act"], y["d"], h, f, 1)

        st.update(w=w, xs=xs, out=y, graph=graph_of(layer))
    elif kind == "moe":
        st.update(moe_inputs(c, seed))
        e, k, f, h, n, s = c["experts"], c["k"], c["ffn"], c["hidden"], c["tokens"], c["ffn"] * c["shared"]
        st.update(ids=torch.empty(n, k, dtype=torch.int32, device=DEV), rw=torch.empty(n, k, device=DEV),
                  out=torch.empty(n, h, device=DEV))
        t4, td, ts = TYPES["q4_k"], TYPES[c["down"]], TYPES[shared_type(c)]
        shared = (ts, st["sg"], st["su"], qlin.row_bytes(ts, h), st["sd"], qlin.row_bytes(ts, s), s) if s else \
            (t4, 0, 0, 0, 0, 0, 0)
        routed = (t4, st["wg"], st["wu"], st["wg"].numel(), td, st["wd"], st["wd"].numel(), e, f, h, h)
        if n == 1:
            st["act"] = torch.empty(k * f + s, device=DEV)

            def ffn():
                st["out"].zero_()
                qlin.call("qlin_moe_ffn_decode_indexed_logits", *routed, *shared, st["x"], st["logits"], 1.0,
                          st["ids"], st["rw"], st["act"], st["out"], k)
        else:
            nws = qlin.lib().qlin_moe_ffn_workspace_bytes(n, k, e, f, h, s)
            st["ws"] = torch.empty(nws, dtype=torch.uint8, device=DEV)

            def ffn():
                st["out"].zero_()
                qlin.call("qlin_moe_ffn_decode_grouped_logits", *routed, *shared, st["x"], st["logits"], 1.0,
                          st["ids"], st["rw"], st["ws"], nws, st["out"], n, k)
        st["graph"] = graph_of(ffn)
    elif kind == "mla":
        st.update(mla_inputs(c, seed))
        t, h, qn, qr, vh, kl, T = TYPES[c["type"]], c["heads"], 128, 64, 128, 512, c["max_seq"]
        rb, crb = qlin.row_bytes(t, kl), qlin.lib().qlin_q8_1_row_bytes(kl)
        cache = quantize_q8_1(st["kv"][:, :kl])[0]
        cache[c["pos"]:] = 0  # this position's row is the step's to write
        st.update(cache=cache, pos=torch.tensor([c["pos"]], dtype=torch.int32, device=DEV),
                  q_abs=torch.empty(h, kl, device=DEV), delta=torch.zeros(h, kl // 32, device=DEV),
                  delta2=torch.empty(h, kl // 32, device=DEV), scores=torch.zeros(h, T, device=DEV),
                  latent=torch.empty(h, kl, device=DEV), attn=torch.empty(h, vh, device=DEV))
        scale = 1.0 / math.sqrt(qn + qr)

        def step():
            s = st
            qlin.call("qlin_launch_mla_absorb_q_nope", t, s["q"], s["w"], rb, s["q_abs"], h, qn, qr, vh, kl)
            if c["type"] == "q4_k":
                qlin.call("qlin_launch_mla_absorb_q4_xsum_delta", s["q"], s["w"], rb, s["delta"], h, qn, qr, vh, kl)
            qlin.call("qlin_launch_mla_store_latent_q8_1_device_pos", s["kv"], s["cache"], kl, qr, crb, s["pos"])
            if c["fused"]:
                qlin.call("qlin_launch_mla_absorb_attend_device_pos", s["q_abs"], s["q"], s["cache"], crb, s["delta"],
                          s["delta2"], s["kv"], s["latent"], h, qn, qr, kl, s["pos"], T, scale)
            else:
                qlin.call("qlin_launch_mla_absorb_scores_device_pos", s["q_abs"], s["q"], s["cache"], crb, s["delta"],
                          s["kv"], s["scores"], h, qn, qr, kl, s["pos"], T, scale)
                qlin.call("qlin_launch_mla_absorb_context_device_pos", s["scores"], s["cache"], crb, s["delta2"],
                          s["latent"], h, kl, s["pos"], T)
            qlin.call("qlin_launch_mla_absorb_v", t, s["w"], rb, s["latent"], s["delta2"], s["attn"], h, qn, vh, kl)

        st["graph"] = graph_of(step)
    elif kind == "dequant":
        st.update(w=packed(c["type"], c["n"], c["k"], generator(seed)),
                  out=torch.empty(c["n"], c["k"], dtype=torch.float16 if c["f16"] else torch.float32, device=DEV))
    else:
        cfg = decoder_config()
        weights, ids, cache = decoder_inputs(c, seed)
        if kind == "decoder_prefill":
            dec = Qwen2Decoder(torch, cfg, weights, max_seq=c["prompt"] + 128, max_prompt=c["prompt"])
            st.update(dec=dec, ids=ids)
        else:
            dec = Qwen2Decoder(torch, cfg, weights, max_seq=c["max_seq"], max_prompt=32)
            for i, (k, v) in enumerate(cache):
                dec.kc[i][:c["pos"]] = k
                dec.vc[i][:c["pos"]] = v

            def step():
                torch.add(ids, 0, out=dec.token)
                dec.pos.fill_(c["pos"])
                dec.step()

            st.update(dec=dec, ids=ids, graph=graph_of(step))
    qlin.set_stream(torch.cuda.current_stream())
    return st


def run(st):
    c, kind = st["case"], st["case"]["kind"]
    if "graph" in st:
        st["graph"].replay()
    if kind == "linear":
        qlin.call("qlin_gemm", TYPES[c["type"]], st["w"], st["w"].numel(), st["x"], st["y"], c["n"], c["k"], c["m"])
        return st["y"]
    if kind == "linear_q8_1":
        t = TYPES[c["type"]]
        qlin.quantize_q8_1(st["x"], st["xq"], c["k"], c["m"])
        qlin.quant_matmul_q8_1(t, st["w"], st["w"].numel() // c["n"], st["xq"], st["y"], c["n"], c["k"], c["m"])
        return {"xq": st["xq"], "y": st["y"]}
    if kind == "decode_layer":
        return st["out"]
    if kind == "moe":
        return {"out": st["out"], "ids": st["ids"], "weights": st["rw"]}
    if kind == "mla":
        out = {"attn": st["attn"], "latent": st["latent"], "cache": st["cache"]}
        return out if c["fused"] else dict(out, scores=st["scores"])
    if kind == "dequant":
        qlin.dequantize(TYPES[c["type"]], st["w"], st["out"], c["n"] * c["k"], f16=c["f16"])
        return st["out"]
    dec = st["dec"]
    if kind == "decoder_prefill":
        dec.prefill(st["ids"])
    return {"logits": dec.logits, "k": dec.kc, "v": dec.vc}


def work(case):
    c, kind = case, case["kind"]

    def wb(t, n, k):
        return n * (k // BLOCK[t][0]) * BLOCK[t][1]

    if kind == "linear":
        n, k, m = c["n"], c["k"], c["m"]
        return {"bytes": wb(c["type"], n, k) + 4 * m * (k + n), "flops": 2 * m * n * k}
    if kind == "linear_q8_1":
        n, k, m = c["n"], c["k"], c["m"]
        return {"bytes": wb(c["type"], n, k) + 4 * m * (k + n) + m * (k // 32) * 36, "flops": 2 * m * n * k}
    if kind == "decode_layer":
        h, kv, f = c["hidden"], c["kv"], c["ffn"]
        mats = [(h, h), (kv, h), (kv, h), (h, h), (f, h), (f, h), (h, f)]
        return {"bytes": sum(wb(c["type"], n, k) for n, k in mats) + 4 * (3 * h + 3 * h + 2 * kv + 2 * f),
                "flops": sum(2 * n * k for n, k in mats)}
    if kind == "moe":
        e, k, f, h, n, s = c["experts"], c["k"], c["ffn"], c["hidden"], c["tokens"], c["ffn"] * c["shared"]
        k = min(k, e)
        distinct = e * (1 - (1 - k / e) ** n)  # expected over uniform routings
        b = distinct * (2 * wb("q4_k", f, h) + wb(c["down"], h, f)) + 4 * n * (2 * h + e + 2 * k)
        if s:
            b += 2 * wb(shared_type(c), s, h) + wb(shared_type(c), h, s)
        return {"bytes": int(b), "flops": 6 * n * (k * f + s) * h}
    if kind == "mla":
        h, kl, p = c["heads"], 512, c["pos"] + 1
        b = wb(c["type"], h * 256, kl) + p * (576 + 64 * 4) + 4 * h * (192 + 512 + 128) + (0 if c["fused"] else 8 * h * p)
        return {"bytes": b, "flops": 2 * h * (256 * kl + p * (2 * kl + 64))}
    if kind == "dequant":
        return {"bytes": wb(c["type"], c["n"], c["k"]) + (2 if c["f16"] else 4) * c["n"] * c["k"],
                "flops": 2 * c["n"] * c["k"]}
    cfg = decoder_config()
    h, f, q, kv, v, L = cfg.hidden, cfg.ffn, cfg.q_dim, cfg.kv_dim, cfg.vocab, cfg.layers
    per_layer = 2 * h * q + 2 * kv * h + 3 * h * f
    rows = c["prompt"] if kind == "decoder_prefill" else 1
    before = 0 if kind == "decoder_prefill" else c["pos"]
    attn = sum(4 * q * (before + r + 1) for r in range(rows))
    return {"bytes": (L * per_layer + v * h) // 32 * 34 + 8 * L * kv * (before + rows) + 4 * v + rows * 4 * h,
            "flops": 2 * (rows * L * per_layer + v * h) + L * attn}


def tolerance(case):
    return TOLERANCE[case["kind"]]


# About four times the relative errors against float64 seen over the ranges above (linear 3.7e-7 .. 2e-6,
# Q8_1 1.5e-7, a decode layer 3.4e-6, MoE 6.1e-6, MLA 3.7e-7, the whole model 2.5e-6), and no less than
# what 32-bit sums in another order give.
TOLERANCE = {
    "linear": {"rel": 1e-5},
    "linear_q8_1": {"rel": 1e-5},
    "decode_layer": {"rel": 1.5e-5},
    "moe": {"rel": 2.5e-5},
    "mla": {"rel": 1e-5},
    "dequant": "exact",
    "decoder_step": {"rel": 2e-5},
    "decoder_prefill": {"rel": 2e-5},
}


# ---- the same in float64 -----------------------------------------------------------------------

def f16_at(b, i):
    return b[..., i:i + 2].contiguous().view(torch.float16)[..., 0].double()


def q4_k_fields(b):
    """(d, dmin, sc [.., 8], m [.., 8]) of Q4_K super-blocks b [.., 144], float64."""
    lo, mid, hi = b[..., 4:8], b[..., 8:12], b[..., 12:16]
    sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], -1).double()
    mn = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], -1).double()
    return f16_at(b, 0), f16_at(b, 2), sc, mn


def quants(t, b):
    """Integer quants (float64, offsets taken off) and their scales, broadcastable to [.., elements]."""
    if t == "q8_0":
        return b[..., 2:].contiguous().view(torch.int8).double(), f16_at(b, 0)[..., None]
    if t in ("q4_0", "q5_0"):
        qs = b[..., 2:] if t == "q4_0" else b[..., 6:]
        q = torch.cat([qs & 15, qs >> 4], -1).double()
        if t == "q4_0":
            return q - 8, f16_at(b, 0)[..., None]
        bits = torch.arange(8, device=b.device, dtype=torch.uint8)
        q += 16 * ((b[..., 2:6, None] >> bits) & 1).flatten(-2).double()
        return q - 16, f16_at(b, 0)[..., None]
    if t == "q4_k":
        d, _, sc, _ = q4_k_fields(b)
        qs = b[..., 16:].unflatten(-1, (4, 32))
        return torch.stack([qs & 15, qs >> 4], -2).flatten(-3).double(), (d[..., None] * sc).repeat_interleave(32, -1)
    ql, qh = b[..., :128].unflatten(-1, (2, 2, 32)), b[..., 128:192].unflatten(-1, (2, 1, 32))
    lo = torch.cat([ql & 15, ql >> 4], -2)                                   # [.., half, group, 32]
    sh = torch.tensor([0, 2, 4, 6], device=b.device, dtype=torch.uint8)[:, None]
    q = (lo | (((qh >> sh) & 3) << 4)).flatten(-3).double() - 32
    sc = b[..., 192:208].contiguous().view(torch.int8).double()
    return q, (f16_at(b, 208)[..., None] * sc).repeat_interleave(16, -1)


def weights64(t, w, n, k):
    be, bb = BLOCK[t]
    b = w.view(n, k // be, bb)
    q, s = quants(t, b)
    v = q * s
    if t == "q4_k":
        _, dmin, _, mn = q4_k_fields(b)
        v -= (dmin[..., None] * mn).repeat_interleave(32, -1)
    return v.reshape(n, k)


def product64(t, w, n, k, x):
    """x [m, k] times the matrix's transpose, in slices of rows that keep the float64 weights small."""
    rb = w.numel() // n
    step = max(1, (1 << 26) // k)
    return torch.cat([x @ weights64(t, w[i * rb:(i + step) * rb], min(step, n - i), k).T for i in range(0, n, step)], 1)


def quantize_q8_1(x):
    """Q8_1 rows (uint8 [m, k / 32 * 36]) of f32 x, with d, s (float64 values of their f16) and q."""
    xb = x.reshape(x.shape[0], -1, 32)
    amax = xb.abs().amax(-1)
    d = amax / torch.full_like(amax, 127.0)  # (by a Python number it would be a product with the reciprocal)
    inv = torch.where(d > 0, torch.ones_like(d) / d, torch.zeros_like(d))
    q = torch.round(xb * inv[..., None]).clamp(-127, 127)
    dh, sh = d.half(), (d * q.sum(-1)).half()
    rows = torch.cat([dh[..., None].view(torch.uint8), sh[..., None].view(torch.uint8),
                      q.to(torch.int8).view(torch.uint8)], -1)
    return rows.reshape(x.shape[0], -1).contiguous(), dh.double(), sh.double(), q.double()


def linear_q8_1_64(c, w, x):
    t, n, k = c["type"], c["n"], c["k"]
    _, d, s, q = quantize_q8_1(x)
    xd = (d[..., None] * q).flatten(1)
    if t != "q4_k":
        return product64(t, w, n, k, xd)
    rb, step, out = w.numel() // n, max(1, (1 << 26) // k), []
    for i in range(0, n, step):
        rows = min(step, n - i)
        b = w[i * rb:(i + step) * rb].view(rows, k // 256, 144)
        wq, ws = quants(t, b)
        _, dmin, _, mn = q4_k_fields(b)
        out.append(xd @ (wq * ws).reshape(rows, k).T - s @ (dmin[..., None] * mn).reshape(rows, k // 32).T)
    return torch.cat(out, 1)


def silu_mul(g, u):
    return g / (1.0 + torch.exp(-g)) * u


def moe_64(c, st):
    e, f, h, s = c["experts"], c["ffn"], c["hidden"], c["ffn"] * c["shared"]
    x, p = st["x"].double(), torch.softmax(st["logits"].double(), 1)
    w, ids = torch.topk(p, min(c["k"], e), 1)
    out = torch.zeros(c["tokens"], h, dtype=torch.float64, device=DEV)

    def of(name, t, i, n, k):
        size = st[name].numel() // e
        return weights64(t, st[name][i * size:(i + 1) * size], n, k)

    for i in ids.unique().tolist():
        tok, slot = torch.nonzero(ids == i, as_tuple=True)
        act = silu_mul(x[tok] @ of("wg", "q4_k", i, f, h).T, x[tok] @ of("wu", "q4_k", i, f, h).T)
        out.index_add_(0, tok, w[tok, slot][:, None] * (act @ of("wd", c["down"], i, h, f).T))
    if s:
        act = silu_mul(x @ weights64(shared_type(c), st["sg"], s, h).T, x @ weights64(shared_type(c), st["su"], s, h).T)
        out += act @ weights64(shared_type(c), st["sd"], h, s).T
    return {"out": out, "ids": None, "weights": w}


def mla_64(c, st):
    t, h, qn, qr, vh, kl, pos = c["type"], c["heads"], 128, 64, 128, 512, c["pos"]
    w = weights64(t, st["w"], h * (qn + vh), kl).view(h, qn + vh, kl)
    _, d, s, q = quantize_q8_1(st["kv"][:pos + 1, :kl])
    lat = (d[..., None] * q).flatten(1)
    corr = s - (d[..., None] * q).sum(-1)
    q64, kr = st["q"].double(), st["kv"][:pos + 1, kl:].double()
    q_abs = torch.einsum("hd,hdl->hl", q64[:, :qn], w[:, :qn])
    mins = torch.zeros(h, qn + vh, kl // 32, dtype=torch.float64, device=DEV)
    if t == "q4_k":
        _, dmin, _, mn = q4_k_fields(st["w"].view(h, qn + vh, kl // 256, 144))
        mins = -(dmin[..., None] * mn).reshape(h, qn + vh, kl // 32)
    delta = torch.einsum("hd,hdb->hb", q64[:, :qn], mins[:, :qn])
    sc = (q_abs @ lat.T + q64[:, qn:] @ kr.T + delta @ corr.T) / math.sqrt(qn + qr)
    p = torch.softmax(sc, 1)
    latent, dsum = p @ lat, p @ corr
    attn = torch.einsum("hl,hvl->hv", latent, w[:, qn:]) + torch.einsum("hb,hvb->hv", dsum, mins[:, qn:])
    out = {"attn": attn, "latent": latent, "cache": None}
    if c["fused"]:
        return out
    scores = torch.zeros(h, c["max_seq"], dtype=torch.float64, device=DEV)
    scores[:, :pos + 1] = sc
    return dict(out, scores=scores)


def decoder_64(c, seed):
    cfg = decoder_config()
    weights, ids, cache = decoder_inputs(c, seed)
    h, hd, nh, nkv = cfg.hidden, cfg.head_dim, cfg.n_heads, cfg.kv_heads
    n, start = ids.numel(), 0 if cache is None else c["pos"]

    def norm(x, w):
        return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + cfg.eps) * w.view(torch.bfloat16).double()

    pos = torch.arange(start, start + n, device=DEV, dtype=torch.float64)
    freq = cfg.theta ** (-torch.arange(0, hd, 2, device=DEV, dtype=torch.float64) / hd)
    cos, sin = torch.cos(pos[:, None] * freq), torch.sin(pos[:, None] * freq)

    def rope(x):
        a, b = x[..., :hd // 2], x[..., hd // 2:]
        return torch.cat([a * cos[:, None] - b * sin[:, None], b * cos[:, None] + a * sin[:, None]], -1)

    rb = weights["table"].numel() // cfg.vocab
    rows = weights["table"].view(cfg.vocab, rb)[ids.long()].contiguous()
    x = weights64("q8_0", rows, n, h)
    ks, vs = [], []
    for i, w in enumerate(weights["layers"]):
        a = norm(x, w["attn_norm"])
        q = rope((a @ weights64("q8_0", w["wq"], cfg.q_dim, h).T).view(n, nh, hd))
        k = rope((a @ weights64("q8_0", w["wk"], cfg.kv_dim, h).T).view(n, nkv, hd))
        v = (a @ weights64("q8_0", w["wv"], cfg.kv_dim, h).T).view(n, nkv, hd)
        if cache is not None:
            k = torch.cat([cache[i][0].double().view(-1, nkv, hd), k])
            v = torch.cat([cache[i][1].double().view(-1, nkv, hd), v])
        full = torch.zeros(2, c["max_seq"] if cache is not None else n + 128, cfg.kv_dim, dtype=torch.float64,
                           device=DEV)
        full[0, :start + n], full[1, :start + n] = k.flatten(1), v.flatten(1)
        ks.append(full[0])
        vs.append(full[1])
        kg, vg = k.repeat_interleave(nh // nkv, 1).transpose(0, 1), v.repeat_interleave(nh // nkv, 1).transpose(0, 1)
        s = q.transpose(0, 1) @ kg.transpose(1, 2) / math.sqrt(hd)
        mask = torch.arange(start + n, device=DEV)[None] > torch.arange(start, start + n, device=DEV)[:, None]
        o = torch.softmax(s.masked_fill(mask, -math.inf), -1) @ vg
        x = x + o.transpose(0, 1).reshape(n, nh * hd) @ weights64("q8_0", w["wo"], h, cfg.q_dim).T
        a = norm(x, w["ffn_norm"])
        act = silu_mul(a @ weights64("q8_0", w["wg"], cfg.ffn, h).T, a @ weights64("q8_0", w["wu"], cfg.ffn, h).T)
        x = x + act @ weights64("q8_0", w["wd"], h, cfg.ffn).T
    last = norm(x[-1:], weights["final_norm"])
    return {"logits": product64("q8_0", weights["table"], cfg.vocab, h, last)[0], "k": ks, "v": vs}


def exact(case, seed):
    c, kind = case, case["kind"]
    g = generator(seed)
    if kind in ("linear", "linear_q8_1"):
        w, x = packed(c["type"], c["n"], c["k"], g), normal(g, c["m"], c["k"])
        if kind == "linear":
            return product64(c["type"], w, c["n"], c["k"], x.double())
        return {"xq": None, "y": linear_q8_1_64(c, w, x)}
    if kind == "decode_layer":
        h, kv, f, t = c["hidden"], c["kv"], c["ffn"], c["type"]
        w = {name: (packed(t, n, k, g), n, k) for name, n, k in
             (("q", h, h), ("k", kv, h), ("v", kv, h), ("o", h, h), ("g", f, h), ("u", f, h), ("d", h, f))}
        xs = [normal(g, h).double()[None] for _ in range(3)]
        y = {name: product64(t, *w[name], xs[i])[0] for name, i in (("q", 0), ("k", 0), ("v", 0), ("o", 1))}
        act = silu_mul(product64(t, *w["g"], xs[2]), product64(t, *w["u"], xs[2]))
        return dict(y, act=act[0], d=product64(t, *w["d"], act)[0])
    if kind == "moe":
        return moe_64(c, moe_inputs(c, seed))
    if kind == "mla":
        return mla_64(c, mla_inputs(c, seed))
    if kind == "dequant":
        return weights64(c["type"], packed(c["type"], c["n"], c["k"], g), c["n"], c["k"])
    return decoder_64(c, seed)
