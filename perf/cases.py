"""The work that programs have this package do, as measurable cases.

Seven kinds of case cover the package's public entry points:

``linear``            ``W4A8Linear``: quant + GEMM (+ bias or SwiGLU) of one projection, called eagerly
``layer_linears``     the four projections of one decoder layer at decode row counts, in a HIP graph
``midgroup``          ``MidGroupW4A8Linear``: the mid-group pair on an asymmetric group-1024 weight
``attention_prefill`` ``torch.ops.npu.w4a8_attention`` over a prompt
``attention_decode``  ``torch.ops.npu.w4a8_attention_rope``: one decode step of one layer
``decoder_prefill``   ``W4A8Decoder.prefill`` of a few layers
``decoder_decode``    ``W4A8Decoder.decode``: one greedy step, replayed from the captured graph

Shapes are the QwQ-32B projections (hidden 5120, 40 heads over 8 KV heads of 128, ffn 27648) and
their tensor-parallel quarter (10 heads over 2 KV heads, ffn 6912).
"""
from __future__ import annotations

import math

import torch

import __graft_entry__

w4a8 = __graft_entry__.package()

DEV = "cuda"
HIDDEN, HEADS, KV_HEADS, HEAD_DIM, FFN = 5120, 40, 8, 128, 27648


def _projections(tp):
    """K, N of one GPU's slice of a layer's projections."""
    qkv = (HEADS + 2 * KV_HEADS) * HEAD_DIM
    return {"qkv": (HIDDEN, qkv // tp), "o": (HEADS * HEAD_DIM // tp, HIDDEN),
            "gate_up": (HIDDEN, 2 * FFN // tp), "down": (FFN // tp, HIDDEN)}


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# ------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # one token through one small projection, called from Python: launches and latency
        {"name": "linear_token", "kind": "linear", "M": 1, "K": 5120, "N": 5120, "group": 128, "scales": "bf16",
         "bias": False, "act": ""},
        # a serving step's projections with 16 and 64 sequences in flight (weights stream from memory)
        {"name": "layer_linears_16", "kind": "layer_linears", "M": 16, "tp": 1, "group": 128, "scales": "bf16"},
        {"name": "layer_linears_64", "kind": "layer_linears", "M": 64, "tp": 1, "group": 128, "scales": "bf16"},
        # a short prompt (ragged row count) through the biased qkv projection
        {"name": "linear_qkv_1000", "kind": "linear", "M": 1000, "K": 5120, "N": 7168, "group": 128,
         "scales": "bf16", "bias": True, "act": ""},
        # a prefill batch of 4096 tokens through the merged gate/up projection with its SwiGLU
        {"name": "linear_gate_up_4096", "kind": "linear", "M": 4096, "K": 5120, "N": 55296, "group": 128,
         "scales": "bf16", "bias": False, "act": "swiglu"},
        # the largest prefill batch through the long-K projection, fp16 scales
        {"name": "linear_down_16384", "kind": "linear", "M": 16384, "K": 27648, "N": 5120, "group": 128,
         "scales": "fp16", "bias": False, "act": ""},
        # an exported mid-group checkpoint: 16 decode rows on long K, and a prompt on wide N
        {"name": "midgroup_16", "kind": "midgroup", "M": 16, "K": 27648, "N": 5120, "group": 1024, "bias": False},
        {"name": "midgroup_2048", "kind": "midgroup", "M": 2048, "K": 5120, "N": 55296, "group": 1024, "bias": False},
        # a long prompt's attention in one layer
        {"name": "attention_prefill_4096", "kind": "attention_prefill", "B": 1, "T": 4096, "H": 40, "KVH": 8,
         "D": 128},
        # one layer's attention in a step of 64 sequences a little past 1024 tokens
        {"name": "attention_decode_64", "kind": "attention_decode", "B": 64, "L": 1280, "pos": 1100, "H": 40,
         "KVH": 8, "D": 128},
        # a model with one user: the prompt, then a token of the answer (embedding to logits)
        {"name": "decoder_prefill_1024", "kind": "decoder_prefill", "B": 1, "S": 1024, "layers": 2, "vocab": 16384},
        {"name": "decoder_decode_1", "kind": "decoder_decode", "B": 1, "S": 1024, "layers": 4, "vocab": 16384},
    ]


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "layer_linears", "layer_linears", "midgroup", "midgroup",
                       "attention_prefill", "attention_decode", "decoder_prefill", "decoder_decode"])
    tp = rng.choice([1, 1, 4])
    group = rng.choice([128, 128, 128, 64, 256, 512])
    scales = rng.choice(["bf16", "fp16"])
    if kind in ("linear", "midgroup"):
        proj = rng.choice(["qkv", "o", "gate_up", "down"])
        K, N = _projections(tp)[proj]
        # no more work than the largest listed case of the kind
        most = 16384 * 27648 * 5120 if kind == "linear" else 2048 * 5120 * 55296
        M = _log_int(rng, 1, min(16384, most // (K * N)))
        if kind == "midgroup":
            return {"kind": kind, "M": M, "K": K, "N": N, "group": 1024, "bias": proj == "qkv"}
        if rng.random() < 0.1:
            group = K              # one scale per output channel
        return {"kind": kind, "M": M, "K": K, "N": N, "group": group, "scales": scales, "bias": proj == "qkv",
                "act": "swiglu" if proj == "gate_up" else ""}
    if kind == "layer_linears":
        return {"kind": kind, "M": _log_int(rng, 1, 64), "tp": tp, "group": group, "scales": scales}
    heads = rng.choice([(40, 8, 128), (40, 8, 128), (10, 2, 128), (32, 8, 64)])
    if kind == "attention_prefill":
        B = _log_int(rng, 1, 8)
        T = _log_int(rng, 16, int(8192 / math.sqrt(B)))
        return {"kind": kind, "B": B, "T": T, "H": heads[0], "KVH": heads[1], "D": heads[2]}
    if kind == "attention_decode":
        B = _log_int(rng, 1, 64)
        L = _log_int(rng, 64, min(16384, 262144 // B))
        return {"kind": kind, "B": B, "L": L, "pos": rng.randrange(L // 2, L), "H": heads[0], "KVH": heads[1],
                "D": heads[2]}
    if kind == "decoder_prefill":
        B = _log_int(rng, 1, 8)
        return {"kind": kind, "B": B, "S": _log_int(rng, 16, 4096 // B), "layers": 2, "vocab": 16384}
    B = _log_int(rng, 1, 64)
    return {"kind": kind, "B": B, "S": _log_int(rng, 16, min(2048, 16384 // B)), "layers": 2, "vocab": 16384}


# ------------------------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _activations(M, K, gen):
    """bf16 N(0, 1) with 0.1% of the channels scaled by 20 (the outlier channels of a real layer)."""
    x = torch.randn((M, K), device=DEV, generator=gen)
    ch = torch.randperm(K, device=DEV, generator=gen)[:max(1, round(K * 0.001))]
    x[:, ch] *= 20
    return x.to(torch.bfloat16)


def _load_linear(K, N, group, scales, bias, act, gen):
    """A W4A8Linear holding a random checkpoint: int4 codes over their whole range, scales U[0.002, 0.02]."""
    dt = torch.bfloat16 if scales == "bf16" else torch.float16
    m = w4a8.W4A8Linear(K, N, group, bias=bias, scale_dtype=dt, device=DEV, act=act or None)
    kp, last = 2 * m.weight_packed.shape[1], K - (-(-K // group) - 1) * group
    codes = torch.randint(-128, 128, (N, kp // 2), dtype=torch.int8, device=DEV, generator=gen)
    tail = (kp - (-last % 64)) // 2          # a ragged last group's padding slots hold zero codes
    codes[:, tail:] = 0
    m.weight_packed.copy_(codes)
    m.weight_scale.copy_(torch.rand(m.weight_scale.shape, device=DEV, generator=gen) * 0.018 + 0.002)
    if bias:
        m.bias.copy_((torch.rand((N,), device=DEV, generator=gen) - 0.5) * 0.2)
    m.process_weights_after_loading()
    return m


def _decoder(case, seed, max_len):
    cfg = w4a8.decoder.DecoderConfig(layers=case["layers"], vocab=case["vocab"])
    dec = w4a8.decoder.W4A8Decoder(cfg, case["B"], max_len, device=DEV, seed=seed)
    prompt = torch.randint(0, cfg.vocab, (case["B"], case["S"]), device=DEV, generator=_gen(seed + 1))
    return dec, prompt


def prepare(case, seed):
    kind, gen = case["kind"], _gen(seed)
    if kind == "linear":
        m = _load_linear(case["K"], case["N"], case["group"], case["scales"], case["bias"], case["act"], gen)
        return {"kind": kind, "m": m, "x": _activations(case["M"], case["K"], gen)}
    if kind == "midgroup":
        K, N = case["K"], case["N"]
        lin = torch.nn.Linear(K, N, bias=case["bias"], device="meta").to_empty(device=DEV)
        with torch.no_grad():
            lin.weight.normal_(0, 0.02, generator=gen)
            if case["bias"]:
                lin.bias.uniform_(-0.1, 0.1, generator=gen)
        m = w4a8.MidGroupW4A8Linear.from_float(lin, case["group"])
        return {"kind": kind, "m": m, "x": _activations(case["M"], K, gen)}
    if kind == "layer_linears":
        ms = {p: _load_linear(K, N, case["group"], case["scales"], False, "swiglu" if p == "gate_up" else "", gen)
              for p, (K, N) in _projections(case["tp"]).items()}
        xs = {p: _activations(case["M"], ms[p].in_features, gen) for p in ("qkv", "o", "gate_up")}
        st = {"kind": kind, "ms": ms, "xs": xs}

        def step():
            return {"qkv": ms["qkv"](xs["qkv"]), "o": ms["o"](xs["o"]),
                    "down": ms["down"](ms["gate_up"](xs["gate_up"]))}

        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            step()                        # outside the capture first, as serving programs warm their graphs
        torch.cuda.current_stream().wait_stream(side)
        st["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["graph"], stream=side):
            st["out"] = step()
        return st
    if kind in ("attention_prefill", "attention_decode"):
        B, H, KVH, D = case["B"], case["H"], case["KVH"], case["D"]
        L = case["T"] if kind == "attention_prefill" else case["L"]
        Lc = -(-L // 64) * 64
        k = torch.randn((B, KVH, Lc, D), device=DEV, generator=gen).to(torch.bfloat16)
        v = torch.randn((B, KVH, Lc, D), device=DEV, generator=gen).to(torch.bfloat16)
        k[:, :, L:], v[:, :, L:] = 0, 0
        st = {"kind": kind, "k": k, "vt": v.transpose(2, 3).contiguous(), "L": L, "H": H, "KVH": KVH,
              "cps": w4a8.ops.attention_chunks_per_split(B, H, KVH, Lc)}
        if kind == "attention_prefill":
            # queries at twice unit scale: rows that attend to a few keys more than to the rest
            st["q"] = (2 * torch.randn((B, L, H, D), device=DEV, generator=gen)).to(torch.bfloat16)
            st["pos"] = torch.zeros((1,), dtype=torch.long, device=DEV)
            return st
        st["qkv"] = torch.randn((B, (H + 2 * KVH) * D), device=DEV, generator=gen).to(torch.bfloat16)
        st["bias"] = (0.2 * torch.rand(((H + 2 * KVH) * D,), device=DEV, generator=gen) - 0.1).to(torch.bfloat16)
        inv = 1.0e6 ** (-torch.arange(0, D, 2, device=DEV, dtype=torch.float32) / D)
        ang = torch.arange(L, device=DEV, dtype=torch.float32)[:, None] * inv
        st["cos"], st["sin"] = torch.cos(ang), torch.sin(ang)
        st["pos"] = torch.full((1,), case["pos"], dtype=torch.long, device=DEV)
        return st
    if kind == "decoder_prefill":
        dec, prompt = _decoder(case, seed, case["S"])
        return {"kind": kind, "dec": dec, "prompt": prompt}
    dec, prompt = _decoder(case, seed, case["S"] + 8)
    first = dec.prefill(prompt)
    dec.capture()
    return {"kind": kind, "dec": dec, "prompt": prompt, "first": first, "S": case["S"]}


def run(state):
    kind = state["kind"]
    if kind in ("linear", "midgroup"):
        return state["m"](state["x"])
    if kind == "layer_linears":
        state["graph"].replay()
        return state["out"]
    if kind == "attention_prefill":
        return torch.ops.npu.w4a8_attention(state["q"], state["k"], state["vt"], state["pos"], state["L"],
                                            state["cps"], False)
    if kind == "attention_decode":
        return torch.ops.npu.w4a8_attention_rope(state["qkv"], state["cos"], state["sin"], state["pos"], state["k"],
                                                 state["vt"], state["H"], state["KVH"], state["L"], state["cps"],
                                                 state["bias"])
    dec = state["dec"]
    if kind == "decoder_prefill":
        dec.prefill(state["prompt"])
        return dec.last_logits
    dec.decode(state["first"], state["S"], 1)
    return dec.last_logits


# ------------------------------------------------------------------------------------ what a pass needs
def _linear_work(M, K, N, group, outs, extra=4):
    """Packed weight, group scales (and `extra` - 2 bytes more a group), bf16 rows in and out."""
    return {"bytes": N * K / 2 + -(-K // group) * N * extra + 2 * M * K + 2 * M * outs, "flops": 2.0 * M * N * K}


def _sum(works):
    return {k: sum(w[k] for w in works) for k in ("bytes", "flops")}


def work(case):
    kind = case["kind"]
    if kind == "linear":
        return _linear_work(case["M"], case["K"], case["N"], case["group"],
                            case["N"] // 2 if case["act"] else case["N"], 2)
    if kind == "midgroup":       # bf16 scale and zero point
        return _linear_work(case["M"], case["K"], case["N"], case["group"], case["N"], 4)
    if kind == "layer_linears":
        return _sum([_linear_work(case["M"], K, N, case["group"], N // 2 if p == "gate_up" else N, 2)
                     for p, (K, N) in _projections(case["tp"]).items()])
    if kind == "attention_prefill":
        B, T, H, KVH, D = (case[k] for k in ("B", "T", "H", "KVH", "D"))
        return {"bytes": 4.0 * B * T * (H + KVH) * D, "flops": 2.0 * B * H * D * T * (T + 1)}
    if kind == "attention_decode":
        B, n, H, KVH, D = case["B"], case["pos"] + 1, case["H"], case["KVH"], case["D"]
        return {"bytes": 4.0 * B * n * KVH * D + 2.0 * B * (2 * H + 2 * KVH) * D, "flops": 4.0 * B * H * D * n}
    B, S, layers, vocab = case["B"], case["S"], case["layers"], case["vocab"]
    T = S if kind == "decoder_prefill" else 1
    pairs = S * (S + 1) / 2 if T > 1 else S + 1
    per = [_linear_work(B * T, K, N, 128, N // 2 if p == "gate_up" else N, 2)
           for p, (K, N) in _projections(1).items()]
    per.append({"bytes": 4.0 * B * (S + T) * KV_HEADS * HEAD_DIM, "flops": 4.0 * B * HEADS * HEAD_DIM * pairs})
    head = {"bytes": 2.0 * vocab * HIDDEN + 2.0 * B * vocab + 2.0 * B * T * HIDDEN, "flops": 2.0 * B * vocab * HIDDEN}
    return _sum(per * layers + [head])


def tolerance(case):
    kind = case["kind"]
    if kind.startswith("decoder"):
        # int8 codes flip where a bf16 input moves by one rounding, in every layer behind it
        return {"rel": 2e-2, "max": 0.3}
    if kind == "layer_linears":
        # down's int8 codes follow gate_up's bf16 outputs
        return {"rel": 1e-2, "max": 0.2}
    # one bf16 rounding of each output (and the rounded probabilities in attention)
    return {"rel": 8e-3, "max": 0.06}


# ------------------------------------------------------------------------------------ in 64 bits
def _codes(m, K, group):
    """int4 codes [N, K] of a packed weight (even k in the low nibble, groups padded to 64)."""
    p = m.weight_packed
    v = torch.stack([(p << 4) >> 4, p >> 4], -1).reshape(p.shape[0], -1)
    stride = -(-group // 64) * 64
    if stride != group:
        v = torch.cat([v[:, g * stride:g * stride + group] for g in range(-(-K // group))], 1)
    return v[:, :K]


def _spread(t, K, group):
    """[N, G] -> [N, K] fp64."""
    return t.double().repeat_interleave(group, 1)[:, :K]


def _quant(x, step):
    """Per `step` columns: scale bf16(max|x| / 127), codes rounded half to even; fp64."""
    out = torch.empty(x.shape, dtype=torch.float64, device=x.device)
    for i in range(0, x.shape[1], step):
        b = x[:, i:i + step]
        s = (b.abs().amax(1, keepdim=True).float() / 127).to(torch.bfloat16).double()
        s = torch.where(s == 0, torch.full_like(s, torch.finfo(torch.bfloat16).tiny), s)
        out[:, i:i + step] = torch.clamp(torch.round(b.double() / s), -128, 127) * s
    return out


def _exact_linear(m, x, act=""):
    K, N, group = m.in_features, m.out_features, m.group
    a, codes = _quant(x, K), _codes(m, K, group)
    y = torch.cat([a @ (codes[i:i + 8192].double() * _spread(m.weight_scale[i:i + 8192], K, group)).t()
                   for i in range(0, N, 8192)], 1)
    if act:
        return torch.nn.functional.silu(y[:, :N // 2]) * y[:, N // 2:]
    return y + m.bias.double() if m.bias is not None else y


def _rope(t, cos, sin):
    h = t.shape[-1] // 2
    a, b = t[..., :h], t[..., h:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _bf16(t):
    return t.to(torch.bfloat16).double()


def _attend(q, k, v, pos):
    """q [B, T, H, D], k and v [B, KVH, n, D] in fp64; token t attends to 0 .. pos + t."""
    B, T, H, D = q.shape
    KVH, n = k.shape[1], k.shape[2]
    out = torch.empty_like(q)
    rows = max(1, (1 << 27) // n)
    for b in range(B):
        for h in range(H):
            kk, vv = k[b, h * KVH // H], v[b, h * KVH // H]
            for i in range(0, T, rows):
                s = q[b, i:i + rows, h] @ kk.t() / math.sqrt(D)
                last = torch.arange(i, i + s.shape[0], device=q.device) + pos
                s.masked_fill_(torch.arange(n, device=q.device) > last[:, None], float("-inf"))
                out[b, i:i + rows, h] = torch.softmax(s, -1) @ vv
    return out


def _exact_decoder(case, seed):
    """Logits of the last token: the model in fp64, its bf16 tensors rounded where they are defined."""
    dec, tokens = _decoder(case, seed, case["S"] + 8)
    if case["kind"] == "decoder_decode":
        tokens = torch.cat([tokens, dec.prefill(tokens)[:, None]], 1)
    # a second model of the same seed keeps its int4 codes
    m = w4a8.decoder.W4A8Decoder(dec.cfg, 1, 64, device=DEV, seed=seed, keep_weights=True)
    del dec
    c, (B, S) = m.cfg, tokens.shape

    def qlinear(x, lin):
        a = _quant(x, x.shape[1])
        y = torch.cat([a @ (lin.codes[i:i + 8192].double() * _spread(lin.scales.t()[i:i + 8192], lin.K, c.group)).t()
                       for i in range(0, lin.N, 8192)], 1)
        return _bf16(_bf16(y) + lin.bias.double()) if lin.bias is not None else _bf16(y)

    def rms(x, w):
        return _bf16(_bf16(x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + c.rms_eps)) * w.double())

    inv = 1.0 / (c.rope_theta ** (torch.arange(0, c.head_dim, 2, device=DEV, dtype=torch.float32) / c.head_dim))
    ang = torch.arange(S, device=DEV, dtype=torch.float32)[:, None] * inv
    cos, sin = torch.cos(ang).double()[:, None], torch.sin(ang).double()[:, None]
    x = m.embed[tokens.reshape(-1)].double()
    for lw in m.layers:
        qkv = qlinear(rms(x, lw["ln1"]), lw["qkv"]).view(B, S, -1, c.head_dim)
        q, k = _bf16(_rope(qkv[:, :, :c.heads], cos, sin)), qkv[:, :, c.heads:c.heads + c.kv_heads]
        k, v = _bf16(_rope(k, cos, sin)).transpose(1, 2), qkv[:, :, c.heads + c.kv_heads:].transpose(1, 2)
        o = qlinear(_bf16(_attend(q, k, v, 0)).reshape(B * S, -1), lw["o"])
        x = _bf16(x + o)
        gu = qlinear(rms(x, lw["ln2"]), lw["gate_up"])
        g, u = gu[:, :c.ffn], gu[:, c.ffn:]
        x = _bf16(x + qlinear(_bf16(_bf16(torch.nn.functional.silu(g)) * u), lw["down"]))
    last = x.view(B, S, -1)[:, -1]
    return rms(last, m.final_norm) @ m.lm_head.double().t()


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind.startswith("decoder"):
        return _exact_decoder(case, seed) if case["B"] * case["S"] <= 4096 else None
    st = prepare(case, seed)
    if kind == "linear":
        return _exact_linear(st["m"], st["x"], case["act"])
    if kind == "midgroup":
        m, K, group = st["m"], case["K"], case["group"]
        a = _quant(st["x"], group)
        w = (_codes(m, K, group).double() - _spread(m.weight_zero, K, group)) * _spread(m.weight_scale, K, group)
        y = a @ w.t()
        return y + m.bias.double() if m.bias is not None else y
    if kind == "layer_linears":
        ms, xs = st["ms"], st["xs"]
        # gate_up's output is a bf16 tensor: down's quant starts from its rounded values
        gu = _bf16(_exact_linear(ms["gate_up"], xs["gate_up"]))
        g, u = gu.chunk(2, 1)
        h = _bf16(_bf16(torch.nn.functional.silu(g)) * u)
        return {"qkv": _exact_linear(ms["qkv"], xs["qkv"]), "o": _exact_linear(ms["o"], xs["o"]),
                "down": _exact_linear(ms["down"], h)}
    H, KVH, D = case["H"], case["KVH"], case["D"]
    k, v = st["k"].double(), st["vt"].double().transpose(2, 3)
    if kind == "attention_prefill":
        return _attend(st["q"].double(), k, v, 0)
    B, p = case["B"], case["pos"]
    x = (st["qkv"] + st["bias"]).double().view(B, 1, H + 2 * KVH, D)
    cos, sin = st["cos"][p].double(), st["sin"][p].double()
    k[:, :, p] = _bf16(_rope(x[:, 0, H:H + KVH], cos, sin))
    v[:, :, p] = x[:, 0, H + KVH:]
    return _attend(_bf16(_rope(x[:, :, :H], cos, sin)), k[:, :, :p + 1], v[:, :, :p + 1], p)
