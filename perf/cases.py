"""What this framework's speed is measured on: the calls a program makes through its public entry points.

Each case is one kind of call at one size. `listed()` holds the sizes that the configurations, the tests and the
benchmark of this repository use (Llama-3.2-1B widths: hidden 2048, FFN 8192, 32/8 heads of 64, prompts of 512 and
3968 tokens); `draw(rng)` gives other sizes of the same ranges, odd and ragged ones among them.

Kinds:
  gemm            flm.GEMM, a projection of a prompt's tokens by a packed (N, K) weight, with its epilogues
  gemm_rowmajor   GEMM with its default row-major (K, N) second operand
  gemm_int4       GEMMInt4, a projection that reads int4 group-32 weights
  mha             MHA, the causal (grouped-query) attention of a prompt
  swiglu_prefill  SwiGLUPrefill, the feed-forward block of a prompt as an operator sequence
  gqa_decode      GQADecode, the attention of one new token against its KV cache
  gemv_int4       GEMVInt4, a projection of one token by int4 group-32 weights
  prefill         LlamaHIP.prefill of a whole prompt (int4 group-32 weights, 8 layers): logits and the KV rows it wrote
  decode          LlamaHIP.decode of one token (int4 group-32 weights, 8 layers): logits and the KV rows it wrote
"""

from __future__ import annotations

import math

import torch

BF16 = torch.bfloat16
DEV = "cuda"

# The model of the two whole calls: Llama-3.2-1B widths and vocabulary, 8 of its 16 layers. A change of rounding in the
# first layer travels through all that follow: at 16 layers o_proj summed in another order alone moves the logits by
# 0.02 (2-norm) and 64-bit arithmetic by 0.025, too much for a comparison of two correct programs to say anything.
VOCAB, EMB, LAYERS, HEADS, KV_HEADS, FFN, HEAD_DIM = 128256, 2048, 8, 32, 8, 8192, 64
EPS = 1e-5
# The largest product a drawn GEMM may be (that of the gate and up projections of 3968 tokens together).
MOST_MNK = 3968 * 2048 * 16384


def listed():
    return [
        # The gate (or up) projection of a 512-token prompt: the ordinary prefill GEMM.
        {"name": "gemm_gate_512", "kind": "gemm", "M": 512, "K": 2048, "N": 8192, "epilogue": "silu"},
        # The down projection of a long prompt: the largest single GEMM of a prefill.
        {"name": "gemm_down_3968", "kind": "gemm", "M": 3968, "K": 8192, "N": 2048, "epilogue": "none"},
        # The qkv projection of a 13-token chat turn: few rows, so the weights are the traffic.
        {"name": "gemm_qkv_13", "kind": "gemm", "M": 13, "K": 2048, "N": 3072, "epilogue": "none"},
        # GEMM as it is by default, the second operand row-major (K, N), ordinary size.
        {"name": "gemm_rowmajor_2048", "kind": "gemm_rowmajor", "M": 2048, "K": 2048, "N": 2048},
        # The gate projection of a 512-token prompt from the int4 weights that decode keeps.
        {"name": "gemm_int4_512", "kind": "gemm_int4", "M": 512, "K": 2048, "N": 8192},
        # The attention of a long prompt, grouped-query.
        {"name": "mha_3968", "kind": "mha", "S": 3968, "heads": 32, "kv_heads": 8},
        # The attention of a short, ragged prompt.
        {"name": "mha_333", "kind": "mha", "S": 333, "heads": 32, "kv_heads": 8},
        # The feed-forward block of a 256-token prompt as the reference's operator sequence, weights (K, N).
        {"name": "swiglu_prefill_256", "kind": "swiglu_prefill", "S": 256, "E": 2048, "H": 8192, "b_col_maj": False},
        # One token's attention against 2048 cached positions.
        {"name": "gqa_decode_2048", "kind": "gqa_decode", "pos": 2047, "max_len": 2048, "heads": 32, "kv_heads": 8},
        # One token's gate projection: the smallest call, where launch latency counts.
        {"name": "gemv_int4_gate", "kind": "gemv_int4", "M": 8192, "K": 2048},
        # A 512-token prompt through the whole model, replaying the graph captured for its length.
        {"name": "prefill_512", "kind": "prefill", "S": 512, "graph": True},
        # One token through the whole model behind a long context.
        {"name": "decode_3968", "kind": "decode", "pos": 3968},
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "gemm", "gemm_rowmajor", "gemm_int4", "mha", "mha", "swiglu_prefill",
                       "gqa_decode", "gemv_int4", "prefill", "decode"])
    if kind in ("gemm", "gemm_rowmajor", "gemm_int4"):
        while True:
            M, K, N = _log(rng, 1, 3968), 64 * _log(rng, 8, 128), _log(rng, 256, 16384)
            if rng.random() < 0.5:  # the widths of layers are mostly multiples of 64
                N = (N + 63) // 64 * 64
            if M * K * N <= MOST_MNK:
                break
        c = {"kind": kind, "M": M, "K": K, "N": N}
        if kind == "gemm":
            c["epilogue"] = rng.choice(["none", "none", "gelu", "silu", "sigmoid"])
        return c
    if kind == "mha":
        heads, kv = rng.choice([(32, 8), (32, 8), (8, 8), (16, 4), (8, 2)])
        return {"kind": kind, "S": _log(rng, 32, 3968), "heads": heads, "kv_heads": kv}
    if kind == "swiglu_prefill":
        return {"kind": kind, "S": _log(rng, 16, 512), "E": rng.choice([1024, 2048]), "H": rng.choice([2048, 4096, 8192]),
                "b_col_maj": rng.random() < 0.5}
    if kind == "gqa_decode":
        heads, kv = rng.choice([(32, 8), (32, 8), (16, 16), (64, 8), (8, 2)])
        pos = _log(rng, 16, 4095)
        return {"kind": kind, "pos": pos, "max_len": (pos // 512 + 1) * 512, "heads": heads, "kv_heads": kv}
    if kind == "gemv_int4":
        return {"kind": kind, "M": _log(rng, 512, 131072), "K": rng.choice([2048, 2048, 4096, 8192, 32 * _log(rng, 16, 256)])}
    if kind == "prefill":
        return {"kind": kind, "S": _log(rng, 16, 511), "graph": rng.random() < 0.5}
    return {"kind": "decode", "pos": _log(rng, 16, 4480)}


# --------------------------------------------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _normal(g, *shape, std=1.0, mean=0.0):
    return (torch.randn(*shape, generator=g, device=DEV) * std + mean).to(BF16)


def _int4(g, rows, K):
    """Codes (two's complement, low nibble first) and scales of an int4 group-32 weight."""
    codes = torch.randint(0, 256, (rows, K // 2), generator=g, dtype=torch.uint8, device=DEV)
    scales = (0.001 + 0.009 * torch.rand(rows, K // 32, generator=g, device=DEV)).to(BF16)
    return codes, scales


def _layer_names(i):
    p = f"model.layers.{i}."
    return {n: p + n + ".weight" for n in
            ("input_layernorm", "post_attention_layernorm", "self_attn.q_proj", "self_attn.k_proj", "self_attn.v_proj",
             "self_attn.o_proj", "mlp.gate_proj", "mlp.up_proj", "mlp.down_proj")}


def _model_weights(g):
    w = {"model.embed_tokens.weight": _normal(g, VOCAB, EMB, std=0.02), "model.norm.weight": _normal(g, EMB, std=0.1, mean=1.0)}
    rows = {"self_attn.q_proj": (HEADS * HEAD_DIM, EMB), "self_attn.k_proj": (KV_HEADS * HEAD_DIM, EMB),
            "self_attn.v_proj": (KV_HEADS * HEAD_DIM, EMB), "self_attn.o_proj": (EMB, HEADS * HEAD_DIM),
            "mlp.gate_proj": (FFN, EMB), "mlp.up_proj": (FFN, EMB), "mlp.down_proj": (EMB, FFN)}
    for i in range(LAYERS):
        for n, full in _layer_names(i).items():
            w[full] = _normal(g, EMB, std=0.1, mean=1.0) if "layernorm" in n else _normal(g, *rows[n], std=0.02)
    return w


def _kv(g, n):
    """Rows of a model's KV cache (of one layer): rotated keys and values have about this spread at these weights."""
    return _normal(g, KV_HEADS, n, HEAD_DIM, std=0.9), _normal(g, KV_HEADS, n, HEAD_DIM, std=0.9)


def _angles(rows):
    """RoPE angles (rows, 32) of the model (theta 500000, llama3 band scaling with factor 32), in float32 as the model keeps them."""
    inv = 1.0 / (500000.0 ** (torch.arange(0, HEAD_DIM, 2, dtype=torch.float32) / HEAD_DIM))
    wl = 2 * math.pi / inv
    smooth = (8192 / wl - 1.0) / (4.0 - 1.0)
    mid = (1 - smooth) * inv / 32.0 + smooth * inv
    inv = torch.where(wl > 8192 / 1.0, inv / 32.0, torch.where(wl < 8192 / 4.0, inv, mid))
    return torch.outer(torch.arange(rows, dtype=torch.float32), inv)


def _rope_table(rows):
    a = _angles(rows)
    return torch.stack([torch.cos(a), torch.sin(a)], dim=2).reshape(rows, HEAD_DIM).to(DEV)


def _inputs(case, seed):
    """The values a case works on, from the seed alone."""
    g, kind = _gen(seed), case["kind"]
    if kind in ("gemm", "gemm_rowmajor"):
        W = _normal(g, case["N"], case["K"], std=0.02)
        return {"A": _normal(g, case["M"], case["K"]), "B": W if kind == "gemm" else W.t().contiguous()}
    if kind == "gemm_int4":
        codes, scales = _int4(g, case["N"], case["K"])
        return {"A": _normal(g, case["M"], case["K"]), "codes": codes, "scales": scales}
    if kind == "gemv_int4":
        codes, scales = _int4(g, case["M"], case["K"])
        return {"x": _normal(g, case["K"]), "codes": codes, "scales": scales}
    if kind == "mha":
        return {"q": _normal(g, case["heads"], case["S"], HEAD_DIM), "k": _normal(g, case["kv_heads"], case["S"], HEAD_DIM),
                "v": _normal(g, case["kv_heads"], case["S"], HEAD_DIM)}
    if kind == "gqa_decode":
        H, Hk, L = case["heads"], case["kv_heads"], case["max_len"]
        return {"q": _normal(g, H, HEAD_DIM), "k_new": _normal(g, Hk, HEAD_DIM), "v_new": _normal(g, Hk, HEAD_DIM),
                "k": _normal(g, Hk, L, HEAD_DIM), "v": _normal(g, Hk, L, HEAD_DIM)}
    if kind == "swiglu_prefill":
        E, H, t = case["E"], case["H"], case["b_col_maj"]
        lay = (lambda W: W) if t else (lambda W: W.t().contiguous())
        return {"in": _normal(g, case["S"], E), "w_gate": lay(_normal(g, H, E, std=0.02)),
                "w_up": lay(_normal(g, H, E, std=0.02)), "w_down": lay(_normal(g, E, H, std=0.02))}
    w = _model_weights(g)
    if kind == "prefill":
        ids = torch.randint(0, VOCAB, (case["S"],), generator=g, device=DEV, dtype=torch.int32).cpu()
        return {"weights": w, "ids": ids}
    token = int(torch.randint(0, VOCAB, (1,), generator=g, device=DEV))
    return {"weights": w, "token": token, "kv": [_kv(g, case["pos"]) for _ in range(LAYERS)]}


# ------------------------------------------------------------------------------------------- prepare and run
def prepare(case, seed):
    from iron_amd import operators as ops

    t, kind = _inputs(case, seed), case["kind"]
    if kind == "gemm":
        op = ops.flm.GEMM(M=case["M"], K=case["K"], N=case["N"], epilogue=case["epilogue"])
        return {"fn": op.get_callable(), "args": (t["A"], t["B"]), "out": torch.empty(case["M"], case["N"], dtype=BF16, device=DEV)}
    if kind == "gemm_rowmajor":
        op = ops.GEMM(M=case["M"], K=case["K"], N=case["N"])
        return {"fn": op.get_callable(), "args": (t["A"], t["B"]), "out": torch.empty(case["M"], case["N"], dtype=BF16, device=DEV)}
    if kind == "gemm_int4":
        op = ops.GEMMInt4(M=case["M"], K=case["K"], N=case["N"])
        return {"fn": op.get_callable(), "args": (t["A"], t["codes"], t["scales"]),
                "out": torch.empty(case["M"], case["N"], dtype=BF16, device=DEV)}
    if kind == "gemv_int4":
        op = ops.GEMVInt4(M=case["M"], K=case["K"])
        return {"fn": op.get_callable(), "args": (t["codes"], t["scales"], t["x"]), "out": torch.empty(case["M"], dtype=BF16, device=DEV)}
    if kind == "mha":
        op = ops.MHA(num_heads=case["heads"], seq_len=case["S"], d=HEAD_DIM, num_KV_heads=case["kv_heads"])
        pad = op.seq_padded - case["S"]
        args = tuple(torch.nn.functional.pad(t[n], (0, 0, 0, pad)).reshape(-1) for n in ("q", "k", "v"))
        return {"fn": op.get_callable(), "args": args, "out": torch.empty_like(args[0])}
    if kind == "gqa_decode":
        op = ops.GQADecode(num_heads=case["heads"], num_kv_heads=case["kv_heads"], head_dim=HEAD_DIM, max_len=case["max_len"])
        op.set_position(case["pos"])
        return {"fn": op.get_callable(), "args": (t["q"], t["k_new"], t["v_new"], t["k"], t["v"], _rope_table(case["max_len"])),
                "out": torch.empty(case["heads"], HEAD_DIM, dtype=BF16, device=DEV)}
    if kind == "swiglu_prefill":
        seq = ops.SwiGLUPrefill(seq_len=case["S"], embedding_dim=case["E"], hidden_dim=case["H"], b_col_maj=case["b_col_maj"]).compile()
        fn = seq.get_callable()
        for n, v in t.items():
            fn.get_buffer(n).device_view().copy_(v.reshape(-1))
        return {"fn": fn, "out": fn.get_buffer("out").device_view().view(case["S"], case["E"])}

    from iron_amd.applications.llama_3_2_1b import LlamaConfig, LlamaHIP

    model = LlamaHIP(LlamaConfig(n_layers=LAYERS), t["weights"], device=torch.device(DEV, 0))
    if kind == "prefill":
        return {"model": model, "ids": t["ids"], "graph": case["graph"]}
    pos = case["pos"]
    for i, (k, v) in enumerate(t["kv"]):
        model.k_cache[i][:, :pos] = k
        model.v_cache[i][:, :pos] = v
    model.capture_decode_graph()
    model.set_token(t["token"])
    return {"model": model, "pos": pos, "key": model.keys[:1].clone(), "dev_pos": torch.tensor([pos - 1], dtype=torch.int32, device=DEV)}


def run(state):
    if "model" not in state:
        fn = state["fn"]
        if "args" in state:
            fn(*state["args"], state["out"])
            if len(state["args"]) == 6:  # the decode attention also appends to its caches
                return {"out": state["out"], "k": state["args"][3], "v": state["args"][4]}
        else:
            fn.launch()
        return state["out"]
    m = state["model"]
    if "ids" in state:
        m.reset()
        m.prefill(state["ids"], use_graph=state["graph"])
        rows = slice(0, state["ids"].numel())
    else:  # back to the position and the token of the state, so that a pass can be repeated
        m.host_pos = state["pos"]
        m.pos.copy_(state["dev_pos"])
        m.keys[:1].copy_(state["key"])
        m.decode(1)
        rows = slice(state["pos"], state["pos"] + 1)
    return {"logits": m.logits, "k": [c[:, rows] for c in m.k_cache], "v": [c[:, rows] for c in m.v_cache]}


# ------------------------------------------------------------------------------------------ work and tolerance
_LINEAR = EMB * (HEADS + 2 * KV_HEADS) * HEAD_DIM + EMB * HEADS * HEAD_DIM + 3 * EMB * FFN  # weights of a layer


def work(case):
    kind = case["kind"]
    if kind in ("gemm", "gemm_rowmajor"):
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": 2 * (M * K + N * K + M * N), "flops": 2 * M * N * K}
    if kind == "gemm_int4":
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": 2 * (M * K + M * N) + N * K // 2 + N * K // 16, "flops": 2 * M * N * K}
    if kind == "gemv_int4":
        M, K = case["M"], case["K"]
        return {"bytes": M * K // 2 + M * K // 16 + 2 * K + 2 * M, "flops": 2 * M * K}
    if kind == "mha":
        S, H, Hk = case["S"], case["heads"], case["kv_heads"]
        return {"bytes": 2 * S * HEAD_DIM * (2 * H + 2 * Hk), "flops": 4 * HEAD_DIM * H * S * (S + 1) // 2}
    if kind == "gqa_decode":
        n, H, Hk = case["pos"] + 1, case["heads"], case["kv_heads"]
        return {"bytes": 2 * HEAD_DIM * (2 * Hk * n + 2 * H + 2 * Hk) + 4 * HEAD_DIM, "flops": 4 * HEAD_DIM * H * n}
    if kind == "swiglu_prefill":
        S, E, H = case["S"], case["E"], case["H"]
        return {"bytes": 2 * (3 * E * H + 2 * S * E), "flops": 6 * S * E * H}
    head = 2 * VOCAB * EMB
    if kind == "prefill":  # each layer's int4 weights, the head, the embeddings' rows and the KV rows written
        S = case["S"]
        kv = 2 * 2 * LAYERS * KV_HEADS * HEAD_DIM * S
        return {"bytes": LAYERS * _LINEAR * 9 // 16 + head + 2 * S * EMB + kv + 2 * VOCAB,
                "flops": 2 * LAYERS * S * _LINEAR + LAYERS * 4 * HEAD_DIM * HEADS * S * (S + 1) // 2 + head}
    n = case["pos"] + 1
    kv = 2 * 2 * LAYERS * KV_HEADS * HEAD_DIM * n
    return {"bytes": LAYERS * _LINEAR * 9 // 16 + head + kv + 2 * EMB + 2 * VOCAB,
            "flops": 2 * LAYERS * _LINEAR + LAYERS * 4 * HEAD_DIM * HEADS * n + head}


def tolerance(case):
    # About four times what the start is off 64-bit arithmetic: 1.7e-3 for one bf16 rounding of a 32-bit sum (at most
    # 3.9e-3 in a value). A whole model rounds its activations to bf16 some fifty times on the way to its logits: 0.013
    # to 0.022 off 64 bits, and 0.014 between two orders of its o_proj sums alone.
    kind = case["kind"]
    if kind in ("prefill", "decode"):
        return {"rel": 0.03, "max": 0.3}
    if kind == "swiglu_prefill":  # bf16 gate, up and product on the way
        return {"rel": 0.012, "max": 0.06}
    if kind == "mha":  # the probabilities of the product with V are bf16
        return {"rel": 0.01, "max": 0.06}
    return {"rel": 0.007, "max": 0.02}


# ------------------------------------------------------------------------------------------------------- exact
def _deq(codes, scales):
    """int4 group-32 weights in 64 bits."""
    c = codes.to(torch.int16)
    q = torch.stack([c & 15, c >> 4], dim=2).reshape(codes.shape[0], -1)
    q = torch.where(q > 7, q - 16, q)
    return q.double() * scales.double().repeat_interleave(32, dim=1)


def _quantized(W):
    """bf16 weights after int4 group-32 quantisation (scale bf16(max / 7), nearest code in [-8, 7]), in 64 bits."""
    v = W.float().reshape(W.shape[0], -1, 32)
    s = (v.abs().amax(dim=2).clamp_min(1e-8) / 7.0).to(BF16)
    q = torch.clamp(torch.round(v / s.float().unsqueeze(2)), -8, 7)
    return (q.double() * s.double().unsqueeze(2)).reshape(W.shape)


def _silu(x):
    return x * torch.sigmoid(x)


def _causal(q, k, v):
    """Attention of the last q.shape[1] positions of k, v: (heads, S, d) x (kv heads, L, d)."""
    H, S, d = q.shape
    L, G = k.shape[1], H // k.shape[0]
    out = torch.empty_like(q)
    hide = torch.ones(S, L, dtype=torch.bool, device=q.device).triu(L - S + 1)
    for h in range(H):
        s = (q[h] @ k[h // G].t() / math.sqrt(d)).masked_fill(hide, -math.inf)
        out[h] = torch.softmax(s, dim=1) @ v[h // G]
    return out


def _rotate(x, ang):
    """Two-halves RoPE of x (..., S, 64) by angles (S, 32); cosines and sines as the float32 table has them."""
    c, s = torch.cos(ang).to(x.device).double(), torch.sin(ang).to(x.device).double()
    a, b = x[..., :32], x[..., 32:]
    return torch.cat([a * c - b * s, b * c + a * s], dim=-1)


def _exact_model(case, t):
    w, kind = t["weights"], case["kind"]
    S, pos = (case["S"], 0) if kind == "prefill" else (1, case["pos"])
    ids = t["ids"].to(DEV).long() if kind == "prefill" else torch.tensor([t["token"]], device=DEV)
    ang = _angles(pos + S)[pos:]
    # the norms' weights are folded into the matrices before these are quantised; a prompt's GEMMs take the int4
    # weights rounded to bf16, a token's GEMVs take them as they are
    fold = lambda n, norm: (w[n].float() * w[norm].float().unsqueeze(0)).to(BF16)
    used = (lambda W: _quantized(W).to(BF16).double()) if kind == "prefill" else _quantized
    norm = lambda x: x * torch.rsqrt(x.square().mean(dim=1, keepdim=True) + EPS)
    x = w["model.embed_tokens.weight"][ids].double()
    ks, vs = [], []
    for i in range(LAYERS):
        n = _layer_names(i)
        xn = norm(x)
        proj = lambda p: (xn @ used(fold(n[p], n["input_layernorm"])).t()).view(S, -1, HEAD_DIM).transpose(0, 1)
        q, k, v = _rotate(proj("self_attn.q_proj"), ang), _rotate(proj("self_attn.k_proj"), ang), proj("self_attn.v_proj")
        ks.append(k.contiguous())
        vs.append(v.contiguous())
        if pos:
            k, v = torch.cat([t["kv"][i][0].double(), k], dim=1), torch.cat([t["kv"][i][1].double(), v], dim=1)
        o = _causal(q, k, v).transpose(0, 1).reshape(S, -1)
        x = x + o @ used(w[n["self_attn.o_proj"]]).t()
        xn = norm(x)
        h = _silu(xn @ used(fold(n["mlp.gate_proj"], n["post_attention_layernorm"])).t())
        h = h * (xn @ used(fold(n["mlp.up_proj"], n["post_attention_layernorm"])).t())
        x = x + h @ used(w[n["mlp.down_proj"]]).t()
    head = fold("model.embed_tokens.weight", "model.norm.weight")
    xl = norm(x)[-1]
    logits = torch.cat([part.double() @ xl for part in head.split(16384)])
    return {"logits": logits, "k": ks, "v": vs}


def exact(case, seed):
    t, kind = _inputs(case, seed), case["kind"]
    if kind in ("gemm", "gemm_rowmajor"):
        y = t["A"].double() @ (t["B"].double().t() if kind == "gemm" else t["B"].double())
        act = {"none": lambda v: v, "gelu": lambda v: v * torch.sigmoid(1.702 * v), "silu": _silu, "sigmoid": torch.sigmoid}
        return act[case.get("epilogue", "none")](y)
    if kind == "gemm_int4":  # its weights are rounded to bf16, as the dequantised copy would be
        return t["A"].double() @ _deq(t["codes"], t["scales"]).to(BF16).double().t()
    if kind == "gemv_int4":
        return _deq(t["codes"], t["scales"]) @ t["x"].double()
    if kind == "mha":
        o = _causal(t["q"].double(), t["k"].double(), t["v"].double())
        return torch.nn.functional.pad(o, (0, 0, 0, -case["S"] % 64)).reshape(-1)
    if kind == "gqa_decode":
        p = case["pos"]
        ang = _angles(p + 1)[p:]
        q = _rotate(t["q"].double().unsqueeze(1), ang)
        k, v = t["k"].double(), t["v"].double()
        k[:, p : p + 1] = _rotate(t["k_new"].double().unsqueeze(1), ang)
        v[:, p] = t["v_new"].double()
        return {"out": _causal(q, k[:, : p + 1], v[:, : p + 1])[:, 0], "k": k, "v": v}
    if kind == "swiglu_prefill":
        f = (lambda W: W.double().t()) if case["b_col_maj"] else (lambda W: W.double())
        x = t["in"].double()
        return (_silu(x @ f(t["w_gate"])) * (x @ f(t["w_up"]))) @ f(t["w_down"])
    return _exact_model(case, t)
