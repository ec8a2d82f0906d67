"""What this framework is measured on: the work a program that serves the
Qwen3-4B shape (checkpoint.QWEN3_4B) has it do, through the public calls of
enginekernel_amd.ek_model and enginekernel_amd.ek_kernels.

Kinds of case (the "kind" entry):

  step          one captured-step body of the engine: Qwen3.step, every layer,
                the head, the argmax and the step's bookkeeping, 1..8 rows
  decode        the same layers as single launches: Qwen3.decode and
                argmax_token, replayed as a graph (the engine's form where the
                one-launch step is switched off or does not take the shape)
  prefill       Qwen3.prefill of a left-padded batch of prompts, one or two
                layers of the model (every layer is alike)
  attn_prefill  the prompt's causal attention of one layer alone
  attn_verify   the attention of a speculative verify step
  attn_decode   one layer's decode attention from the raw qkv rows (QK-norm,
                rotary, cache write: rope_attn_decode) or from rotated query
                heads (flash_decode)
  add_norm      the residual add + RMSNorm between two projections
  qk_rope       the QK-norm + rotary + cache write of a prompt's qkv rows

Shapes are the 4B model's except where a case says otherwise; everything is
bf16, the one data type the framework computes in.
"""

import math

import torch
import torch.nn.functional as F

from enginekernel_amd import ek_kernels as K
from enginekernel_amd.checkpoint import QWEN3_4B
from enginekernel_amd.ek_model import Qwen3

HIDDEN, INTER, NQ, NKV, D, VOCAB = 2560, 9728, 32, 8, 128, 151936
EPS, THETA = 1e-6, 5000000.0
BF, F32, F64, I32, I64 = torch.bfloat16, torch.float32, torch.float64, torch.int32, torch.int64
STEPS = 16        # rows of a step's output buffer


def listed():
    return [
        # the headline: one greedy token of a single stream, at the end of a
        # 512-token answer to a 128-token prompt. Six of the model's 36 layers
        # (they are alike) and the head: over 36, a change of summation order
        # in one layer grows past what outputs can be compared by
        {"name": "step_1row_ctx640", "kind": "step", "rows": 1, "ctx": 640, "ragged": False, "layers": 6},
        # one token of a batch of eight left-padded streams (prompts of 64..2048 tokens)
        {"name": "step_8rows_ragged", "kind": "step", "rows": 8, "ctx": 1900, "ragged": True, "layers": 6},
        # the per-launch decode of a small batch
        {"name": "decode_4rows_ctx1000", "kind": "decode", "rows": 4, "ctx": 1000, "ragged": True, "layers": 4},
        # time to first token of a short prompt: few rows, launches count
        {"name": "prefill_1x128", "kind": "prefill", "b": 1, "s": 128, "ragged": False, "layers": 2},
        # a batch of ragged prompts, the longest 1805 tokens
        {"name": "prefill_8x1805_ragged", "kind": "prefill", "b": 8, "s": 1805, "ragged": True, "layers": 2},
        # a long document, where the attention is most of the prefill
        {"name": "attn_prefill_1x16000", "kind": "attn_prefill", "b": 1, "s": 16000, "ragged": False,
         "nq": 32, "nkv": 8, "d": 128},
        # ordinary prompts in a small batch, two query heads per kv head, no size a multiple of a tile
        {"name": "attn_prefill_4x777", "kind": "attn_prefill", "b": 4, "s": 777, "ragged": True,
         "nq": 16, "nkv": 8, "d": 128},
        # three tokens scored at once against a cached text (n-gram drafts)
        {"name": "attn_verify_1x3_ctx2100", "kind": "attn_verify", "b": 1, "n": 3, "ctx": 2100,
         "nq": 32, "nkv": 8, "d": 128},
        # the decode attention of a ragged batch
        {"name": "attn_decode_8rows_ragged", "kind": "attn_decode", "b": 8, "ctx": 1805, "ragged": True, "rope": True,
         "nq": 32, "nkv": 8, "d": 128},
        # the decode attention of one long stream
        {"name": "attn_decode_1row_32768", "kind": "attn_decode", "b": 1, "ctx": 32768, "ragged": False, "rope": False,
         "nq": 32, "nkv": 8, "d": 128},
        # the rows of the ragged prompt batch between two projections
        {"name": "add_norm_14440rows", "kind": "add_norm", "m": 14440, "n": 2560},
        {"name": "qk_rope_8x1805", "kind": "qk_rope", "b": 8, "s": 1805, "nq": 32, "nkv": 8, "d": 128},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "decode", "prefill", "attn_prefill", "attn_verify", "attn_decode", "add_norm",
                       "qk_rope"])
    nq, nkv = rng.choice([(32, 8), (16, 8), (8, 8), (64, 8)])
    d = rng.choice([128, 128, 64])
    if kind == "step":
        rows = rng.randint(1, 8)
        return {"kind": kind, "rows": rows, "ctx": _log_int(rng, 24, 16000 // rows), "ragged": rng.random() < 0.5,
                "layers": rng.randint(2, 6)}
    if kind == "decode":
        rows = rng.randint(1, 8)
        return {"kind": kind, "rows": rows, "ctx": _log_int(rng, 24, 16000 // rows), "ragged": rng.random() < 0.5,
                "layers": rng.randint(1, 4)}
    if kind == "prefill":
        b = rng.randint(1, 8)
        return {"kind": kind, "b": b, "s": _log_int(rng, 17, 14000 // b), "ragged": rng.random() < 0.5,
                "layers": rng.randint(1, 2)}
    if kind == "attn_prefill":
        b = rng.randint(1, 8)
        return {"kind": kind, "b": b, "s": _log_int(rng, 17, 9000 / math.sqrt(b)), "ragged": rng.random() < 0.5,
                "nq": nq, "nkv": nkv, "d": d}
    if kind == "attn_verify":
        return {"kind": kind, "b": rng.randint(1, 2), "n": rng.randint(2, 4), "ctx": _log_int(rng, 20, 16000),
                "nq": nq, "nkv": nkv, "d": d}
    if kind == "attn_decode":
        b = rng.randint(1, 8)
        return {"kind": kind, "b": b, "ctx": _log_int(rng, 24, 32768 // b), "ragged": rng.random() < 0.5,
                "rope": rng.random() < 0.5, "nq": nq, "nkv": nkv, "d": d}
    if kind == "add_norm":
        return {"kind": kind, "m": _log_int(rng, 1, 16000), "n": rng.choice([1024, 2048, 2560, 4096])}
    b = rng.randint(1, 8)
    return {"kind": kind, "b": b, "s": _log_int(rng, 1, 14000 // b), "nq": nq, "nkv": nkv, "d": d}


# ----------------------------------------------------------------------------
# inputs
# ----------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, shape, std=1.0):
    return torch.empty(shape, dtype=BF, device="cuda").normal_(0.0, std, generator=g)


def _gain(g, n):
    return (1.0 + 0.1 * torch.randn(n, dtype=F32, device="cuda", generator=g)).to(BF)


def _lens(b, longest, ragged, seed):
    """Row lengths: the longest as stated, the others (ragged) anywhere from a 32nd of it."""
    if not ragged or b == 1:
        return [longest] * b
    g = torch.Generator().manual_seed(seed)
    lens = torch.randint(max(1, longest // 32), longest + 1, (b,), generator=g).tolist()
    lens[seed % b] = longest
    return lens


def _tables(length, d):
    inv = 1.0 / (THETA ** (torch.arange(0, d, 2, dtype=F32) / d))
    f = torch.outer(torch.arange(length, dtype=F32), inv)
    f = torch.cat((f, f), dim=-1)
    return f.cos().to(BF).cuda(), f.sin().to(BF).cuda()


def _weights(layers, seed):
    """Random weights under the checkpoint's tensor names (normal, 0.02; gains about 1)."""
    g = _gen(seed)
    t = {"model.embed_tokens.weight": _normal(g, (VOCAB, HIDDEN), 0.02), "model.norm.weight": _gain(g, HIDDEN)}
    for i in range(layers):
        p = "model.layers.%d." % i
        for name, rows, cols in (("self_attn.q_proj", NQ * D, HIDDEN), ("self_attn.k_proj", NKV * D, HIDDEN),
                                 ("self_attn.v_proj", NKV * D, HIDDEN), ("self_attn.o_proj", HIDDEN, NQ * D),
                                 ("mlp.gate_proj", INTER, HIDDEN), ("mlp.up_proj", INTER, HIDDEN),
                                 ("mlp.down_proj", HIDDEN, INTER)):
            t[p + name + ".weight"] = _normal(g, (rows, cols), 0.02)
        for name, n in (("self_attn.q_norm", D), ("self_attn.k_norm", D), ("input_layernorm", HIDDEN),
                        ("post_attention_layernorm", HIDDEN)):
            t[p + name + ".weight"] = _gain(g, n)
    return t


def _model(layers, weights):
    return Qwen3(None, torch.device("cuda:0"), tensors=weights, config=dict(QWEN3_4B, num_hidden_layers=layers))


def _decode_inputs(case, seed):
    """The state of `rows` streams in front of a step: cached keys and values
    of the slots [0, ctx), each row's text ending at slot ctx - 1."""
    b, ctx, n = case["rows"], case["ctx"], case["layers"]
    g = _gen(seed + 1)
    cap = -(-(ctx + 1) // 256) * 256
    lens = _lens(b, ctx, case["ragged"], seed)
    keys = torch.zeros((n, b, NKV, cap, D), dtype=BF, device="cuda")
    values = torch.zeros((n, b, NKV, cap, D), dtype=BF, device="cuda")
    keys[:, :, :, :ctx] = _normal(g, (n, b, NKV, ctx, D))
    values[:, :, :, :ctx] = _normal(g, (n, b, NKV, ctx, D))
    tokens = torch.randint(0, VOCAB, (b,), generator=g, device="cuda")
    return tokens, lens, keys, values, cap


def prepare(case, seed):
    kind = case["kind"]
    g = _gen(seed)
    if kind in ("step", "decode"):
        b, ctx = case["rows"], case["ctx"]
        model = _model(case["layers"], _weights(case["layers"], seed))
        tokens, lens, keys, values, cap = _decode_inputs(case, seed)
        # token, position, slot per row, then the shared length and the step counter: one block, set by one copy
        seed_state = torch.cat([tokens, torch.tensor(lens + [0] * b + [ctx, 0], dtype=I64, device="cuda")])
        state = seed_state.clone()
        st = {"case": case, "model": model, "k": [x for x in keys], "v": [x for x in values], "seed_state": seed_state,
              "state": state, "tokens": state[:b], "positions": state[b:2 * b], "slot": state[2 * b:3 * b],
              "len": state[3 * b:3 * b + 1], "step_idx": state[3 * b + 1:],
              "start": torch.tensor([ctx - n for n in lens], dtype=I32, device="cuda"),
              "out_buf": torch.zeros((STEPS, b), dtype=I32, device="cuda"),
              "ws": K.make_workspace(b, NQ, NKV, D, cap, "cuda"),
              "logits": torch.empty((b, VOCAB), dtype=BF, device="cuda"),
              "k_new": keys[:, :, :, ctx], "v_new": values[:, :, :, ctx]}
        if kind == "decode":
            st["graph"] = None
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                _decode_body(st)
            torch.cuda.current_stream().wait_stream(side)
            torch.cuda.synchronize()
            st["state"].copy_(st["seed_state"])
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                st["hidden"] = _decode_body(st)
            st["graph"] = graph
        return st
    if kind == "prefill":
        b, s, n = case["b"], case["s"], case["layers"]
        model = _model(n, _weights(n, seed))
        lens = _lens(b, s, case["ragged"], seed)
        pad = torch.tensor([s - x for x in lens], device="cuda")
        col = torch.arange(s, device="cuda")
        real = col[None] >= pad[:, None]
        ids = torch.randint(0, VOCAB, (b, s), generator=g, device="cuda") * real
        pos = (col[None] - pad[:, None]) * real
        bias = None
        if case["ragged"] and b > 1:
            seen = (col[:, None] >= col[None])[None] & real[:, None, :]
            bias = torch.where(seen, 0.0, -math.inf).to(BF).unsqueeze(1)
        return {"case": case, "model": model, "ids": ids, "pos": pos, "bias": bias,
                "k": [torch.zeros((b, NKV, s, D), dtype=BF, device="cuda") for _ in range(n)],
                "v": [torch.zeros((b, NKV, s, D), dtype=BF, device="cuda") for _ in range(n)]}
    if kind == "add_norm":
        return {"case": case, "x": _normal(g, (case["m"], case["n"]), 0.5), "residual": _normal(g, (case["m"], case["n"])),
                "w": _gain(g, case["n"])}
    nq, nkv, d = case["nq"], case["nkv"], case["d"]
    b = case["b"]
    st = {"case": case, "nq": nq}
    if kind == "qk_rope":
        s = case["s"]
        cos, sin = _tables(s, d)
        st.update(qkv=_normal(g, (b * s, (nq + 2 * nkv) * d)), qn=_gain(g, d), kn=_gain(g, d),
                  cos=cos.repeat(b, 1), sin=sin.repeat(b, 1), slot=torch.zeros(b, dtype=I64, device="cuda"),
                  k=torch.zeros((b, nkv, s, d), dtype=BF, device="cuda"),
                  v=torch.zeros((b, nkv, s, d), dtype=BF, device="cuda"))
        return st
    if kind == "attn_prefill":
        s = case["s"]
        lens = _lens(b, s, case["ragged"], seed)
        st.update(qkv=_normal(g, (b * s, (nq + 2 * nkv) * d)), k=_normal(g, (b, nkv, s, d)), v=_normal(g, (b, nkv, s, d)),
                  start=torch.tensor([s - x for x in lens], dtype=I32, device="cuda"), s=s)
        return st
    if kind == "attn_verify":
        n, ctx = case["n"], case["ctx"]
        cap = -(-(ctx + n) // 256) * 256
        lens = [ctx] + [max(1, ctx - 3 * i) for i in range(1, b)]
        st.update(qkv=_normal(g, (b * n, (nq + 2 * nkv) * d)), k=_normal(g, (b, nkv, cap, d)), v=_normal(g, (b, nkv, cap, d)),
                  start=torch.zeros(b, dtype=I32, device="cuda"), len=torch.tensor(lens, dtype=I64, device="cuda"), n=n)
        return st
    # attn_decode: slots [0, ctx) hold the text; with rope the newest of them is written by the call
    ctx = case["ctx"]
    cap = -(-ctx // 256) * 256
    lens = _lens(b, ctx, case["ragged"], seed)
    st.update(k=_normal(g, (b, nkv, cap, d)), v=_normal(g, (b, nkv, cap, d)),
              len=torch.full((1,), ctx, dtype=I64, device="cuda"),
              start=torch.tensor([ctx - x for x in lens], dtype=I32, device="cuda"),
              ws=K.make_workspace(b, nq, nkv, d, cap, "cuda"))
    if case["rope"]:
        cos, sin = _tables(ctx, d)
        st.update(qkv=_normal(g, (b, (nq + 2 * nkv) * d)), qn=_gain(g, d), kn=_gain(g, d), cos=cos, sin=sin,
                  positions=torch.tensor([x - 1 for x in lens], dtype=I64, device="cuda"),
                  k_new=st["k"][:, :, ctx - 1], v_new=st["v"][:, :, ctx - 1])
    else:
        st.update(q=_normal(g, (b, nq, d)))
    return st


# ----------------------------------------------------------------------------
# one pass
# ----------------------------------------------------------------------------
def _decode_body(st):
    m = st["model"]
    hidden = m.decode(st["tokens"], st["positions"], st["k"], st["v"], st["slot"], st["len"], st["start"], st["ws"])
    m.argmax_token(hidden, logits=st["logits"])
    return hidden


def run(st):
    c = st["case"]
    kind = c["kind"]
    if kind == "step":
        st["state"].copy_(st["seed_state"])
        st["model"].step(st["tokens"], st["positions"], st["k"], st["v"], st["slot"], st["len"], st["start"], st["ws"],
                         st["out_buf"], st["step_idx"], logits=st["logits"])
        return {"logits": st["logits"], "k_new": st["k_new"], "v_new": st["v_new"]}
    if kind == "decode":
        st["state"].copy_(st["seed_state"])
        st["graph"].replay()
        return {"hidden": st["hidden"], "logits": st["logits"], "k_new": st["k_new"], "v_new": st["v_new"]}
    if kind == "prefill":
        hidden = st["model"].prefill(st["ids"], st["pos"], st["k"], st["v"], st["bias"])
        return {"hidden": hidden, "k": st["k"], "v": st["v"]}
    if kind == "attn_prefill":
        return K.attn_prefill(st["qkv"], st["k"], st["v"], st["start"], st["s"], st["nq"], c["d"] ** -0.5)
    if kind == "attn_verify":
        return K.attn_verify(st["qkv"], st["k"], st["v"], st["start"], st["len"], st["n"], st["nq"], c["d"] ** -0.5)
    if kind == "attn_decode":
        if not c["rope"]:
            return K.flash_decode(st["q"], st["k"], st["v"], st["len"], st["start"], st["ws"], c["d"] ** -0.5)
        out = K.rope_attn_decode(st["qkv"], st["qn"], st["kn"], st["cos"], st["sin"], st["k"], st["v"], st["len"],
                                 st["start"], st["ws"], c["d"] ** -0.5, st["nq"], EPS, positions=st["positions"])
        return {"out": out, "k_new": st["k_new"], "v_new": st["v_new"]}
    if kind == "add_norm":
        y, residual = K.add_rms_norm(st["x"], st["residual"], st["w"], EPS)
        return {"y": y, "residual": residual}
    K.qk_norm_rope_kv(st["qkv"], st["qn"], st["kn"], st["cos"], st["sin"], st["k"], st["v"], st["slot"], c["nq"],
                      c["nkv"], EPS, c["s"])
    return {"q": st["qkv"][:, :c["nq"] * c["d"]], "k": st["k"], "v": st["v"]}


# ----------------------------------------------------------------------------
# what a pass cannot do without
# ----------------------------------------------------------------------------
LAYER_W = (NQ + 2 * NKV) * D * HIDDEN + HIDDEN * NQ * D + 3 * INTER * HIDDEN     # weights of a layer


def _keys(lens):
    """(query, key) pairs of the causal attention over prompts of these lengths."""
    return sum(n * (n + 1) // 2 for n in lens)


def work(case):
    kind = case["kind"]
    if kind in ("step", "decode"):
        b, n = case["rows"], case["layers"]
        # a ragged batch's rows are about half the longest on average
        keys = case["ctx"] * (b if not case["ragged"] else 1 + 0.52 * (b - 1))
        return {"bytes": 2 * (n * LAYER_W + VOCAB * HIDDEN) + n * keys * 4 * NKV * D + 2 * b * VOCAB,
                "flops": 2 * b * (n * LAYER_W + VOCAB * HIDDEN) + n * keys * 4 * NQ * D}
    if kind == "prefill":
        b, s, n = case["b"], case["s"], case["layers"]
        rows = b * s if not (case["ragged"] and b > 1) else s * (1 + 0.52 * (b - 1))     # real tokens, about
        pairs = _keys([s]) * (1 if b == 1 else b if not case["ragged"] else 1 + 0.36 * (b - 1))
        return {"bytes": n * (2 * LAYER_W + rows * 4 * NKV * D) + 2 * rows * HIDDEN,
                "flops": n * (2 * rows * LAYER_W + pairs * 4 * NQ * D)}
    if kind == "add_norm":
        return {"bytes": 8 * case["m"] * case["n"], "flops": 6 * case["m"] * case["n"]}
    nq, nkv, d, b = case["nq"], case["nkv"], case["d"], case["b"]
    if kind == "qk_rope":
        rows = b * case["s"]
        return {"bytes": rows * d * (4 * (nq + 2 * nkv) + 4), "flops": 10 * rows * (nq + nkv) * d}
    if kind == "attn_prefill":
        s = case["s"]
        pairs = _keys([s]) * (1 if b == 1 else b if not case["ragged"] else 1 + 0.36 * (b - 1))
        return {"bytes": b * s * d * (4 * nq + 4 * nkv), "flops": pairs * 4 * nq * d}
    if kind == "attn_verify":
        n = case["n"]
        return {"bytes": b * (case["ctx"] + n) * 4 * nkv * d + 4 * b * n * nq * d,
                "flops": b * n * (case["ctx"] + n) * 4 * nq * d}
    keys = case["ctx"] * (b if not case["ragged"] else 1 + 0.52 * (b - 1))
    return {"bytes": keys * 4 * nkv * d + 4 * b * nq * d, "flops": keys * 4 * nq * d}


# ----------------------------------------------------------------------------
# how far another correct implementation may be
# ----------------------------------------------------------------------------
def tolerance(case):
    kind = case["kind"]
    # bf16 through several layers (each is 0.010..0.017 off the 64-bit result)
    if kind in ("step", "decode", "prefill"):
        return {"rel": 0.03, "max": 0.3}
    # one bf16 product chain and its rounding (0.002..0.004 off)
    if kind in ("attn_prefill", "attn_verify", "attn_decode"):
        return {"rel": 0.01, "max": 0.1}
    # a rounded row (0.003 off); another order of the row's sum moves single roundings
    return {"rel": 0.005, "max": 0.05}


# ----------------------------------------------------------------------------
# the same in 64 bits
# ----------------------------------------------------------------------------
def _norm64(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.to(F64)


def _rope64(x, cos, sin):
    """x [..., rows, heads, d], cos/sin [rows, d]."""
    half = x.shape[-1] // 2
    turned = torch.cat((-x[..., half:], x[..., :half]), dim=-1)
    return x * cos.to(F64).unsqueeze(-2) + turned * sin.to(F64).unsqueeze(-2)


def _attend64(q, k, v, seen):
    """q [n, heads, d], k/v [heads_kv, keys, d], seen [n, keys] -> [n, heads, d]; a query that sees nothing gets zeros."""
    n, heads, d = q.shape
    group = heads // k.shape[0]
    out = torch.empty_like(q)
    for h in range(heads):
        s = (q[:, h] @ k[h // group].to(F64).t()) * d ** -0.5
        s.masked_fill_(~seen, -math.inf)
        out[:, h] = torch.nan_to_num(torch.softmax(s, dim=-1)) @ v[h // group].to(F64)
    return out


def _prompt64(q, k, v, start, s):
    """Causal attention of one left-padded prompt; padding tokens see themselves. In blocks of queries."""
    at = torch.arange(s, device=q.device)
    out = torch.empty_like(q)
    for t0 in range(0, s, 4096):
        t = at[t0:t0 + 4096, None]
        end = min(s, t0 + 4096)
        seen = ((at[None, :end] <= t) & (at[None, :end] >= start)) | ((t < start) & (at[None, :end] == t))
        out[t0:end] = _attend64(q[t0:end], k[:, :end], v[:, :end], seen)
    return out


def _layer64(w, i, x, cos, sin, attend):
    """One layer over residual rows x (float64); attend(q, k, v) does the attention. Returns (x, k, v)."""
    p = "model.layers.%d." % i

    def proj(rows, name):
        return rows @ w[p + name + ".weight"].to(F64).t()

    h = _norm64(x, w[p + "input_layernorm.weight"])
    q = _norm64(proj(h, "self_attn.q_proj").view(-1, NQ, D), w[p + "self_attn.q_norm.weight"])
    k = _norm64(proj(h, "self_attn.k_proj").view(-1, NKV, D), w[p + "self_attn.k_norm.weight"])
    q, k = _rope64(q, cos, sin), _rope64(k, cos, sin)
    v = proj(h, "self_attn.v_proj").view(-1, NKV, D)
    x = x + proj(attend(q, k, v).reshape(x.shape[0], -1), "self_attn.o_proj")
    h = _norm64(x, w[p + "post_attention_layernorm.weight"])
    return x + proj(F.silu(proj(h, "mlp.gate_proj")) * proj(h, "mlp.up_proj"), "mlp.down_proj"), k, v


def exact(case, seed):
    kind = case["kind"]
    if kind in ("step", "decode"):
        b, ctx, n = case["rows"], case["ctx"], case["layers"]
        w = _weights(n, seed)
        tokens, lens, keys, values, _ = _decode_inputs(case, seed)
        cos, sin = _tables(ctx + 1, D)
        pos = torch.tensor(lens, device="cuda")
        x = w["model.embed_tokens.weight"][tokens].to(F64)
        k_new, v_new = [], []
        for i in range(n):
            def attend(q, k, v):
                rows = []
                for r in range(b):
                    lo = ctx - lens[r]
                    kr = torch.cat((keys[i, r, :, lo:ctx].to(F64), k[r].unsqueeze(1)), dim=1)
                    vr = torch.cat((values[i, r, :, lo:ctx].to(F64), v[r].unsqueeze(1)), dim=1)
                    rows.append(_attend64(q[r:r + 1], kr, vr, torch.ones((1, kr.shape[1]), dtype=torch.bool, device="cuda")))
                return torch.cat(rows)
            x, k, v = _layer64(w, i, x, cos[pos], sin[pos], attend)
            k_new.append(k)
            v_new.append(v)
        hidden = _norm64(x, w["model.norm.weight"])
        emb = w["model.embed_tokens.weight"]
        logits = torch.cat([hidden @ emb[r:r + 32768].to(F64).t() for r in range(0, VOCAB, 32768)], dim=1)
        out = {"logits": logits, "k_new": torch.stack(k_new), "v_new": torch.stack(v_new)}
        return dict(out, hidden=hidden) if kind == "decode" else out
    if kind == "prefill":
        st = prepare(case, seed)
        b, s, n = case["b"], case["s"], case["layers"]
        w = _weights(n, seed)
        cos, sin = _tables(s, D)
        pos = st["pos"].reshape(-1)
        starts = [s - x for x in _lens(b, s, case["ragged"], seed)]
        x = w["model.embed_tokens.weight"][st["ids"].reshape(-1)].to(F64)
        ks, vs = [], []
        for i in range(n):
            def attend(q, k, v):
                return torch.cat([_prompt64(q[r * s:(r + 1) * s], k[r * s:(r + 1) * s].transpose(0, 1),
                                            v[r * s:(r + 1) * s].transpose(0, 1), starts[r], s) for r in range(b)])
            x, k, v = _layer64(w, i, x, cos[pos], sin[pos], attend)
            ks.append(k.view(b, s, NKV, D).transpose(1, 2))
            vs.append(v.view(b, s, NKV, D).transpose(1, 2))
        return {"hidden": _norm64(x.view(b, s, HIDDEN)[:, -1], w["model.norm.weight"]), "k": ks, "v": vs}
    st = prepare(case, seed)
    if kind == "add_norm":
        r = st["x"].to(F64) + st["residual"].to(F64)
        return {"y": _norm64(r, st["w"]), "residual": r}
    nq, nkv, d, b = case["nq"], case["nkv"], case["d"], case["b"]
    if kind == "qk_rope":
        s = case["s"]
        x = st["qkv"].view(b * s, nq + 2 * nkv, d).to(F64)
        q = _rope64(_norm64(x[:, :nq], st["qn"]), st["cos"], st["sin"])
        k = _rope64(_norm64(x[:, nq:nq + nkv], st["kn"]), st["cos"], st["sin"])
        return {"q": q.reshape(b * s, -1), "k": k.view(b, s, nkv, d).transpose(1, 2),
                "v": x[:, nq + nkv:].reshape(b, s, nkv, d).transpose(1, 2)}
    if kind == "attn_prefill":
        s = case["s"]
        q = st["qkv"].view(b, s, nq + 2 * nkv, d)[:, :, :nq].to(F64)
        return torch.cat([_prompt64(q[r], st["k"][r], st["v"][r], int(st["start"][r]), s).reshape(s, -1)
                          for r in range(b)])
    if kind == "attn_verify":
        n = case["n"]
        q = st["qkv"].view(b, n, nq + 2 * nkv, d)[:, :, :nq].to(F64)
        rows = []
        for r in range(b):
            ln = int(st["len"][r])
            at = torch.arange(ln + n, device="cuda")
            seen = at[None] <= ln + torch.arange(n, device="cuda")[:, None]
            rows.append(_attend64(q[r], st["k"][r, :, :ln + n], st["v"][r, :, :ln + n], seen).reshape(n, -1))
        return torch.cat(rows)
    ctx = case["ctx"]
    k, v = st["k"][:, :, :ctx].to(F64), st["v"][:, :, :ctx].to(F64)
    if case["rope"]:
        x = st["qkv"].view(b, nq + 2 * nkv, d).to(F64)
        cos, sin = st["cos"][st["positions"]], st["sin"][st["positions"]]
        q = _rope64(_norm64(x[:, :nq], st["qn"]), cos, sin)
        k[:, :, ctx - 1] = _rope64(_norm64(x[:, nq:nq + nkv], st["kn"]), cos, sin)
        v[:, :, ctx - 1] = x[:, nq + nkv:]
    else:
        q = st["q"].to(F64)
    out = torch.cat([_attend64(q[r:r + 1], k[r, :, int(st["start"][r]):], v[r, :, int(st["start"][r]):],
                               torch.ones((1, ctx - int(st["start"][r])), dtype=torch.bool, device="cuda")) for r in range(b)])
    return {"out": out, "k_new": k[:, :, ctx - 1], "v_new": v[:, :, ctx - 1]} if case["rope"] else out
