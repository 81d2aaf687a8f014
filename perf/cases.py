"""Performance cases of the framework's public entry points.

Five kinds of work, each over the range of sizes and types a user runs:

* ``decode``  -- one token of a loaded model (``Engine``): the chat loop's step.
* ``prefill`` -- a prompt through ``Engine.prefill``.
* ``gemm``    -- one weight matrix times T tokens (``ops.matmul_tokens``): the
  layer matrices of a prompt, each quantized type on its own.
* ``attn``    -- one layer's decode attention (``ops.attention``).
* ``embed`` / ``query`` -- the chat memory: sentence embeddings of many texts
  (``Bert.embed_batch``) and the lookup of one user line (``Bert.query``).

Models have the layer widths of the repository's own configurations, few
layers (a pass over more repeats the same work) and weight blocks drawn on
the GPU.  Values spread like N(0, 0.02), those of the two matrices that add
to the residual stream (attention output and ffn down) by 1/sqrt(2 layers of
the full model) less, as such models are initialised.
"""
import math

import numpy as np
import torch

from ligguf_amd import ops
from ligguf_amd.bert import MINILM_L6, Bert, HostBert, synthetic_vocab
from ligguf_amd.lib import (F16, F32, Q1_0, Q1_G, Q2_K, Q3_K, Q4_K, Q5_K, Q6_K, Q8_0, TYPE_NAMES, load, row_size)
from ligguf_amd.model import QWEN3_8B_Q4K, TINY, Engine, HostModel

DEV = "cuda"
TYPES = {TYPE_NAMES[t]: t for t in (F32, F16, Q8_0, Q2_K, Q3_K, Q4_K, Q5_K, Q6_K, Q1_0, Q1_G)}
# the layer types models are run with, and the type of their output matrix
HEADS = {"Q4_K": "Q6_K", "Q4_K_M": "Q6_K", "Q5_K": "Q6_K", "Q6_K": "Q6_K", "Q8_0": "Q8_0", "Q1_G": "Q8_0", "F16": "F16"}
VOCAB = 32000


# --------------------------------------------------------------------------
# weights
# --------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _halves(x):
    """float tensor -> its fp16 bytes, two per value along the last axis"""
    return x.to(torch.float16).contiguous().view(torch.uint8)


def _weights(t, rows, cols, g, sigma=0.02):
    """rows of type t on the GPU, uint8 [rows, row_size]: random quants and
    sub-block scales, block scales so that the values spread like sigma."""
    if t == F32:
        return (torch.randn(rows, cols, generator=g, device=DEV) * sigma).view(torch.uint8)
    if t == F16:
        return _halves(torch.randn(rows, cols, generator=g, device=DEV) * sigma)
    rsz = row_size(t, cols)
    w = torch.randint(-2 ** 62, 2 ** 62, ((rows * rsz + 7) // 8,), generator=g, device=DEV, dtype=torch.int64)
    w = w.view(torch.uint8)[:rows * rsz].clone().view(rows, rsz)
    block, d_at, dmin_at, unit, dmin = {
        Q8_0: (34, 0, None, 74.0, 0.0), Q1_0: (6, 0, None, 1.0, 0.0), Q1_G: (18, 0, None, 1.0, 0.0),
        Q2_K: (84, 80, 82, 11.0, 1.5), Q3_K: (110, 108, None, 42.0, 0.0), Q4_K: (144, 0, 2, 200.0, 7.5),
        Q5_K: (176, 0, 2, 400.0, 15.5), Q6_K: (210, 208, None, 1370.0, 0.0)}[t]
    b = w.view(rows, rsz // block, block)
    d = (0.6 + 0.8 * torch.rand(rows, rsz // block, 1, generator=g, device=DEV)) * (sigma / unit)
    b[:, :, d_at:d_at + 2] = _halves(d)
    if dmin_at is not None:
        b[:, :, dmin_at:dmin_at + 2] = _halves(d * dmin)   # centres the values on zero
    return w


def _dequant(t, w, cols):
    """float64 values of rows w (uint8 [rows, row_size]) of type t."""
    rows = w.shape[0]
    if t in (F32, F16):
        return w.contiguous().view(torch.float32 if t == F32 else torch.float16).double()

    def half(b, at):
        return b[:, :, at:at + 2].contiguous().view(torch.float16).double()

    def bits(b, n):       # little-endian fields of n bits, in value order
        s = torch.arange(0, 8, n, device=w.device, dtype=torch.uint8)
        return ((b.unsqueeze(-1) >> s) & (2 ** n - 1)).reshape(*b.shape[:-1], -1)

    if t in (Q8_0, Q1_0, Q1_G):
        b = w.view(rows, -1, {Q8_0: 34, Q1_0: 6, Q1_G: 18}[t])
        q = b[:, :, 2:].contiguous().view(torch.int8).double() if t == Q8_0 else 2.0 * bits(b[:, :, 2:], 1).double() - 1.0
        return (half(b, 0) * q).reshape(rows, cols)
    b = w.view(rows, cols // 256, -1)
    if t in (Q4_K, Q5_K):
        s = b[:, :, 4:16].int()
        lo, hi, top = s[:, :, 0:4], s[:, :, 4:8], s[:, :, 8:12]
        sc = torch.cat([lo & 63, (top & 15) | ((lo >> 6) << 4)], -1).double()
        mn = torch.cat([hi & 63, (top >> 4) | ((hi >> 6) << 4)], -1).double()
        qs = b[:, :, -128:].reshape(rows, -1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 3).reshape(rows, -1, 8, 32)
        if t == Q5_K:
            s8 = torch.arange(8, device=w.device, dtype=torch.uint8).view(8, 1)
            q = q + 16 * ((b[:, :, 16:48].unsqueeze(2) >> s8) & 1)
        v = half(b, 0).unsqueeze(-1) * sc.unsqueeze(-1) * q.double() - half(b, 2).unsqueeze(-1) * mn.unsqueeze(-1)
        return v.reshape(rows, cols)
    s4 = torch.arange(0, 8, 2, device=w.device, dtype=torch.uint8).view(4, 1)
    if t == Q6_K:
        ql, qh = b[:, :, 0:128].reshape(rows, -1, 2, 1, 64), b[:, :, 128:192].reshape(rows, -1, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 3).reshape(rows, -1, 2, 4, 32)
        q = (lo | (((qh >> s4) & 3) << 4)).double() - 32.0
        sc = b[:, :, 192:208].contiguous().view(torch.int8).double()
        return (half(b, 208) * sc).unsqueeze(-1).mul(q.reshape(rows, -1, 16, 16)).reshape(rows, cols)
    at = 16 if t == Q2_K else 32
    q = ((b[:, :, at:at + 64].reshape(rows, -1, 2, 1, 32) >> s4) & 3).reshape(rows, -1, 16, 16)
    if t == Q2_K:
        sm = b[:, :, 0:16]
        v = (half(b, 80) * (sm & 15).double()).unsqueeze(-1) * q.double() - (half(b, 82) * (sm >> 4).double()).unsqueeze(-1)
        return v.reshape(rows, cols)
    s8 = torch.arange(8, device=w.device, dtype=torch.uint8).view(8, 1)
    hb = ((b[:, :, 0:32].unsqueeze(2) >> s8) & 1).reshape(rows, -1, 16, 16)
    s = b[:, :, 96:108].int()
    lo = torch.cat([s[:, :, 0:8] & 15, s[:, :, 0:8] >> 4], -1)
    hi = torch.cat([(s[:, :, 8:12] >> (2 * k)) & 3 for k in range(4)], -1)
    sc = (lo | (hi << 4)).double() - 32.0
    return ((half(b, 108) * sc).unsqueeze(-1) * (q.double() + 4.0 * hb.double() - 4.0)).reshape(rows, cols)


def _quantized(t, x):
    """float64 values of the int8 activation a matrix of type t multiplies:
    blocks of 256 (K-quants) or 32 values, rounded in fp32 as the format
    defines; F32/F16 matrices take x itself."""
    if t in (F32, F16):
        return x.double()
    n = 32 if t in (Q8_0, Q1_0, Q1_G) else 256
    v = x.reshape(-1, n)
    at = v.abs().argmax(1, keepdim=True)
    peak = v.gather(1, at)
    if n == 32:
        peak = peak.abs()
        d, inv = (peak * np.float32(1 / 127)).to(torch.float16).double(), torch.div(torch.full_like(peak, 127.0), peak)
    else:
        d, inv = (peak * np.float32(-1 / 127)).double(), torch.div(torch.full_like(peak, -127.0), peak)
    f = v * inv
    if n == 32:         # roundf's halves away from zero; the K form adds its half in fp32
        f = f.double()
    q = torch.trunc(f + torch.copysign(torch.full_like(f, 0.5), f)).double().clamp(max=127)
    return (q * d).reshape(x.shape)


# --------------------------------------------------------------------------
# the cases
# --------------------------------------------------------------------------
def listed():
    return [
        # a small assistant model answering: the smallest step, launches count
        {"name": "decode tiny Q8_0", "kind": "decode", "model": "tiny", "type": "Q8_0", "layers": 6, "pos": 24, "pick": "host"},
        # the usual chat turn: 4-bit weights, some hundred tokens of context
        {"name": "decode Q4_K", "kind": "decode", "model": "wide", "type": "Q4_K", "layers": 4, "pos": 515, "pick": "greedy"},
        # a long conversation on 1-bit weights, sampled
        {"name": "decode Q1_G long", "kind": "decode", "model": "wide", "type": "Q1_G", "layers": 4, "pos": 8200, "pick": "topp"},
        # a prompt of one pass
        {"name": "prefill Q4_K", "kind": "prefill", "type": "Q4_K", "layers": 2, "tokens": 512, "pos": 0},
        # a document pasted into a long conversation: passes with a ragged end over many keys
        {"name": "prefill Q1_G long", "kind": "prefill", "type": "Q1_G", "layers": 2, "tokens": 1100, "pos": 6900},
        # an unquantized model
        {"name": "prefill F16", "kind": "prefill", "type": "F16", "layers": 2, "tokens": 500, "pos": 0},
        # the largest layer matrix (up|gate) over a full pass
        {"name": "gemm Q4_K up", "kind": "gemm", "type": "Q4_K", "rows": 24576, "cols": 4096, "tokens": 512},
        # the down matrix of a 4-bit mix over a short prompt
        {"name": "gemm Q6_K down", "kind": "gemm", "type": "Q6_K", "rows": 4096, "cols": 12288, "tokens": 77},
        # a square matrix of an 8-bit model, a user turn of some hundred tokens
        {"name": "gemm Q8_0", "kind": "gemm", "type": "Q8_0", "rows": 4096, "cols": 4096, "tokens": 200},
        # attention of one layer at the far end of a long context
        {"name": "attn 32k", "kind": "attn", "heads": 32, "kv_heads": 8, "head_dim": 128, "pos": 32767},
        # one user line looked up in the chat memory
        {"name": "query F16", "kind": "query", "type": "F16", "tokens": 23, "rows": 100000},
        # the turns of a chat log embedded at start-up
        {"name": "embed batch F16", "kind": "embed", "type": "F16", "texts": 64, "tokens": 126},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "prefill", "prefill", "gemm", "gemm", "gemm", "attn", "query", "embed"])
    if kind == "decode":
        if rng.random() < 0.3:
            return {"kind": kind, "model": "tiny", "type": "Q8_0", "layers": 6, "pos": rng.randint(1, 250), "pick": "host"}
        return {"kind": kind, "model": "wide", "type": rng.choice(sorted(HEADS)), "layers": 2, "pos": _log(rng, 8, 8190),
                "pick": rng.choice(["host", "greedy", "topp"])}
    if kind == "prefill":
        t = rng.choice(sorted(HEADS))
        return {"kind": kind, "type": t, "layers": 2, "tokens": _log(rng, 3, 480 if t == "F16" else 900),
                "pos": rng.choice([0, 0, _log(rng, 16, 6000)])}
    if kind == "gemm":
        t = rng.choice(sorted(TYPES))
        rows, cols, tokens = 8 * _log(rng, 32, 3000), 256 * _log(rng, 2, 48), _log(rng, 2, 512)
        most = (4096 if t in ("F16", "F32") else 12288) * 4096 * 512
        while rows * cols * tokens > most:
            rows = max(256, rows // 2)
            tokens = max(2, tokens - tokens // 4)
        return {"kind": kind, "type": t, "rows": rows, "cols": cols, "tokens": tokens}
    if kind == "attn":
        nh, nkv, hd = rng.choice([(32, 8, 128), (32, 8, 128), (32, 4, 64), (6, 6, 48), (40, 8, 128)])
        return {"kind": kind, "heads": nh, "kv_heads": nkv, "head_dim": hd, "pos": _log(rng, 2, 32760)}
    if kind == "query":
        return {"kind": kind, "type": rng.choice(["F16", "F16", "F32", "Q8_0"]), "tokens": _log(rng, 2, 500), "rows": _log(rng, 300, 150000)}
    return {"kind": kind, "type": rng.choice(["F16", "F16", "F32", "Q8_0"]), "texts": _log(rng, 2, 60), "tokens": _log(rng, 8, 120)}


def _shape(case):
    """(n_embed, kv_dim, n_ff, heads, kv_heads, head_dim, layer types) of a model case"""
    c = TINY if case.get("model") == "tiny" else QWEN3_8B_Q4K
    t = case["type"]
    types = {n: TYPES["Q4_K" if t == "Q4_K_M" else t] for n in
             ("attn_q", "attn_k", "attn_v", "attn_output", "ffn_up", "ffn_gate", "ffn_down")}
    if t == "Q4_K_M":
        types["attn_v"] = types["ffn_down"] = Q6_K
    return c, types


def _mats(c):
    ne, kv, ff = c.n_embed, c.kv_dim, c.n_ff
    return {"attn_q": (ne, ne), "attn_k": (kv, ne), "attn_v": (kv, ne), "attn_output": (ne, ne), "ffn_up": (ff, ne),
            "ffn_gate": (ff, ne), "ffn_down": (ne, ff)}


def _model_weights(case, seed):
    """{tensor: (type, rows, cols, uint8 GPU rows)} of a model case"""
    c, types = _shape(case)
    g = _gen(seed * 7 + 1)
    head = TYPES[HEADS[case["type"]]]
    w = {"token_embd.weight": (head if case["type"] in ("F16", "Q8_0", "Q1_G") else Q4_K, VOCAB, c.n_embed),
         "output.weight": (head, VOCAB, c.n_embed)}
    for layer in range(case["layers"]):
        for n, (rows, cols) in _mats(c).items():
            w[f"blk.{layer}.{n}.weight"] = (types[n], rows, cols)
    def sigma(n):
        if "attn_output" in n or "ffn_down" in n:
            return 0.02 / math.sqrt(2 * c.n_layers)
        return 0.5 if n.startswith("token_embd") else 0.02

    return {n: (t, rows, cols, _weights(t, rows, cols, g, sigma(n))) for n, (t, rows, cols) in w.items()}


def _context(case):
    if case.get("model") == "tiny":
        return TINY.n_context
    need = case["pos"] + case.get("tokens", 1)
    return 1024 if need <= 1024 else 8704


def _past(case, seed):
    """fp16 K and V rows of the context before the call: per layer [pos][kv_dim]"""
    c, _ = _shape(case)
    g = _gen(seed * 7 + 2)
    n = case["layers"] * case["pos"] * c.kv_dim
    return [torch.randn(n, generator=g, device=DEV).to(torch.float16) for _ in range(2)]


def _rope_freq(c):
    """theta^(-2i/hd) in fp32: the table a model's loader hands over"""
    return (float(c.rope_theta) ** (-2.0 * np.arange(c.head_dim // 2) / c.head_dim)).astype(np.float32)


def _prepare_model(case, seed):
    c, types = _shape(case)
    cfg = c.with_(name="case", n_layers=case["layers"], vocab=VOCAB, n_context=_context(case), layer_type=types["attn_q"],
                  overrides=tuple((n, t) for n, t in types.items() if t != types["attn_q"]))
    w = _model_weights(case, seed)
    cfg = cfg.with_(embd_type=w["token_embd.weight"][0], out_type=w["output.weight"][0])
    hm = HostModel(cfg)
    hm.rope_freq = _rope_freq(cfg)
    for n, (t, rows, cols, data) in w.items():
        hm.weights[n] = (t, rows, cols, data.reshape(-1).cpu().numpy())
    ones = {"attn_norm": cfg.n_embed, "ffn_norm": cfg.n_embed}
    if case.get("model") != "tiny":
        ones.update(attn_q_norm=cfg.head_dim, attn_k_norm=cfg.head_dim)
    for layer in range(cfg.n_layers):
        for n, width in ones.items():
            hm.norms[f"blk.{layer}.{n}.weight"] = np.ones(width, np.float32)
    hm.norms["output_norm.weight"] = np.ones(cfg.n_embed, np.float32)
    eng = Engine(0)
    eng.load(hm)
    if case["pos"]:
        k, v = (p.view(torch.int16).cpu().numpy().view(np.uint16) for p in _past(case, seed))
        eng.kv_write(0, cfg.n_layers, 0, case["pos"], k, v)
    return eng


def _tokens(case, seed):
    return np.random.default_rng(seed).integers(0, VOCAB, case.get("tokens", 1)).astype(np.int32)


class _DeviceFloats:
    """n device floats at an address that `owner` keeps, for torch.as_tensor"""

    def __init__(self, owner, ptr, n):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f4", "data": (ptr, False), "version": 2}


def _encoder_weights(case, seed):
    c = MINILM_L6
    g = _gen(seed * 7 + 3)
    t = TYPES[case["type"]]
    ne, ff = c.n_embed, c.n_ff
    w = {"token_embd.weight": (F16, c.vocab, ne, 1.0), "position_embd.weight": (F16, c.n_context, ne, 0.3),
         "token_types.weight": (F16, 2, ne, 0.3)}
    v = {"token_embd_norm.weight": (ne, 1.0, 0.1), "token_embd_norm.bias": (ne, 0.0, 0.05)}
    for layer in range(c.n_layers):
        b = f"blk.{layer}."
        for n, rows, cols, s in (("attn_q", ne, ne, 0.1), ("attn_k", ne, ne, 0.1), ("attn_v", ne, ne, 0.05),
                                 ("attn_output", ne, ne, 0.05), ("ffn_up", ff, ne, 0.05), ("ffn_down", ne, ff, 0.025)):
            w[b + n + ".weight"] = (t, rows, cols, s)
            v[b + n + ".bias"] = (rows, 0.0, 0.02)
        for n in ("attn_output_norm", "layer_output_norm"):
            v[b + n + ".weight"] = (ne, 1.0, 0.1)
            v[b + n + ".bias"] = (ne, 0.0, 0.05)
    w = {n: (t, rows, cols, _weights(t, rows, cols, g, s)) for n, (t, rows, cols, s) in w.items()}
    v = {n: m + s * torch.randn(k, generator=g, device=DEV) for n, (k, m, s) in v.items()}
    return w, v


def _texts(case, seed):
    """token ids of the case's texts: lengths spread around the case's mean"""
    r = np.random.default_rng(seed)
    n, mean = case.get("texts", 1), case["tokens"]
    lens = r.integers(max(1, mean // 2), mean + mean // 2 + 1, n) if n > 1 else [mean]
    return [r.integers(5, MINILM_L6.vocab, k).astype(np.int32) for k in lens]


def _memory(case, seed):
    g = _gen(seed * 7 + 4)
    m = torch.randn(case["rows"], MINILM_L6.n_embed, generator=g, device=DEV)
    return (m / m.norm(dim=1, keepdim=True)).to(torch.float16)


def _gemm_inputs(case, seed):
    g = _gen(seed * 7 + 5)
    w = _weights(TYPES[case["type"]], case["rows"], case["cols"], g)
    return w, torch.randn(case["tokens"], case["cols"], generator=g, device=DEV)


def _attn_inputs(case, seed):
    g = _gen(seed * 7 + 6)
    nh, nkv, hd, pos = case["heads"], case["kv_heads"], case["head_dim"], case["pos"]
    q, k, v = (torch.randn(n * hd, generator=g, device=DEV) for n in (nh, nkv, nkv))
    kc, vc = (torch.randn(pos * nkv * hd, generator=g, device=DEV).to(torch.float16) for _ in range(2))
    return q, k, v, kc, vc


def prepare(case, seed):
    kind, s = case["kind"], {"case": case}
    if kind in ("decode", "prefill"):
        s["engine"] = _prepare_model(case, seed)
        s["tokens"] = _tokens(case, seed)
        if kind == "decode":
            s["logits"] = torch.as_tensor(
                _DeviceFloats(s["engine"], int(load().lg_logits_device(s["engine"].ctx)), VOCAB), device=DEV)
    elif kind == "gemm":
        w, x = _gemm_inputs(case, seed)
        s.update(w=w.reshape(-1), x=x, rsz=w.shape[1])
    elif kind == "attn":
        s["in"] = _attn_inputs(case, seed)
        need = load().lg_attn_workspace_size(case["heads"], case["head_dim"], case["pos"])
        s["ws"] = torch.empty(max(16, need), dtype=torch.uint8, device=DEV)
    else:
        w, v = _encoder_weights(case, seed)
        hb = HostBert(MINILM_L6, synthetic_vocab(MINILM_L6.vocab)[:MINILM_L6.vocab])
        hb.weights = {n: (t, rows, cols, data.reshape(-1).cpu().numpy()) for n, (t, rows, cols, data) in w.items()}
        hb.vectors = {n: a.cpu().numpy() for n, a in v.items()}
        s["bert"] = Bert(0)
        s["bert"].load(hb)
        s["texts"] = _texts(case, seed)
        if kind == "query":
            s["bert"].vdb_set(_memory(case, seed).view(torch.int16).cpu().numpy().view(np.uint16))
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "decode":
        e, tok, pos = s["engine"], int(s["tokens"][0]), case["pos"]
        if case["pick"] == "host":              # the caller samples from the logits itself
            return e.decode(tok, pos)
        e.decode_async(tok, pos)                # the next token is picked on the device (the logits say how well)
        if case["pick"] == "greedy":
            e.argmax()
        else:
            e.sample_topp(0.8, 0.9, 40, 0.37)
        return s["logits"]
    if kind == "prefill":
        return s["engine"].prefill(s["tokens"], case["pos"])
    if kind == "gemm":
        return ops.matmul_tokens(TYPES[case["type"]], s["w"], s["rsz"], case["cols"], case["rows"], s["x"])
    if kind == "attn":
        return ops.attention(*s["in"], case["heads"], case["kv_heads"], case["head_dim"], case["pos"], s["ws"])
    if kind == "query":
        # every row is a candidate, the three best come back
        return s["bert"].query(s["texts"][0], -1.0, 3)
    return s["bert"].embed_batch(s["texts"])


# --------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        c, types = _shape(case)
        T, pos, head = case.get("tokens", 1), case["pos"], TYPES[HEADS[case["type"]]]
        mats = _mats(c)
        wb = case["layers"] * sum(rows * row_size(types[n], cols) for n, (rows, cols) in mats.items())
        macs = case["layers"] * T * sum(rows * cols for rows, cols in mats.values()) + VOCAB * c.n_embed
        keys = T * pos + T * (T + 1) // 2
        macs += case["layers"] * 2 * keys * c.n_heads * c.head_dim
        kvb = case["layers"] * 2 * 2 * c.kv_dim * (pos + T)
        return {"bytes": wb + kvb + VOCAB * row_size(head, c.n_embed) + 4 * VOCAB, "flops": 2 * macs}
    if kind == "gemm":
        r, c, T = case["rows"], case["cols"], case["tokens"]
        return {"bytes": r * row_size(TYPES[case["type"]], c) + 4 * T * (r + c), "flops": 2 * r * c * T}
    if kind == "attn":
        nh, nkv, hd, pos = case["heads"], case["kv_heads"], case["head_dim"], case["pos"]
        return {"bytes": 4 * pos * nkv * hd + 4 * (2 * nh + 2 * nkv) * hd, "flops": 4 * (pos + 1) * nh * hd}
    c = MINILM_L6.with_(layer_type=TYPES[case["type"]])
    n, mean = case.get("texts", 1), case["tokens"] + 2
    rows = case.get("rows", 0)
    return {"bytes": c.weight_bytes() + n * (mean + 1) * c.n_embed * 2 + 2 * rows * c.n_embed,
            "flops": n * c.flops(mean) + 2 * rows * c.n_embed}


def tolerance(case):
    """Differences another correct implementation shows.

    fp32 sums in another order: 1e-7 for integer block sums, 1.2e-6 for the
    fp32 products of a gemm, 2e-7 for attention; through the layers of an
    unquantized model 2.6e-6 (a prompt in one pass against token by token; 1.1e-5
    of some tokens, whose few fp16 cache values weigh more), of an encoder 2e-6
    (against 64 bits).  Where a layer's output is rounded to
    int8 for the next one, a last-bit difference moves some value to the next
    integer, and within a layer or two the rounding of most activations has
    changed: 8.5e-3 measured between a prompt in one pass and token by token,
    or none where no value was near enough to a boundary."""
    if case["kind"] in ("gemm", "attn"):
        return {"rel": 5e-6, "max": 1e-4}
    if case["type"] in ("F16", "F32"):
        return {"rel": 1e-5, "max": 1e-4} if case["kind"] in ("query", "embed") else {"rel": 4e-5, "max": 4e-4}
    return {"rel": 0.03, "max": 0.3}


# --------------------------------------------------------------------------
# the same in 64 bits
# --------------------------------------------------------------------------
def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _rope(x, pos, freq):
    """adjacent pairs of x [T, heads, hd] turned by pos * freq, the angle in fp32"""
    a = (pos.float().unsqueeze(1) * torch.from_numpy(freq).to(DEV)).double().unsqueeze(1)
    e, o = x[..., 0::2], x[..., 1::2]
    return torch.stack([e * a.cos() - o * a.sin(), e * a.sin() + o * a.cos()], -1).reshape(x.shape)


def _exact_model(case, seed):
    c, _ = _shape(case)
    w = {n: _dequant(t, data, cols) for n, (t, rows, cols, data) in _model_weights(case, seed).items()}
    T, pos0, L = case.get("tokens", 1), case["pos"], case["layers"]
    past = [p.view(L, pos0, c.n_kv_heads, c.head_dim) for p in _past(case, seed)] if pos0 else None
    pos = torch.arange(pos0, pos0 + T, device=DEV)
    x = w["token_embd.weight"][torch.from_numpy(_tokens(case, seed)).long().to(DEV)]
    nh, nkv, hd = c.n_heads, c.n_kv_heads, c.head_dim
    own, freq = torch.arange(T, device=DEV), _rope_freq(c)
    seen = torch.arange(pos0 + T, device=DEV).unsqueeze(0) <= pos.unsqueeze(1)
    for layer in range(L):
        def m(n, a):
            return a @ w[f"blk.{layer}.{n}.weight"].T
        h = _rms(x, c.rms_eps)
        q = _rope(_rms(m("attn_q", h).view(T, nh, hd), c.rms_eps), pos, freq)
        k = _rope(_rms(m("attn_k", h).view(T, nkv, hd), c.rms_eps), pos, freq)
        v = m("attn_v", h).view(T, nkv, hd)
        # earlier positions come from the fp16 cache, a token's own row is exact
        kc, vc = (a.to(torch.float16).double() for a in (k, v))
        if pos0:
            kc, vc = (torch.cat([p[layer].double(), a]) for p, a in zip(past, (kc, vc)))
        out = []
        for g in range(nkv):
            qg = q[:, g * (nh // nkv):(g + 1) * (nh // nkv)].transpose(0, 1).contiguous()
            s = qg @ kc[:, g].T.contiguous()
            s[:, own, pos0 + own] = (qg * k[:, g]).sum(-1)
            p = torch.softmax((s / math.sqrt(hd)).masked_fill(~seen, -math.inf), -1)
            o = p @ vc[:, g].contiguous() + p[:, own, pos0 + own].unsqueeze(-1) * (v[:, g] - vc[pos0:, g])
            out.append(o.transpose(0, 1).reshape(T, -1))
        x = x + m("attn_output", torch.cat(out, 1))
        h = _rms(x, c.rms_eps)
        x = x + m("ffn_down", torch.nn.functional.silu(m("ffn_gate", h)) * m("ffn_up", h))
    return _rms(x[-1], c.rms_eps) @ w["output.weight"].T


def _exact_embed(case, seed):
    c = MINILM_L6
    w, vec = _encoder_weights(case, seed)
    w = {n: _dequant(t, data, cols) for n, (t, rows, cols, data) in w.items()}
    vec = {n: a.double() for n, a in vec.items()}
    cls, sep = 2, 3     # of the synthetic vocabulary

    def ln(x, n):
        d = x - x.mean(-1, keepdim=True)
        return d / torch.sqrt((d * d).mean(-1, keepdim=True) + c.eps) * vec[n + ".weight"] + vec[n + ".bias"]

    out = []
    for ids in _texts(case, seed):
        t = torch.tensor([cls, *ids[:c.n_context - 2].tolist(), sep], device=DEV)
        n, nh, hd = t.numel(), c.n_heads, c.head_dim
        x = ln(w["token_embd.weight"][t] + w["position_embd.weight"][:n] + w["token_types.weight"][0], "token_embd_norm")
        for layer in range(c.n_layers):
            b = f"blk.{layer}."

            def m(name, a):
                return a @ w[b + name + ".weight"].T + vec[b + name + ".bias"]
            q, k, v = (m(name, x).view(n, nh, hd).transpose(0, 1).contiguous() for name in ("attn_q", "attn_k", "attn_v"))
            p = torch.softmax(q @ k.transpose(1, 2).contiguous() / math.sqrt(hd), -1)
            y = ln(x + m("attn_output", (p @ v).transpose(0, 1).reshape(n, -1)), b + "attn_output_norm")
            u = m("ffn_up", y)
            u = 0.5 * u * (1 + torch.tanh(0.7978845608 * (u + 0.044715 * u ** 3)))
            x = ln(y + m("ffn_down", u), b + "layer_output_norm")
        e = x.mean(0)
        out.append(e / e.norm())
    return torch.stack(out)


def exact(case, seed):
    kind = case["kind"]
    if kind == "gemm":
        t = TYPES[case["type"]]
        w, x = _gemm_inputs(case, seed)
        a = _quantized(t, x)
        return torch.cat([a @ _dequant(t, p, case["cols"]).T for p in w.split(4096)], 1)
    if kind == "attn":
        nh, nkv, hd, pos = case["heads"], case["kv_heads"], case["head_dim"], case["pos"]
        q, k, v, kc, vc = _attn_inputs(case, seed)
        k, v = (torch.cat([c.view(pos, nkv, hd).double(), a.view(1, nkv, hd).double()]) for c, a in ((kc, k), (vc, v)))
        q = q.view(nkv, nh // nkv, hd).double()
        p = torch.softmax(q @ k.permute(1, 2, 0).contiguous() / math.sqrt(hd), -1)
        return (p @ v.transpose(0, 1).contiguous()).reshape(-1)
    if case["type"] not in ("F16", "F32"):
        # int8 activations between the layers: which of two integers a value
        # next to a boundary is rounded to decides the distance
        return None
    if kind in ("decode", "prefill"):
        return _exact_model(case, seed)
    e = _exact_embed(case, seed)
    if kind == "embed":
        return e
    sim = _memory(case, seed).double() @ e[0]
    best = torch.topk(sim, 3)
    return best.indices.int(), best.values, e[0]
