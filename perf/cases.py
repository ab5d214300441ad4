"""The work this framework is used for, as cases that can be timed and checked.

A case is a dict of plain values; ``kind`` says which public entry point it goes
through:

  linear    one call of quantized linears that share x (``mlq_hip_quant_linear``,
            or ``mlq_hip_quant_linear_fused`` for 2-3 weights): ``rows`` 1 is a
            decode step's projection, ``rows`` > 1 a prefill's or a small batch's
  pick      the output projection with the greedy pick (``mlq_hip_quant_linear_argmax``)
  attention single-token attention over a KV cache (``mlq_hip_attention_decode``)
  quantize  f32 weights to blocks on the device (``mlq_hip_quantize``)
  prefill   a prompt through a whole model (``mlq_hip_decoder_prefill``)
  step      one token through a whole model (``mlq_hip_decoder_forward``)

``listed`` gives the cases to look at first, ``draw`` more of the same ranges.
"""

import math
import os
import struct
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "mini-llama-cpp-release_amd"))
import mlq_hip as hip  # noqa: E402

QTYPE = {"q8_0": hip.Q8_0, "q4_0": hip.Q4_0, "q4_1": hip.Q4_1}
GGML = {"q8_0": 8, "q4_0": 2, "q4_1": 3}
THETA, EPS = 10000.0, 1e-5
#: rows * out_features * in_features of one linear call at the most (q/k/v of 2048 tokens)
MOST_WORK = 2048 * 12288 * 4096


def listed():
    return [
        # Decode, the smallest call: q/k/v of an 896-wide model with grouped KV heads
        # (rows 896 + 128 + 128): launches and the host path count.
        {"name": "step_qkv_896_q8_0", "kind": "linear", "type": "q8_0", "rows": 1, "m": 896, "also": 128, "parts": 3,
         "k": 896},
        # Decode, the largest projection of a LLaMA-7B-shaped layer: gate and up in one call.
        {"name": "step_gate_up_q4_0", "kind": "linear", "type": "q4_0", "rows": 1, "m": 11008, "also": 11008,
         "parts": 2, "k": 4096},
        # Decode, long rows: the down projection.
        {"name": "step_down_q4_1", "kind": "linear", "type": "q4_1", "rows": 1, "m": 4096, "also": 0, "parts": 1,
         "k": 11008},
        # Decode's end: lm_head of a 32000-token vocabulary, logits and greedy token.
        {"name": "pick_32000_q4_0", "kind": "pick", "type": "q4_0", "m": 32000, "k": 4096},
        # A small batch (short prompt or a few sequences together).
        {"name": "batch_16_q8_0", "kind": "linear", "type": "q8_0", "rows": 16, "m": 4096, "also": 0, "parts": 1,
         "k": 4096},
        # A ragged short prompt on a small model's feed-forward (896 -> 4864, gate and up).
        {"name": "prompt_67_gate_up_q4_1", "kind": "linear", "type": "q4_1", "rows": 67, "m": 4864, "also": 4864,
         "parts": 2, "k": 896},
        # Prefill at the batch the decoder itself uses per pass, LLaMA-7B feed-forward.
        {"name": "prefill_512_q4_0", "kind": "linear", "type": "q4_0", "rows": 512, "m": 11008, "also": 0, "parts": 1,
         "k": 4096},
        # The largest: q/k/v of a long prompt in one call.
        {"name": "prefill_2048_qkv_q8_0", "kind": "linear", "type": "q8_0", "rows": 2048, "m": 4096, "also": 4096,
         "parts": 3, "k": 4096},
        # Attention of one token late in a long context, grouped KV heads.
        {"name": "attention_3000", "kind": "attention", "heads": 32, "kv": 8, "hd": 128, "pos": 2999},
        # Quantizing a layer's f32 weights on the device when a model is prepared.
        {"name": "quantize_11008_q8_0", "kind": "quantize", "type": "q8_0", "rows": 11008, "len": 4096},
        # A 300-token prompt through a whole (two-layer, LLaMA-7B-wide) model.
        {"name": "model_prefill_300", "kind": "prefill", "type": "q4_0", "layers": 2, "heads": 32, "kv": 32,
         "hd": 128, "hidden": 11008, "vocab": 8192, "n": 300},
        # One decode step of the same model after 700 tokens.
        {"name": "model_step_700", "kind": "step", "type": "q4_0", "layers": 2, "heads": 32, "kv": 32, "hd": 128,
         "hidden": 11008, "vocab": 8192, "n": 700},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["decode", "rows", "pick", "attention", "quantize", "prefill", "step"],
                       [24, 36, 6, 10, 8, 9, 7])[0]
    qt = rng.choice(["q8_0", "q4_0", "q4_1"])
    if kind in ("decode", "rows"):
        parts = rng.choice([1, 1, 2, 3])
        if kind == "decode":
            # any whole number of blocks; most widths are whole multiples of 128
            k = 32 * _log(rng, 8, 448) if rng.random() < 0.3 else 128 * _log(rng, 2, 112)
            m = _log(rng, 64, 33000)
            rows = 1
        else:
            k = 64 * _log(rng, 4, 224) if rng.random() < 0.2 else 128 * _log(rng, 2, 112)
            rows = _log(rng, 2, 2048)
            m = _log(rng, 64, 16384)
        if rng.random() < 0.6:
            m = max(64, m // 64 * 64)
        also = 0 if parts == 1 else m if parts == 2 or rng.random() < 0.5 else max(64, m // 256 * 64)
        while rows * (m + (parts - 1) * also) * k > MOST_WORK:
            rows = max(1, rows // 2)
        return {"kind": "linear", "type": qt, "rows": rows, "m": m, "also": also, "parts": parts, "k": k}
    if kind == "pick":
        return {"kind": "pick", "type": qt, "m": _log(rng, 8000, 152000), "k": 128 * _log(rng, 4, 32)}
    if kind == "attention":
        kv = rng.choice([2, 4, 8, 16, 32])
        return {"kind": "attention", "heads": kv * rng.choice([1, 2, 4, 7]) if kv < 16 else kv * rng.choice([1, 2]),
                "kv": kv, "hd": rng.choice([64, 64, 128, 128, 128, 256, 80]), "pos": _log(rng, 1, 8000) - 1}
    if kind == "quantize":
        n = 128 * _log(rng, 2, 86) if rng.random() < 0.7 else _log(rng, 200, 4100)
        return {"kind": "quantize", "type": qt, "rows": min(_log(rng, 64, 16384), 11008 * 4096 // n), "len": n}
    hd = rng.choice([64, 128])
    kv = rng.choice([2, 4, 8, 16]) * 128 // hd
    heads = kv * rng.choice([1, 2, 4])
    while heads * hd > 4096:
        heads //= 2
    kv = min(kv, heads)
    return {"kind": kind, "type": qt, "layers": rng.choice([1, 2, 2]), "heads": heads, "kv": kv, "hd": hd,
            "hidden": 128 * _log(rng, 4, 86), "vocab": _log(rng, 1000, 8192),
            "n": _log(rng, 2, 300) if kind == "prefill" else _log(rng, 1, 1500)}


# ---------------------------------------------------------------- inputs

class Dev:
    """A torch tensor's memory in the form the binding takes device buffers."""

    def __init__(self, t):
        self.t, self.ptr, self.nbytes = t, t.data_ptr(), t.numel() * t.element_size()


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda") * std


def _blocks(g, qt, m, k, std=0.02):
    """An [m, k] weight of N(0, std) in blocks: uint8 [m, blocks * bytes]."""
    w = _randn(g, m, k // 32, 32, std=std)
    if qt == "q8_0":
        d = (w.abs().amax(-1, keepdim=True) / 127).half()
        q = (w / d.float()).round().clamp(-127, 127).to(torch.int8).view(torch.uint8)
        return torch.cat([d.view(torch.uint8), q], -1).reshape(m, -1).contiguous()
    if qt == "q4_0":
        d = (w.abs().amax(-1, keepdim=True) / 7).half()
        q = ((w / d.float()).round() + 8).clamp(0, 15).to(torch.uint8)
        head = [d.view(torch.uint8)]
    else:
        lo, hi = w.amin(-1, keepdim=True), w.amax(-1, keepdim=True)
        d, mn = ((hi - lo) / 15).half(), lo.half()
        q = ((w - mn.float()) / d.float()).round().clamp(0, 15).to(torch.uint8)
        head = [d.view(torch.uint8), mn.view(torch.uint8)]
    return torch.cat(head + [q[..., :16] | (q[..., 16:] << 4)], -1).reshape(m, -1).contiguous()


def _dequant(qt, b, k):
    """The weight of _blocks in 64 bits, [m, k]."""
    m = b.shape[0]
    b = b.reshape(m, k // 32, -1)
    d = b[..., 0:2].contiguous().view(torch.float16).double()
    if qt == "q8_0":
        return (d * b[..., 2:].contiguous().view(torch.int8).double()).reshape(m, k)
    at = 2 if qt == "q4_0" else 4
    q = torch.cat([b[..., at:] & 15, b[..., at:] >> 4], -1).double()
    if qt == "q4_0":
        return (d * (q - 8)).reshape(m, k)
    return (d * q + b[..., 2:4].contiguous().view(torch.float16).double()).reshape(m, k)


def _parts(case):
    return [case["m"]] + [case["also"]] * (case["parts"] - 1)


def _linear_inputs(case, seed):
    g = _gen(seed)
    ms = _parts(case) if case["kind"] == "linear" else [case["m"]]
    ws = [_blocks(g, case["type"], m, case["k"]) for m in ms]
    return ws, _randn(g, case.get("rows", 1), case["k"])


def _attention_inputs(case, seed):
    g = _gen(seed)
    seq = (case["pos"] // 512 + 1) * 512
    q = _randn(g, case["heads"], case["hd"])
    keys = _randn(g, 2, seq, case["kv"], case["hd"])
    return q, keys, _randn(g, 2, seq, case["kv"], case["hd"])


def _model(case, seed):
    """Tensors of a llama model: name -> (dims ne0 first, ggml type, tensor)."""
    g = _gen(seed)
    qt, hd, hidden, vocab = case["type"], case["hd"], case["hidden"], case["vocab"]
    dim, kv = case["heads"] * hd, case["kv"] * hd
    out = {"token_embd.weight": ([dim, vocab], 0, _randn(g, vocab, dim, std=0.5))}

    def linear(name, m, k):
        out[name] = ([k, m], GGML[qt], _blocks(g, qt, m, k, std=k ** -0.5))

    for i in range(case["layers"]):
        p = "blk.%d." % i
        out[p + "attn_norm.weight"] = ([dim], 0, 1 + _randn(g, dim, std=0.1))
        linear(p + "attn_q.weight", dim, dim)
        linear(p + "attn_k.weight", kv, dim)
        linear(p + "attn_v.weight", kv, dim)
        linear(p + "attn_output.weight", dim, dim)
        out[p + "ffn_norm.weight"] = ([dim], 0, 1 + _randn(g, dim, std=0.1))
        linear(p + "ffn_gate.weight", hidden, dim)
        linear(p + "ffn_up.weight", hidden, dim)
        linear(p + "ffn_down.weight", dim, hidden)
    out["output_norm.weight"] = ([dim], 0, 1 + _randn(g, dim, std=0.1))
    linear("output.weight", vocab, dim)
    return out, torch.randint(0, vocab, (case["n"] + 1,), generator=g, device="cuda").cpu().numpy().astype(np.int32)


def _write_gguf(f, case, tensors):
    def s(v):
        return struct.pack("<Q", len(v)) + v.encode()

    u32 = {"llama.block_count": case["layers"], "llama.embedding_length": case["heads"] * case["hd"],
           "llama.feed_forward_length": case["hidden"], "llama.attention.head_count": case["heads"],
           "llama.attention.head_count_kv": case["kv"], "llama.context_length": (case["n"] // 256 + 1) * 256}
    f32 = {"llama.rope.freq_base": THETA, "llama.attention.layer_norm_rms_epsilon": EPS}
    meta = [s("general.architecture") + struct.pack("<I", 8) + s("llama")]
    meta += [s(k) + struct.pack("<II", 4, v) for k, v in u32.items()]
    meta += [s(k) + struct.pack("<If", 6, v) for k, v in f32.items()]
    meta += [s("tokenizer.ggml.tokens") + struct.pack("<IIQ", 9, 8, case["vocab"]) +
             b"".join(s("t%d" % i) for i in range(case["vocab"]))]
    infos, at = [], 0
    for name, (dims, kind, t) in tensors.items():
        at = (at + 31) // 32 * 32
        infos.append(s(name) + struct.pack("<I%dQIQ" % len(dims), len(dims), *dims, kind, at))
        at += t.numel() * t.element_size()
    head = b"GGUF" + struct.pack("<IQQ", 3, len(tensors), len(meta)) + b"".join(meta + infos)
    f.write(head + b"\0" * (-len(head) % 32))
    at = 0
    for _, _, t in tensors.values():
        f.write(b"\0" * (-at % 32))
        at += -at % 32 + t.numel() * t.element_size()
        f.write(t.cpu().numpy().data)


def prepare(case, seed):
    hip.init(0)
    kind = case["kind"]
    if kind in ("linear", "pick"):
        ws, x = _linear_inputs(case, seed)
        rows, k, qt = x.shape[0], case["k"], QTYPE[case["type"]]
        ys = [torch.empty(rows, w.shape[0], device="cuda") for w in ws]
        weights = [hip.Weight.wrap(qt, Dev(w), w.shape[0] * (k // 32), w.shape[0], k) for w in ws]
        st = {"kind": kind, "w": weights, "x": Dev(x), "y": [Dev(y) for y in ys], "rows": rows}
        if kind == "pick":
            st["token"] = Dev(torch.zeros(1, dtype=torch.int32, device="cuda"))
        elif len(ws) > 1:
            st["calls"] = hip.make_calls([(w, st["x"], y, rows) for w, y in zip(weights, st["y"])])
        torch.cuda.synchronize()
        return st
    if kind == "attention":
        q, keys, values = _attention_inputs(case, seed)
        st = {"kind": kind, "t": (q, keys, values), "out": torch.empty_like(q), "seq": keys.shape[1], "case": case}
        torch.cuda.synchronize()
        return st
    if kind == "quantize":
        src = _randn(_gen(seed), case["rows"], case["len"], std=0.02)
        nb = (case["len"] + 31) // 32 * hip.BLOCK_BYTES[QTYPE[case["type"]]]
        dst = torch.zeros(case["rows"], nb, dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        return {"kind": kind, "case": case, "src": Dev(src), "dst": Dev(dst)}
    tensors, tokens = _model(case, seed)
    with tempfile.NamedTemporaryFile(suffix=".gguf") as f:
        _write_gguf(f, case, tensors)
        f.flush()
        dec = hip.Decoder(f.name)
    n = case["n"]
    if kind == "step":
        dec.prefill(tokens[:n])
    return {"kind": kind, "decoder": dec, "tokens": tokens, "n": n}


def run(st):
    kind = st["kind"]
    if kind == "linear":
        if "calls" in st:
            hip.linear_fused(st["calls"])
        else:
            st["w"][0].linear_device(st["x"], st["y"][0], rows=st["rows"], sync=False)
        return [y.t for y in st["y"]]
    if kind == "pick":
        st["w"][0].linear_argmax(st["x"], st["y"][0], st["token"])
        return {"logits": st["y"][0].t, "token": st["token"].t}
    if kind == "attention":
        c, (q, keys, values) = st["case"], st["t"]
        hip._check(hip.load().mlq_hip_attention_decode(0, q.data_ptr(), keys.data_ptr(), values.data_ptr(), 2, 1,
                                                       st["seq"], c["heads"], c["kv"], c["hd"], c["pos"],
                                                       st["out"].data_ptr(), None))
        return st["out"]
    if kind == "quantize":
        c = st["case"]
        hip.quantize_device(QTYPE[c["type"]], st["src"], c["rows"], c["len"], st["dst"])
        return st["dst"].t
    if kind == "prefill":
        return st["decoder"].prefill(st["tokens"][:st["n"]])
    return st["decoder"].forward(int(st["tokens"][st["n"]]), st["n"])


# ---------------------------------------------------------------- what a pass cannot do without

def _weight_bytes(qt, m, k):
    return m * (k // 32) * hip.BLOCK_BYTES[QTYPE[qt]]


def work(case):
    kind = case["kind"]
    if kind in ("linear", "pick"):
        m, rows, k = sum(_parts(case)) if kind == "linear" else case["m"], case.get("rows", 1), case["k"]
        return {"bytes": _weight_bytes(case["type"], m, k) + 4 * rows * (k + m), "flops": 2 * rows * m * k}
    if kind == "attention":
        n, hd = case["pos"] + 1, case["hd"]
        return {"bytes": 8 * n * case["kv"] * hd + 8 * case["heads"] * hd, "flops": 4 * n * case["heads"] * hd}
    if kind == "quantize":
        nb = (case["len"] + 31) // 32 * hip.BLOCK_BYTES[QTYPE[case["type"]]]
        return {"bytes": case["rows"] * (4 * case["len"] + nb), "flops": 4 * case["rows"] * case["len"]}
    dim, kv, hidden = case["heads"] * case["hd"], case["kv"] * case["hd"], case["hidden"]
    per_layer = 2 * dim * dim + 2 * dim * kv + 3 * dim * hidden
    n, rows = case["n"], case["n"] if kind == "prefill" else 1
    weights = case["layers"] * _weight_bytes(case["type"], 1, 32) * per_layer // 32
    weights += _weight_bytes(case["type"], case["vocab"], dim)
    cache = 8 * case["layers"] * kv * (n + (0 if kind == "prefill" else 1))
    pairs = n * (n + 1) // 2 if kind == "prefill" else n + 1
    flops = 2 * rows * case["layers"] * per_layer + 4 * pairs * dim * case["layers"] + 2 * dim * case["vocab"]
    return {"bytes": weights + cache + 4 * rows * dim + 4 * case["vocab"], "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind == "quantize":
        return "exact"  # bytes
    if kind in ("linear", "pick"):
        # One-row Q4 calls take x as 16-bit integers per 32-element block; the
        # others carry f32 sums (1e-7 to 3e-7 off 64 bits).  A tie may move the token.
        if case.get("rows", 1) == 1 and case["type"] != "q8_0":
            return {"rel": 2e-4, "max": 2e-3, "differ": 0.01}
        return {"rel": 2e-6, "max": 4e-5, "differ": 0.01}
    if kind == "attention":
        return {"rel": 3e-6, "max": 6e-5}
    # A whole model: f32 differences travel through its layers.
    return {"rel": 3e-4, "max": 3e-3}


# ---------------------------------------------------------------- the same in 64 bits

def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _rope(x, pos, hd):
    i = torch.arange(hd // 2, device="cuda", dtype=torch.float64)
    a = pos[:, None, None] * THETA ** (-2 * i / hd)
    c, s = torch.cos(a), torch.sin(a)
    x0, x1 = x[..., 0::2], x[..., 1::2]
    return torch.stack([x0 * c - x1 * s, x0 * s + x1 * c], -1).flatten(-2)


def _forward(case, tensors, tokens):
    """Logits of the last token of a llama model in 64 bits."""
    qt, hd, heads, kv = case["type"], case["hd"], case["heads"], case["kv"]
    n = len(tokens)

    def linear(name, x):
        dims, _, b = tensors[name]
        return x @ _dequant(qt, b, dims[0]).T

    pos = torch.arange(n, device="cuda", dtype=torch.float64)
    mask = torch.full((n, n), -math.inf, device="cuda", dtype=torch.float64).triu(1)
    x = tensors["token_embd.weight"][2][torch.from_numpy(tokens.astype(np.int64)).cuda()].double()
    for i in range(case["layers"]):
        p = "blk.%d." % i
        h = _rms(x, tensors[p + "attn_norm.weight"][2].double())
        q = _rope(linear(p + "attn_q.weight", h).view(n, heads, hd), pos, hd)
        k = _rope(linear(p + "attn_k.weight", h).view(n, kv, hd), pos, hd)
        v = linear(p + "attn_v.weight", h).view(n, kv, hd)
        att = torch.empty_like(q)
        for a in range(heads):
            c = a // (heads // kv)
            att[:, a] = torch.softmax(q[:, a] @ k[:, c].T / math.sqrt(hd) + mask, -1) @ v[:, c]
        x = x + linear(p + "attn_output.weight", att.reshape(n, -1))
        h = _rms(x, tensors[p + "ffn_norm.weight"][2].double())
        g = linear(p + "ffn_gate.weight", h)
        x = x + linear(p + "ffn_down.weight", g / (1 + torch.exp(-g)) * linear(p + "ffn_up.weight", h))
    return linear("output.weight", _rms(x[-1:], tensors["output_norm.weight"][2].double()))[0]


def exact(case, seed):
    kind = case["kind"]
    if kind == "quantize":
        return None
    if kind in ("linear", "pick"):
        ws, x = _linear_inputs(case, seed)
        ys = [x.double() @ _dequant(case["type"], w, case["k"]).T for w in ws]
        return ys if kind == "linear" else {"logits": ys[0], "token": None}
    if kind == "attention":
        q, keys, values = _attention_inputs(case, seed)
        n, per = case["pos"] + 1, case["heads"] // case["kv"]
        out = torch.empty(case["heads"], case["hd"], device="cuda", dtype=torch.float64)
        for h in range(case["heads"]):
            k, v = keys[1, :n, h // per].double(), values[1, :n, h // per].double()
            out[h] = torch.softmax((k @ q[h].double()) / math.sqrt(case["hd"]), -1) @ v
        return out
    tensors, tokens = _model(case, seed)
    return _forward(case, tensors, tokens[:case["n"]] if kind == "prefill" else tokens).cpu().numpy()
