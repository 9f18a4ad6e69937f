"""The work a user of this framework has it do: the layers of a qwen35-27B-shaped model through `HipWeightRuntime`.

Each case is one pass of one part of a forward pass, by the calls that a decode, verify or prompt pass makes:

  layers  every matvec of three gated-delta layers and one attention layer at 1-4 tokens, as one captured graph
  ffn     gate and up from one input, down from another: `qmv_group` + `qmv`; with `prompt` the MFMA contraction
  head    the LM head with its argmax, logits kept
  delta   causal conv, gated delta rule and gated norm of a pass over sequence slots
  attn    gated query split, RoPE, KV append, paged attention and gate of a pass over sequence slots

Matrices that follow each other in a model read inputs of their own here: activations are quantized to 8 bits, so a
last-bit change in one output would move codes of the next input, and what is compared is each matrix's own work.
"""
import math

import numpy as np
import torch

from vinf_3080ti_amd.runtime import HipWeightRuntime
from vinf_3080ti_amd.tables import table

HIDDEN, FFN, VOCAB = 5120, 17408, 248320
KEY_HEADS, VALUE_HEADS, KD, VD, TAPS = 16, 48, 128, 128, 4
CONV = 2 * KEY_HEADS * KD + VALUE_HEADS * VD
HEADS, KV_HEADS, HD, ROT, ROPE_BASE = 24, 4, 256, 64, 1e7
PAGE = 64
EPS = 1e-6

# GGUF type -> (id, elements per block, bytes per block, byte offsets of its fp16 scales)
TYPES = {
    "Q8_0": (8, 32, 34, (0,)),
    "Q2_K": (10, 256, 84, (80, 82)),
    "Q3_K": (11, 256, 110, (108,)),
    "Q4_K": (12, 256, 144, (0, 2)),
    "Q5_K": (13, 256, 176, (0, 2)),
    "Q6_K": (14, 256, 210, (208,)),
    "IQ2_XXS": (16, 256, 66, (0,)),
    "IQ2_XS": (17, 256, 74, (0,)),
    "IQ3_XXS": (18, 256, 98, (0,)),
    "IQ4_NL": (20, 32, 18, (0,)),
    "IQ3_S": (21, 256, 110, (0,)),
    "IQ2_S": (22, 256, 82, (0,)),
    "IQ4_XS": (23, 256, 136, (0,)),
}
# The feed-forward pairs (gate and up, down) that quant mixes use.
MIXES = [("Q3_K", "Q4_K"), ("Q3_K", "Q6_K"), ("Q4_K", "Q6_K"), ("Q4_K", "Q4_K"), ("Q5_K", "Q6_K"), ("Q2_K", "Q3_K"),
         ("IQ2_XXS", "IQ3_S"), ("IQ2_XS", "IQ2_S"), ("IQ3_XXS", "IQ4_XS"), ("IQ4_XS", "IQ4_XS"), ("IQ4_NL", "Q5_K"),
         ("Q8_0", "Q8_0")]


def listed():
    ffn = dict(op="ffn", hidden=HIDDEN, ffn=FFN, prompt=False, f16=False)
    attn = dict(op="attn", elem=2)
    return [
        # a decode step's weight sweep: the headline workload, four layers of it
        dict(name="decode layers, 1 token", op="layers", ntok=1),
        # a decode step's feed-forward in a codebook mix
        dict(ffn, name="ffn IQ, 1 token", gate="IQ2_XXS", down="IQ3_S", ntok=1),
        # four sequences decoded together, or a short draft verified
        dict(ffn, name="ffn K-quants, 4 tokens", gate="Q3_K", down="Q4_K", ntok=4),
        # speculative verify
        dict(ffn, name="ffn K-quants, 8 tokens", gate="Q3_K", down="Q6_K", ntok=8),
        # a prompt chunk with the CPU path's int8 activations
        dict(ffn, name="ffn prompt, 512 tokens", gate="Q4_K", down="Q4_K", ntok=512, prompt=True),
        # a ragged prompt chunk with f16 activations, the down projection of a type that keeps int8 ones
        dict(ffn, name="ffn prompt f16, 243 tokens", gate="Q3_K", down="IQ4_XS", ntok=243, prompt=True, f16=True),
        # the LM head over a verified draft
        dict(name="lm head, 8 tokens", op="head", type="Q6_K", rows=VOCAB, ntok=8),
        # continuous batching, one token of each of 32 sequences, and a lone sequence: the smallest call
        dict(name="gated delta, 32 sequences", op="delta", seqs=32, rows=1, elem=4),
        dict(name="gated delta, 1 sequence", op="delta", seqs=1, rows=1, elem=4),
        # a prompt chunk
        dict(name="gated delta, 512 tokens", op="delta", seqs=1, rows=512, elem=4),
        # continuous batching over contexts of mixed length
        dict(attn, name="attention, 16 sequences", seqs=16, rows=1, ctx=8192),
        # the last chunk of a 2048-token prompt
        dict(attn, name="attention, 512 tokens", seqs=1, rows=512, ctx=2048),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["layers", "ffn", "ffn", "prompt", "prompt", "head", "delta", "attn"])
    if op == "layers":
        return dict(op="layers", ntok=rng.randint(2, 4), hidden=256 * rng.randint(8, 20))
    if op in ("ffn", "prompt"):
        gate, down = rng.choice(MIXES)
        hidden, ffn = 256 * rng.randint(4, 20), 256 * _log_int(rng, 8, 68)
        prompt = op == "prompt"
        return dict(op="ffn", gate=gate, down=down, hidden=hidden, ffn=ffn, prompt=prompt,
                    ntok=_log_int(rng, 9, 512) if prompt else _log_int(rng, 1, 16), f16=prompt and rng.random() < 0.4)
    if op == "head":
        return dict(op="head", type=rng.choice(["Q4_K", "Q5_K", "Q6_K", "Q8_0"]), rows=_log_int(rng, 32000, VOCAB),
                    ntok=rng.randint(1, 8))
    if op == "delta":
        rows = rng.choice([1, 1, rng.randint(2, 8), _log_int(rng, 9, 500)])
        return dict(op="delta", seqs=_log_int(rng, 1, 32 if rows == 1 else 4 if rows <= 8 else 1), rows=rows,
                    elem=rng.choice([4, 4, 2]))
    rows = rng.choice([1, 1, rng.randint(2, 8), _log_int(rng, 9, 500)])
    return dict(op="attn", seqs=_log_int(rng, 1, 16) if rows <= 8 else 1, rows=rows,
                ctx=_log_int(rng, max(128, rows + 1), 8192 if rows <= 8 else 2048), elem=rng.choice([2, 2, 2, 4]))


# ---- inputs ------------------------------------------------------------------------------------------------


def _gen(seed, tag):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1009 + tag)
    return g


def _randn(seed, tag, *shape):
    return torch.randn(*shape, device="cuda", generator=_gen(seed, tag))


def _weight(seed, tag, kind, rows, cols):
    """Random codes, grid indices, signs and sub-block scales, fp16 scales ~ |N(0, 1e-3)|; 256 bytes of padding."""
    _, bs, ts, fields = TYPES[kind]
    n, g = rows * cols // bs, _gen(seed, tag)
    buf = torch.zeros((n * ts + 256 + 7) // 8 * 8, dtype=torch.uint8, device="cuda")
    words = buf[: n * ts // 8 * 8].view(torch.int64)
    words.random_(-(2 ** 63), None, generator=g)
    blocks = buf[: n * ts].view(n, ts)
    for off in fields:
        d = torch.randn(n, device="cuda", generator=g).mul_(1e-3).abs_().half()
        blocks[:, off:off + 2] = d.view(torch.uint8).view(n, 2)
    return buf


def _matrices(case):
    """[(name, type, rows, cols, input)] of the case, in the order of the calls."""
    op = case["op"]
    if op == "ffn":
        h, f = case["hidden"], case["ffn"]
        return [("gate", case["gate"], f, h, "x"), ("up", case["gate"], f, h, "x"), ("down", case["down"], h, f, "h")]
    if op == "head":
        return [("head", case["type"], case["rows"], HIDDEN, "x")]
    hid, out = case.get("hidden", HIDDEN), []
    for layer in range(4):
        if layer == 3:
            mix = [("q", "Q5_K", 12288, hid, "in"), ("k", "Q6_K", 1024, hid, "in"), ("v", "Q6_K", 1024, hid, "in")]
        else:
            mix = [("qkv", "Q5_K", 10240, hid, "in"), ("z", "Q5_K", 6144, hid, "in"), ("beta", "Q8_0", 48, hid, "in"),
                   ("alpha", "Q8_0", 48, hid, "in")]
        mix += [("out", "Q6_K", hid, 6144, "core"), ("gate", "Q3_K", FFN, hid, "mlp"), ("up", "Q3_K", FFN, hid, "mlp"),
                ("down", "Q4_K", hid, FFN, "act")]
        out += [("%d.%s" % (layer, n), t, r, c, "%d.%s" % (layer, x)) for n, t, r, c, x in mix]
    return out


def _inputs(case, seed):
    """The case's plain inputs by name."""
    op = case["op"]
    if op in ("ffn", "head", "layers"):
        v = {}
        for k, (name, kind, rows, cols, x) in enumerate(_matrices(case)):
            v["w:" + name] = _weight(seed, 100 + k, kind, rows, cols)
            if x not in v:
                v[x] = _randn(seed, 500 + k, case["ntok"], cols)
                if x.endswith(("h", "act")):  # silu(gate) * up
                    v[x] = torch.nn.functional.silu(v[x]) * _randn(seed, 700 + k, case["ntok"], cols)
        return v
    n = case["seqs"] * case["rows"]
    if op == "delta":
        state = 0.1 * _randn(seed, 1, case["seqs"], VALUE_HEADS, KD, VD)
        return {"x": _randn(seed, 2, n, CONV), "conv": _randn(seed, 3, case["seqs"], CONV, TAPS),
                "w": 0.5 * _randn(seed, 4, CONV, TAPS), "b": _randn(seed, 5, n, VALUE_HEADS),
                "a": _randn(seed, 6, n, VALUE_HEADS),
                "ssm_a": -torch.rand(VALUE_HEADS, device="cuda", generator=_gen(seed, 7)) - 0.05,
                "dt": _randn(seed, 8, VALUE_HEADS), "z": _randn(seed, 9, n, VALUE_HEADS * VD),
                "norm": 1 + 0.1 * _randn(seed, 10, VD), "state": state if case["elem"] == 4 else state.half()}
    ctxs, pages = _contexts(case), _pages(case)
    dt = torch.float16 if case["elem"] == 2 else torch.float32
    pool = len(ctxs) * pages
    table_ = torch.randperm(pool, device="cuda", generator=_gen(seed, 6)).to(torch.int32)
    return {"raw": _randn(seed, 1, n, HEADS, 2 * HD), "k": _randn(seed, 2, n, KV_HEADS, HD),
            "v": _randn(seed, 3, n, KV_HEADS, HD), "kc": _randn(seed, 4, pool, KV_HEADS, PAGE, HD).to(dt),
            "vc": _randn(seed, 5, pool, KV_HEADS, PAGE, HD).to(dt), "pt": table_.view(torch.float32)}


def _contexts(case):
    """Positions each sequence holds after the pass: from a quarter of ctx to ctx."""
    n, c, r = case["seqs"], case["ctx"], case["rows"]
    return [max(r, c - (3 * c * i) // (4 * n)) for i in range(n)]


def _pages(case):
    return -(-max(_contexts(case)) // PAGE)


def prepare(case, seed):
    v, op = _inputs(case, seed), case["op"]
    rt = HipWeightRuntime()

    def buf(name, n, elem=4):
        rt.alloc(name, n, elem)
        if name in v:
            rt.buffer_tensor(name).copy_(v[name].reshape(-1))

    s = {"rt": rt, "case": case}
    if op in ("ffn", "head", "layers"):
        ntok, ms = case["ntok"], _matrices(case)
        for name, kind, rows, cols, x in ms:
            rt.upload_device(name, v["w:" + name], TYPES[kind][0], cols, rows)
            if x not in rt.buffers:
                buf(x, ntok * cols)
            buf("y:" + name, ntok * rows)
        if op == "ffn" and case["prompt"]:
            rt.set_gemm_min_rows(1)
            rt.set_gemm_f16_activations(case["f16"])
        s["out"] = {name: rt.buffer_tensor("y:" + name).view(ntok, rows) for name, _, rows, _, _ in ms}
        if op == "layers":
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                _layers(rt, case)
                side.synchronize()
                s["graph"] = torch.cuda.CUDAGraph()
                with torch.cuda.graph(s["graph"], stream=side):
                    _layers(rt, case)
            torch.cuda.current_stream().wait_stream(side)
        return s
    n = case["seqs"] * case["rows"]
    if op == "delta":
        for name in ("w", "ssm_a", "dt", "norm"):
            raw = torch.zeros(v[name].numel() * 4 + 256, dtype=torch.uint8, device="cuda")
            raw[: v[name].numel() * 4].view(torch.float32).copy_(v[name].reshape(-1))
            rt.upload_device(name, raw, 0, v[name].numel(), 1)
        for name in ("x", "conv", "b", "a", "z"):
            buf(name, v[name].numel())
        buf("state", v["state"].numel(), case["elem"])
        for name, size in (("u", n * CONV), ("o", n * VALUE_HEADS * VD), ("y", n * VALUE_HEADS * VD), ("none", 64)):
            rt.alloc(name, size)
        rt.set_paging("none", PAGE, max(1, -(-case["rows"] // PAGE)), case["seqs"])
        rt.set_segments([(i, 0, case["rows"]) for i in range(case["seqs"])])
        s["out"] = {"core": rt.buffer_tensor("o").view(n, VALUE_HEADS, VD), "y": rt.buffer_tensor("y").view(n, -1),
                    "conv": rt.buffer_tensor("conv"), "state": rt.buffer_tensor("state")}
        return s
    for name in ("raw", "k", "v", "pt"):
        buf(name, v[name].numel())
    for name in ("kc", "vc"):
        buf(name, v[name].numel(), case["elem"])
    for name in ("q", "g", "o", "y"):
        rt.alloc(name, n * HEADS * HD)
    rt.set_paging("pt", PAGE, _pages(case), case["seqs"])
    rt.set_segments([(i, c - case["rows"], case["rows"]) for i, c in enumerate(_contexts(case))])
    s["out"] = {"q": rt.buffer_tensor("q").view(n, HEADS, HD), "core": rt.buffer_tensor("o").view(n, HEADS, HD),
                "y": rt.buffer_tensor("y").view(n, HEADS, HD)}
    return s


# ---- one pass ----------------------------------------------------------------------------------------------


def _layers(rt, case):
    n = case["ntok"]
    for layer in range(4):
        p = "%d." % layer
        first = ["q", "k", "v"] if layer == 3 else ["qkv", "z", "beta", "alpha"]
        rt.qmv_group([p + k for k in first], p + "in", ["y:" + p + k for k in first], n)
        rt.qmv(p + "out", p + "core", "y:" + p + "out", n)
        rt.qmv_group([p + "gate", p + "up"], p + "mlp", ["y:" + p + "gate", "y:" + p + "up"], n)
        rt.qmv(p + "down", p + "act", "y:" + p + "down", n)


def run(state):
    rt, case = state["rt"], state["case"]
    op = case["op"]
    if op == "layers":
        state["graph"].replay()
    elif op == "ffn":
        rt.qmv_group(["gate", "up"], "x", ["y:gate", "y:up"], case["ntok"])
        rt.qmv("down", "h", "y:down", case["ntok"])
    elif op == "head":
        ids = rt.lmhead_argmax("head", "x", case["ntok"], logits="y:head")
        return {"ids": np.array(ids, np.int64), "logits": state["out"]["head"]}
    elif op == "delta":
        n = case["seqs"] * case["rows"]
        rt.conv_update_seg("x", "conv", "w", "u", CONV, TAPS)
        rt.gated_delta_seg("u", "b", "a", "ssm_a", "dt", "state", "o", KEY_HEADS, VALUE_HEADS, KD, VD, EPS, 1)
        rt.gated_rmsnorm("o", "norm", "z", "y", VD, EPS, n * VALUE_HEADS)
    else:
        n = case["seqs"] * case["rows"]
        rt.split_gated_q("raw", "q", "g", n * HEADS, HD)
        rt.rope_seg("q", HEADS, HD, ROT, ROPE_BASE)
        rt.kv_append_seg("k", "v", "kc", "vc", KV_HEADS, HD)
        rt.attention_seg("q", "kc", "vc", "o", HEADS, KV_HEADS, HD)
        rt.sigmoid_mul("o", "g", "y", n * HEADS * HD)
    return state["out"]


def work(case):
    op = case["op"]
    if op in ("ffn", "head", "layers"):
        n, seen, total, flops = case["ntok"], set(), 0, 0
        for _, kind, rows, cols, x in _matrices(case):
            _, bs, ts, _ = TYPES[kind]
            total += rows * cols // bs * ts + 4 * n * rows + (0 if x in seen else 4 * n * cols)
            flops += 2 * n * rows * cols
            seen.add(x)
        return {"bytes": total, "flops": flops}
    n = case["seqs"] * case["rows"]
    if op == "delta":
        state = 2 * case["seqs"] * (VALUE_HEADS * KD * VD * case["elem"] + CONV * TAPS * 4)
        # conv in and out, its weights, b and a, the core's output, z and y
        rows = n * (2 * CONV + 2 * VALUE_HEADS + 3 * VALUE_HEADS * VD) * 4 + CONV * TAPS * 4
        return {"bytes": state + rows, "flops": n * (VALUE_HEADS * KD * VD * 7 + CONV * 2 * TAPS)}
    pairs = sum(case["rows"] * (c - case["rows"]) + case["rows"] * (case["rows"] + 1) // 2 for c in _contexts(case))
    cache = sum(_contexts(case)) * 2 * KV_HEADS * HD * case["elem"]
    return {"bytes": cache + n * 4 * (2 * HEADS * HD + 4 * HEADS * HD + 2 * KV_HEADS * HD), "flops": 4 * pairs * HEADS * HD}


def tolerance(case):
    # fp32 sums over 32-bit partial results throughout; a gated-delta pass runs its sums through a recurrence, and an
    # fp16 state rounds once at the end of the pass
    if case["op"] == "delta":
        return {"rel": 2e-3, "max": 0.05} if case["elem"] == 2 else {"rel": 1e-5, "max": 1e-3}
    return {"rel": 1e-5, "max": 1e-3, "differ": 0.0}


# ---- the same in 64 bits -----------------------------------------------------------------------------------


def _table(name, width):
    return torch.tensor(list(table(name)), dtype=torch.float64, device="cuda").view(-1, width)


def _signs(bits):
    """+1 / -1 of the 8 bits of each value, [..., 8]."""
    k = torch.arange(8, device=bits.device)
    return 1.0 - 2.0 * ((bits[..., None] >> k) & 1)


def _signs7(i7):
    """ggml's 7 stored sign bits and their even-parity eighth."""
    k = torch.arange(7, device=i7.device)
    return _signs(i7 | (((i7[..., None] >> k) & 1).sum(-1) % 2) << 7)


def _nibbles(b):
    """[..., n] bytes -> low nibbles then high nibbles, [..., 2, n]."""
    return torch.stack([b & 15, b >> 4], -2)


_IQ4 = [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113]


def _dequant(kind, raw, rows, cols, f16=False):
    """float64 [rows, cols]; f16: Q6_K's integer product code * scale rounded to fp16, as that contraction takes it."""
    _, bs, ts, fields = TYPES[kind]
    b = raw[: rows * cols // bs * ts].view(-1, ts)
    f = [b[:, o:o + 2].contiguous().view(torch.float16).double() for o in fields]
    d, n = f[0], b.shape[0]
    b = b.to(torch.int64)

    def le(lo, width, count):
        """`count` little-endian words of `width` bytes from byte lo."""
        return sum(b[:, lo + i:lo + i + width * count:width] << (8 * i) for i in range(width))

    def pairs2(q, groups):  # 2-bit fields of 32-byte runs: [n, run, 32] -> [n, run * 4, 32]
        return torch.stack([(q >> (2 * k)) & 3 for k in range(4)], 2).reshape(n, groups, 32)

    if kind == "Q8_0":
        return (d * b[:, 2:].to(torch.uint8).view(torch.int8).double()).view(rows, cols)
    if kind in ("IQ4_NL", "IQ4_XS"):
        vals = torch.tensor(_IQ4, dtype=torch.float64, device=raw.device)
        if kind == "IQ4_NL":
            return (d * vals[_nibbles(b[:, 2:])].view(n, 32)).view(rows, cols)
        j = torch.arange(8, device=raw.device)
        ls = ((b[:, 4 + j // 2] >> (4 * (j % 2))) & 15) | (((le(2, 2, 1) >> (2 * j)) & 3) << 4)
        c = vals[_nibbles(b[:, 8:].view(n, 8, 16))].view(n, 8, 32)
        return (d[:, :, None] * (ls - 32)[:, :, None] * c).view(rows, cols)
    if kind in ("Q4_K", "Q5_K"):
        s = b[:, 4:16]
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        q = _nibbles(b[:, -128:].view(n, 4, 32)).view(n, 8, 32)
        if kind == "Q5_K":
            q = q | (((b[:, None, 16:48] >> torch.arange(8, device=raw.device)[:, None]) & 1) << 4)
        return ((d * sc)[:, :, None] * q - (f[1] * mn)[:, :, None]).view(rows, cols)
    if kind == "Q6_K":
        lo = b[:, :128].view(n, 2, 64)
        lo = torch.cat([lo & 15, lo >> 4], 2).view(n, 8, 32)
        hi = pairs2(b[:, 128:192].view(n, 2, 32), 8)
        sc = b[:, 192:208].to(torch.uint8).view(torch.int8).double()
        p = ((lo | (hi << 4)) - 32).view(n, 16, 16) * sc[:, :, None]
        return (d[:, :, None] * (p.half().double() if f16 else p)).view(rows, cols)
    if kind == "Q2_K":
        q = pairs2(b[:, 16:80].view(n, 2, 32), 8).view(n, 16, 16)
        return ((d * (b[:, :16] & 15))[:, :, None] * q - (f[1] * (b[:, :16] >> 4))[:, :, None]).view(rows, cols)
    if kind == "Q3_K":
        k, s = torch.arange(16, device=raw.device), b[:, 96:108]
        sc = ((s[:, k % 8] >> (4 * (k // 8))) & 15) | (((s[:, 8 + k % 4] >> (2 * (k // 4))) & 3) << 4)
        hb = (b[:, None, :32] >> torch.arange(8, device=raw.device)[:, None]) & 1
        q = (pairs2(b[:, 32:96].view(n, 2, 32), 8) | (hb << 2)) - 4
        return ((d * (sc - 32))[:, :, None] * q.view(n, 16, 16)).view(rows, cols)
    if kind == "IQ3_S":
        bit = (b[:, 66:74, None] >> torch.arange(8, device=raw.device)) & 1
        c = _table("iq3s_grid", 4)[b[:, 2:66].view(n, 8, 8) | (bit << 8)].view(n, 8, 32)
        sc = 1 + 2 * _nibbles(b[:, 106:110]).transpose(1, 2).reshape(n, 8)
        return ((d * sc)[:, :, None] * c * _signs(b[:, 74:106]).view(n, 8, 32)).view(rows, cols)
    l7 = 7 * torch.arange(4, device=raw.device)
    if kind == "IQ2_XXS":
        aux = le(2, 4, 16).view(n, 8, 2)
        c = _table("iq2xxs_grid", 8)[(aux[:, :, :1] >> (8 * torch.arange(4, device=raw.device))) & 255]
        sg, sc = _signs7((aux[:, :, 1:] >> l7) & 127), d * (0.5 + (aux[:, :, 1] >> 28)) * 0.25
        return (sc[:, :, None, None] * c * sg).view(rows, cols)
    if kind == "IQ3_XXS":
        aux = le(66, 4, 8)
        c = _table("iq3xxs_grid", 4)[b[:, 2:66]].view(n, 8, 4, 8)
        sg, sc = _signs7((aux[:, :, None] >> l7) & 127), d * (0.5 + (aux >> 28)) * 0.5
        return (sc[:, :, None, None] * c * sg).view(rows, cols)
    if kind == "IQ2_XS":
        q = le(2, 2, 32)
        c, sg, s = _table("iq2xs_grid", 8)[q & 511], _signs7(q >> 9), b[:, 66:74]
    else:  # IQ2_S
        hi = (b[:, 66:74, None] >> (2 * torch.arange(4, device=raw.device))) & 3
        c = _table("iq2s_grid", 8)[b[:, 2:34] | (hi.reshape(n, 32) << 8)]
        sg, s = _signs(b[:, 34:66]), b[:, 74:82]
    sc = d * (0.5 + _nibbles(s).transpose(1, 2).reshape(n, 16)) * 0.25
    return (sc[:, :, None] * (c * sg).view(n, 16, 16)).view(rows, cols)


def _activations(x, f16):
    """What the contraction is defined on: 8-bit codes times the scale of their 32, or x rounded to fp16."""
    if f16:  # each token scaled by a power of two into fp16's normal range
        s = torch.exp2(15 - torch.frexp(x.abs().amax(1, keepdim=True))[1].double())
        return (x * s.float()).half().double() / s
    g = x.view(x.shape[0], -1, 32)
    d = g.abs().amax(2, keepdim=True) / 127.0
    return (torch.round(g * torch.where(d > 0, 1.0 / d, 0.0)).double() * d.double()).view(x.shape)


F16X_TYPES = ("Q2_K", "Q3_K", "Q4_K", "Q5_K", "Q6_K", "IQ2_XXS", "IQ2_XS", "IQ2_S", "IQ3_XXS")


def _product(v, kind, name, rows, cols, x, f16):
    f16 = f16 and kind in F16X_TYPES  # the other types keep the 8-bit activations
    xv, out = _activations(v[x], f16), []
    _, bs, ts, _ = TYPES[kind]
    step = max(1, (96 << 20) // cols)
    for r0 in range(0, rows, step):
        n = min(step, rows - r0)
        w = _dequant(kind, v["w:" + name][r0 * cols // bs * ts:], n, cols, f16)
        out.append(xv @ w.T)
    return torch.cat(out, 1)


def exact(case, seed):
    v, op = _inputs(case, seed), case["op"]
    if op in ("ffn", "head", "layers"):
        f16 = op == "ffn" and case["f16"]
        out = {name: _product(v, kind, name, rows, cols, x, f16) for name, kind, rows, cols, x in _matrices(case)}
        return {"ids": None, "logits": out["head"]} if op == "head" else out
    f = {k: t.double() for k, t in v.items() if k != "pt"}
    n, r = case["seqs"], case["rows"]
    if op == "delta":
        x = f["x"].view(n, r, CONV)
        win = torch.cat([f["conv"][:, :, 1:].transpose(1, 2), x], 1)
        u = torch.nn.functional.silu(sum(win[:, k:k + r] * f["w"][:, k] for k in range(TAPS)))
        hk = torch.arange(VALUE_HEADS, device="cuda") % KEY_HEADS

        def unit(t):
            return t / torch.sqrt((t * t).sum(-1, keepdim=True) + EPS)

        q, k, w = u.split([KEY_HEADS * KD, KEY_HEADS * KD, VALUE_HEADS * VD], 2)
        q = unit(q.reshape(n, r, KEY_HEADS, KD))[:, :, hk] / math.sqrt(KD)
        k = unit(k.reshape(n, r, KEY_HEADS, KD))[:, :, hk]
        w = w.reshape(n, r, VALUE_HEADS, VD)
        beta = torch.sigmoid(f["b"]).view(n, r, VALUE_HEADS, 1)
        decay = torch.exp(f["ssm_a"] * torch.nn.functional.softplus(f["a"] + f["dt"])).view(n, r, VALUE_HEADS, 1, 1)
        S, core = f["state"].clone(), []
        for t in range(r):
            S = S * decay[:, t]
            S = S + k[:, t, :, :, None] * ((w[:, t] - (k[:, t, :, :, None] * S).sum(2)) * beta[:, t])[:, :, None, :]
            core.append((q[:, t, :, :, None] * S).sum(2))
        core = torch.stack(core, 1).view(n * r, VALUE_HEADS, VD)
        z = torch.nn.functional.silu(f["z"]).view(n * r, VALUE_HEADS, VD)
        y = core / torch.sqrt((core * core).mean(-1, keepdim=True) + EPS) * f["norm"] * z
        conv = win[:, r - 1:].transpose(1, 2).reshape(-1)
        return {"core": core, "y": y.view(n * r, -1), "conv": conv, "state": S.reshape(-1)}
    raw, ctxs, pages = f["raw"], _contexts(case), _pages(case)
    q, g = raw[..., :HD].clone(), raw[..., HD:]
    pt = v["pt"].view(torch.int32).view(n, pages).long()
    core = torch.empty(n * r, HEADS, HD, dtype=torch.float64, device="cuda")
    freq = ROPE_BASE ** (-2.0 * torch.arange(ROT // 2, dtype=torch.float64, device="cuda") / ROT)
    for i, c in enumerate(ctxs):
        rows = slice(i * r, (i + 1) * r)
        pos = torch.arange(c - r, c, device="cuda")
        ang = (pos.double()[:, None] * freq)[:, None]
        a, b = q[rows, :, :ROT // 2].clone(), q[rows, :, ROT // 2:ROT].clone()
        q[rows, :, :ROT // 2] = a * ang.cos() - b * ang.sin()
        q[rows, :, ROT // 2:ROT] = b * ang.cos() + a * ang.sin()
        cache = []
        for pool, new in (("kc", "k"), ("vc", "v")):
            t = f[pool][pt[i]].transpose(1, 2).reshape(pages * PAGE, KV_HEADS, HD)[:c].clone()
            t[c - r:] = v[new].view(n, r, KV_HEADS, HD)[i].to(v[pool].dtype).double()
            cache.append(t.transpose(0, 1))
        hide = torch.arange(c, device="cuda")[None, :] > pos[:, None]
        for h in range(HEADS):
            kh = h // (HEADS // KV_HEADS)
            p = (q[rows, h] @ cache[0][kh].T.contiguous() / math.sqrt(HD)).masked_fill(hide, -math.inf)
            core[rows, h] = torch.softmax(p, -1) @ cache[1][kh]
    return {"q": q, "core": core, "y": core * torch.sigmoid(g)}
