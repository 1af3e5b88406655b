"""Performance cases of the framework, over its public entry points (the Python package).

A user runs quantised Llama models: single-token decode, speculative verify passes of a few rows,
prompt prefill, temperature sampling, and the operators these are made of, called directly on
device tensors.  The cases cover the five matrix types that real GGUF files hold (Q4_0, Q4_K,
Q5_K, Q6_K, Q8_0), batches from one row to a prompt slice, contexts from a few positions to 8192,
and both attention orders.  Shapes are those of the package's own benchmark configurations
(``SYNTH_CONFIGS``: 1B, 3B, 8B and 70B widths) or generic.

Model cases run a few layers at full width with a small vocabulary (the full 128256-row head is a
case of its own), on a KV cache filled with N(0, 1) rows as the package's long-context benchmark does.
"""
import math
import struct

import numpy as np
import torch

import nanocamelid_amd as nc

TYPES = {"q4_0": nc.NC_TYPE_Q4_0, "q4_k": nc.NC_TYPE_Q4_K, "q5_k": nc.NC_TYPE_Q5_K, "q6_k": nc.NC_TYPE_Q6_K, "q8_0": nc.NC_TYPE_Q8_0}
BLOCK = {"q4_0": (32, 18), "q4_k": (256, 144), "q5_k": (256, 176), "q6_k": (256, 210), "q8_0": (32, 34)}
VOCAB = 8192
ORDER = {"sequential": 0, "split": 1}


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # RMSNorm + Q8_0 of one verify step's rows at the 8B width: twice per layer of every pass
        {"name": "norm_5x4096", "kind": "norm", "rows": 5, "width": 4096},
        # the smallest common matmul: attention output of an 8B layer in single-token decode
        {"name": "matmul_q4_0_1", "kind": "matmul", "type": "q4_0", "rows": 4096, "cols": 4096, "batch": 1},
        # one half of an 8B gate,up pair in a five-row verify pass
        {"name": "matmul_q4_0_5", "kind": "matmul", "type": "q4_0", "rows": 14336, "cols": 4096, "batch": 5},
        # the 3B Q4_K model's up projection in a five-row verify pass
        {"name": "matmul_q4_k_5", "kind": "matmul", "type": "q4_k", "rows": 8192, "cols": 3072, "batch": 5},
        # the down projection of an 8B Q8_0 file in a five-row verify pass
        {"name": "matmul_q8_0_5", "kind": "matmul", "type": "q8_0", "rows": 4096, "cols": 14336, "batch": 5},
        # the Q6_K output projection of most Q4_0 and Q4_K_M files, five verify rows
        {"name": "head_q6_k_5", "kind": "matmul", "type": "q6_k", "rows": 128256, "cols": 4096, "batch": 5},
        # a ragged prompt slice through a 3B Q4_K projection
        {"name": "prompt_q4_k_250", "kind": "matmul", "type": "q4_k", "rows": 8192, "cols": 3072, "batch": 250},
        # temperature softmax of a verify step's rows over the full vocabulary
        {"name": "temperature_5", "kind": "temperature", "rows": 5, "vocab": 128256, "temp": 0.8},
        # a five-row verify pass of an 8B model in the middle of a chat
        {"name": "verify_8b_700", "kind": "pass", "model": "llama-3-8b", "type": "q4_0", "layers": 4, "rows": 5, "pos": 700, "order": "sequential"},
        # one token of a 1B draft model at a long context
        {"name": "decode_1b_3500", "kind": "pass", "model": "llama-3.2-1b", "type": "q4_0", "layers": 4, "rows": 1, "pos": 3500, "order": "sequential"},
        # a nine-row verify pass of a 70B model over a full 8192-position cache
        {"name": "verify_70b_8192", "kind": "pass", "model": "llama-3-70b", "type": "q4_0", "layers": 1, "rows": 9, "pos": 8192, "order": "sequential"},
        # a long prompt into an 8B model
        {"name": "prefill_8b_2048", "kind": "prefill", "model": "llama-3-8b", "type": "q4_0", "layers": 2, "tokens": 2048},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["norm", "matmul", "matmul", "matmul", "matmul", "prompt", "temperature", "pass", "pass", "pass", "prefill"])
    if kind == "norm":
        return {"kind": "norm", "rows": _log_int(rng, 1, 256), "width": rng.choice([2048, 3072, 4096, 5120, 8192])}
    if kind in ("matmul", "prompt"):
        t = rng.choice(["q4_0", "q4_0", "q4_k", "q4_k", "q5_k", "q6_k", "q8_0"])
        batch = _log_int(rng, 1, 16) if kind == "matmul" else _log_int(rng, 17, 400)
        cols = max(1, _log_int(rng, 1024, 16384) // BLOCK[t][0]) * BLOCK[t][0]
        most = 128256 * 4096 if kind == "matmul" else 14336 * 4096
        rows = min(_log_int(rng, 512, 128256), most // cols)
        return {"kind": "matmul", "type": t, "rows": rows, "cols": cols, "batch": batch}
    if kind == "temperature":
        return {"kind": "temperature", "rows": rng.randint(1, 9), "vocab": _log_int(rng, 16000, 160000), "temp": round(rng.uniform(0.5, 1.3), 2)}
    model = rng.choice(["llama-3.2-1b", "llama-3.2-3b-q4k", "llama-3-8b"])
    t = "q4_k" if model == "llama-3.2-3b-q4k" else rng.choice(["q4_0", "q4_0", "q8_0"])
    if kind == "pass":
        return {"kind": "pass", "model": model, "type": t, "layers": rng.randint(2, 4), "rows": _log_int(rng, 1, 16), "pos": _log_int(rng, 16, 8000), "order": rng.choice(["sequential", "sequential", "split"])}
    # Q8_0 prompts stay short: a long one would cost more than the largest listed case
    return {"kind": "prefill", "model": model, "type": t, "layers": 2, "tokens": _log_int(rng, 24, 250 if t == "q8_0" else 2000)}


def tolerance(case):
    """About four times what the path is seen to be off the float64 results of exact()."""
    if case["kind"] == "norm":
        # the f32 scale is up to 7e-7 off; an int8 value flips where the scaled value is a tie to f32
        return {"rel": 3e-6, "differ": 1e-4}
    if case["kind"] == "matmul":
        return {"rel": 1.6e-6}  # f32 sums over the row's blocks: 4e-7
    if case["kind"] == "temperature":
        return {"rel": 8e-4, "max": 2e-3}  # the left-to-right f32 sum of 128256 terms: 2e-4
    # Whole passes: one flipped Q8_0 activation sets off more in every matmul that follows, up to the
    # noise of the quantisation itself: 0.01 to 0.04 off the float64 forward after one to four layers.
    return {"rel": 3e-2, "max": 1.5e-1, "differ": 1e-2}


# ---------------------------------------------------------------- GGUF blocks, both ways
def _half(x):
    return x.to(torch.float16).contiguous().view(torch.uint8).reshape(*x.shape, 2)


def _encode(t, x):
    """GGUF blocks [rows][units][bytes] (uint8) of float values [rows][cols] on their device."""
    unit = BLOCK[t][0]
    b = x.reshape(x.shape[0], -1, unit)
    if t == "q8_0":
        d = b.abs().amax(-1) / 127
        q = torch.round(b / d[..., None].clamp_min(1e-30)).to(torch.int8)
        return torch.cat([_half(d), q.view(torch.uint8)], -1)
    if t == "q4_0":
        d = b.gather(-1, b.abs().argmax(-1, keepdim=True))[..., 0] / -8
        q = torch.clamp(torch.floor(b / torch.where(d == 0, 1.0, d)[..., None] + 8.5), 0, 15).to(torch.uint8)
        return torch.cat([_half(d), q[..., :16] | (q[..., 16:] << 4)], -1)
    if t == "q6_k":
        g = b.reshape(*b.shape[:2], 16, 16)
        s = g.abs().amax(-1) / 31
        d = s.amax(-1) / 127
        sc = torch.round(s / d[..., None].clamp_min(1e-30)).clamp(1, 127)
        q = (torch.round(g / (d[..., None, None] * sc[..., None]).clamp_min(1e-30)).clamp(-32, 31) + 32).to(torch.uint8)
        q = q.reshape(*b.shape[:2], 2, 4, 32)  # half, 32-value group, value
        ql = ((q[..., :2, :] & 15) | ((q[..., 2:, :] & 15) << 4)).flatten(2)
        qh = ((q[..., 0, :] >> 4) | ((q[..., 1, :] >> 4) << 2) | ((q[..., 2, :] >> 4) << 4) | ((q[..., 3, :] >> 4) << 6)).flatten(2)
        return torch.cat([ql, qh, sc.to(torch.int8).view(torch.uint8), _half(d)], -1)
    top = 15 if t == "q4_k" else 31
    g = b.reshape(*b.shape[:2], 8, 32)
    m = (-g.amin(-1)).clamp_min(0)
    s = (g.amax(-1) + m) / top
    d, dm = s.amax(-1) / 63, m.amax(-1) / 63
    sc = torch.round(s / d[..., None].clamp_min(1e-30)).clamp(1, 63).to(torch.uint8)
    mn = torch.round(m / dm[..., None].clamp_min(1e-30)).clamp(0, 63).to(torch.uint8)
    q = torch.round((g + (dm[..., None] * mn)[..., None]) / (d[..., None] * sc)[..., None].clamp_min(1e-30)).clamp(0, top).to(torch.uint8)
    packed = torch.cat([sc[..., :4] | ((sc[..., 4:] >> 4) << 6), mn[..., :4] | ((mn[..., 4:] >> 4) << 6), (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)], -1)
    nib = ((q[..., 0::2, :] & 15) | ((q[..., 1::2, :] & 15) << 4)).flatten(2)
    parts = [_half(d), _half(dm), packed]
    if t == "q5_k":
        bit = (torch.arange(8, device=x.device, dtype=torch.uint8))[:, None]
        parts.append(((q >> 4) << bit).sum(-2, dtype=torch.uint8))
    return torch.cat(parts + [nib], -1)


def _decode(t, blocks):
    """float64 values [rows][cols] of GGUF blocks [rows][units][bytes]."""
    def half(at):
        return blocks[..., at:at + 2].contiguous().view(torch.float16)[..., 0].double()

    rows = blocks.shape[0]
    if t == "q8_0":
        return (half(0)[..., None] * blocks[..., 2:].contiguous().view(torch.int8).double()).reshape(rows, -1)
    if t == "q4_0":
        q = torch.cat([blocks[..., 2:] & 15, blocks[..., 2:] >> 4], -1).double() - 8
        return (half(0)[..., None] * q).reshape(rows, -1)
    if t == "q6_k":
        ql, qh = blocks[..., :128].reshape(rows, -1, 2, 64), blocks[..., 128:192].reshape(rows, -1, 2, 32)
        lo = [ql[..., :32] & 15, ql[..., 32:] & 15, ql[..., :32] >> 4, ql[..., 32:] >> 4]
        q = torch.stack([lo[k] | (((qh >> (2 * k)) & 3) << 4) for k in range(4)], -2).double() - 32
        sc = blocks[..., 192:208].contiguous().view(torch.int8).double() * half(208)[..., None]
        return (q.reshape(rows, -1, 16, 16) * sc[..., None]).reshape(rows, -1)
    s = blocks[..., 4:16]
    sc = torch.cat([s[..., :4] & 63, (s[..., 8:] & 15) | ((s[..., :4] >> 6) << 4)], -1).double() * half(0)[..., None]
    mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:] >> 4) | ((s[..., 4:8] >> 6) << 4)], -1).double() * half(2)[..., None]
    nib = blocks[..., -128:].reshape(rows, -1, 4, 1, 32)
    q = torch.cat([nib & 15, nib >> 4], -2).reshape(rows, -1, 8, 32)
    if t == "q5_k":
        bit = torch.arange(8, device=blocks.device, dtype=torch.uint8)[:, None]
        q = q | (((blocks[..., None, 16:48] >> bit) & 1) << 4)
    return (sc[..., None] * q.double() - mn[..., None]).reshape(rows, -1)


def _quantize(x):
    """Q8_0 activations: int8 [n][cols], scales [n][cols/32] in x's precision."""
    b = x.reshape(x.shape[0], -1, 32)
    s = b.abs().amax(-1) / 127
    v = b * torch.where(s > 0, 1 / s, torch.zeros_like(s))[..., None]
    q = torch.sign(v) * torch.floor(v.abs() + 0.5)
    return q.clamp(-127, 127).to(torch.int8).reshape(x.shape), s


# ---------------------------------------------------------------- what a program has in hand
_CONTEXT = []


def _context():
    if not _CONTEXT:
        _CONTEXT.append(nc.Context(torch.cuda.current_device()))
    return _CONTEXT[0]


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _matrix(case, seed):
    """The weights' GGUF blocks, N(0, 0.02) values, made in row slices on the GPU."""
    g, step = _generator(seed), max(1, (1 << 25) // case["cols"])
    parts = [_encode(case["type"], torch.randn(min(step, case["rows"] - r), case["cols"], device="cuda", generator=g) * 0.02) for r in range(0, case["rows"], step)]
    return torch.cat(parts)


def _inputs(case, seed):
    g = _generator(seed * 7 + 1)
    if case["kind"] == "norm":
        # residual-stream rows with a few large channels, weights around one
        x = torch.randn(case["rows"], case["width"], device="cuda", generator=g)
        x *= torch.exp(torch.randn(case["width"], device="cuda", generator=g) * 0.7)
        return x, 1 + 0.2 * torch.randn(case["width"], device="cuda", generator=g)
    if case["kind"] == "matmul":
        return _quantize(torch.randn(case["batch"], case["cols"], device="cuda", generator=g))
    return torch.randn(case["rows"], case["vocab"], device="cuda", generator=g) * 2.5


def _spec(case):
    return dict(nc.SYNTH_CONFIGS[case["model"]], layers=case["layers"], vocab_size=VOCAB, tied=0, weight_type=TYPES[case["type"]], context_length=8448)


_IMAGE, _MODEL = {}, {}


def _image(case):
    """The model file's bytes (random weights; the last shape asked for is kept, as a file would be)."""
    key = (case["model"], case["type"], case["layers"])
    if key not in _IMAGE:
        _IMAGE.clear()
        _IMAGE[key] = nc.synth_gguf(**_spec(case), seed=17)
    return _IMAGE[key]


def _model(case):
    """The loaded model, shared by the sessions of one program."""
    key = (case["model"], case["type"], case["layers"])
    if key not in _MODEL:
        _MODEL.clear()
        _MODEL[key] = nc.Model(_context(), data=_image(case))
    return _MODEL[key]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "norm":
        x, w = _inputs(case, seed)
        return {"case": case, "ctx": _context(), "x": x, "w": w}
    if kind == "matmul":
        q, s = _inputs(case, seed)
        w = nc.QMat(_context(), TYPES[case["type"]], case["rows"], case["cols"], _matrix(case, seed).cpu().numpy())
        return {"case": case, "ctx": _context(), "w": w, "q": q, "s": s}
    if kind == "temperature":
        return {"case": case, "ctx": _context(), "logits": _inputs(case, seed)}
    if kind == "pass":
        model = _model(case)
        s = nc.Session(model, case["pos"] + 64, 16)
        s.fill_kv(case["pos"], seed)
        model.ctx.set_attention(ORDER[case["order"]])
        return {"case": case, "session": s, "toks": nc.uniform_prompt(seed, case["rows"], VOCAB)}
    s = nc.Session(_model(case), case["tokens"] + 64, 16)
    s.model.ctx.set_attention(ORDER["sequential"])
    return {"case": case, "session": s, "toks": nc.uniform_prompt(seed, case["tokens"], VOCAB)}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "norm":
        return nc.rms_norm_q8_0_batch(state["ctx"], state["x"], state["w"], 1e-5)
    if kind == "matmul":
        return nc.matmul_quantized_batch(state["ctx"], state["w"], state["q"], state["s"])
    if kind == "temperature":
        return nc.temperature_probs_batch(state["ctx"], state["logits"], case["temp"])
    s = state["session"]
    if kind == "prefill":
        last = min(case["tokens"], 16)
        s.prefill_pass_batch(state["toks"], 0)
        return {"logits": s.logits(last - 1), "hidden": s.hidden(last)}
    if case["rows"] == 1:
        pred, logits = s.forward_pass(int(state["toks"][0]), case["pos"])
        return {"preds": pred, "logits": logits}
    accepted, token, _, preds = s.verify_greedy(state["toks"], case["pos"])
    # the row the decode loop goes on from, and the rows' hidden states
    return {"preds": preds.astype(np.int64), "accepted": accepted, "next": token, "logits": s.logits(accepted), "hidden": s.hidden(case["rows"])}


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    kind = case["kind"]
    if kind == "norm":
        n = case["rows"] * case["width"]
        return {"bytes": 4 * n + 4 * case["width"] + n + 4 * n // 32, "flops": 4 * n}
    if kind == "matmul":
        m, k, n = case["rows"], case["cols"], case["batch"]
        unit, size = BLOCK[case["type"]]
        return {"bytes": m * k // unit * size + n * k + 4 * n * k // 32 + 4 * n * m, "flops": 2 * m * k * n}
    if kind == "temperature":
        n = case["rows"] * case["vocab"]
        return {"bytes": 8 * n, "flops": 5 * n}
    spec = _spec(case)
    d, F, h, hkv = (spec[k] for k in ("embedding_length", "feed_forward_length", "head_count", "head_count_kv"))
    hd = d // h
    unit, size = BLOCK[case["type"]]
    weights = (2 * h + 2 * hkv) * hd * d + 3 * d * F
    n, pos = (case["rows"], case["pos"]) if kind == "pass" else (case["tokens"], 0)
    pairs = n * pos + n * (n + 1) // 2
    heads = n if kind == "pass" else 1
    kv = 2 * 4 * (pos + n) * hkv * hd
    return {
        "bytes": case["layers"] * (weights * size // unit + kv) + VOCAB * d * 18 // 32 + 4 * heads * VOCAB + 4 * n * d,
        "flops": case["layers"] * (2 * n * weights + 4 * pairs * h * hd) + 2 * heads * VOCAB * d,
    }


# ---------------------------------------------------------------- the results in 64 bits
class _File:
    """A GGUF image's tensors, read from its header."""

    def __init__(self, data):
        self.data, self.at, self.tensors = data, 8, {}
        count, keys = self._u64(), self._u64()
        for _ in range(keys):
            self._text()
            self._value(self._u32())
        found = []
        for _ in range(count):
            name = self._text()
            dims = [self._u64() for _ in range(self._u32())]
            found.append((name, dims, self._u32(), self._u64()))
        start = (self.at + 31) // 32 * 32
        for name, dims, kind, off in found:
            self.tensors[name] = (dims, kind, start + off)

    def _take(self, fmt):
        v = struct.unpack_from("<" + fmt, self.data, self.at)[0]
        self.at += struct.calcsize(fmt)
        return v

    def _u32(self):
        return self._take("I")

    def _u64(self):
        return self._take("Q")

    def _text(self):
        n = self._u64()
        self.at += n
        return bytes(self.data[self.at - n:self.at]).decode()

    def _value(self, kind):
        if kind == 8:
            return self._text()
        return self._take({4: "I", 6: "f"}[kind])

    def get(self, name):
        """float64 values on the GPU: [cols] of an f32 vector, [rows][cols] of a matrix."""
        dims, kind, off = self.tensors[name]
        n = math.prod(dims)
        if kind == 0:
            return torch.from_numpy(np.array(self.data[off:off + 4 * n])).view(torch.float32).cuda().double()
        t = next(k for k, v in TYPES.items() if v == kind)
        unit, size = BLOCK[t]
        raw = torch.from_numpy(np.array(self.data[off:off + n // unit * size])).cuda()
        return _decode(t, raw.reshape(dims[1], -1, size))


def _q8(x):
    q, s = _quantize(x)
    return (q.double().reshape(x.shape[0], -1, 32) * s[..., None]).reshape(x.shape)


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * w


def _exact_model(case, seed):
    spec = _spec(case)
    f = _File(_image(case))
    d, h, hkv = spec["embedding_length"], spec["head_count"], spec["head_count_kv"]
    hd = d // h
    kind, pos = case["kind"], case.get("pos", 0)
    n = case["rows"] if kind == "pass" else case["tokens"]
    toks = torch.from_numpy(nc.uniform_prompt(seed, n, VOCAB).astype(np.int64)).cuda()
    x = f.get("token_embd.weight")[toks]
    at = torch.arange(pos, pos + n, device="cuda").double()
    angle = at[:, None] * 500000.0 ** (-torch.arange(0, hd, 2, device="cuda").double() / hd)
    sin, cos = torch.sin(angle)[:, None], torch.cos(angle)[:, None]

    def rope(v):
        a, b = v[..., 0::2], v[..., 1::2]
        return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2)

    seen = torch.arange(pos + n, device="cuda")[None, :] <= torch.arange(pos, pos + n, device="cuda")[:, None]
    for layer in range(case["layers"]):
        b = "blk.%d." % layer
        y = _q8(_rms(x, f.get(b + "attn_norm.weight")))
        q = rope((y @ f.get(b + "attn_q.weight").T).reshape(n, h, hd))
        k = rope((y @ f.get(b + "attn_k.weight").T).reshape(n, hkv, hd))
        v = (y @ f.get(b + "attn_v.weight").T).reshape(n, hkv, hd)
        if pos:
            old = [torch.from_numpy(nc.synth_kv_values(seed, layer, e, 0, pos * hkv * hd)).cuda().double().reshape(pos, hkv, hd) for e in (0, 1)]
            k, v = torch.cat([old[0], k]), torch.cat([old[1], v])
        out = torch.empty(n, h, hd, device="cuda", dtype=torch.float64)
        for i in range(h):
            s = q[:, i] @ k[:, i * hkv // h].T / math.sqrt(hd)
            out[:, i] = torch.softmax(s.masked_fill(~seen, -math.inf), -1) @ v[:, i * hkv // h]
        x = x + _q8(out.reshape(n, -1)) @ f.get(b + "attn_output.weight").T
        y = _q8(_rms(x, f.get(b + "ffn_norm.weight")))
        gate = y @ f.get(b + "ffn_gate.weight").T
        x = x + _q8(gate * torch.sigmoid(gate) * (y @ f.get(b + "ffn_up.weight").T)) @ f.get(b + "ffn_down.weight").T
    head = f.get("output.weight")
    logits = _q8(_rms(x, f.get("output_norm.weight"))) @ head.T
    if kind == "prefill":
        return {"logits": logits[-1], "hidden": x[-min(n, 16):]}
    if n == 1:
        return {"preds": None, "logits": logits[0]}
    best = logits.argmax(-1).tolist()
    accepted = 0
    while accepted < n - 1 and best[accepted] == int(toks[accepted + 1]):
        accepted += 1
    return {"preds": None, "accepted": None, "next": None, "logits": logits[accepted], "hidden": x}


def exact(case, seed):
    kind = case["kind"]
    if kind == "norm":
        x, w = _inputs(case, seed)
        q, s = _quantize(_rms(x.double(), w.double()))
        return None, s
    if kind == "matmul":
        q, s = _inputs(case, seed)
        x = (q.double().reshape(q.shape[0], -1, 32) * s.double()[..., None]).reshape(q.shape)
        blocks = _matrix(case, seed)
        step = max(1, (1 << 27) // case["cols"])
        return torch.cat([x @ _decode(case["type"], blocks[r:r + step]).T for r in range(0, case["rows"], step)], 1)
    if kind == "temperature":
        return torch.softmax(_inputs(case, seed).double() / case["temp"], -1)
    return _exact_model(case, seed)
