"""Performance cases: the requests that a user of the token loop makes, at the model shapes and
weight formats that this repository's benchmark, synthetic models and tests name.

A case is one request on a model whose weights are on the GPU already:
  request   reset, a prompt, `gen` greedy tokens on the device, then one more token whose
            logits the caller takes (tf_hip_prefill, tf_hip_generate, tf_hip_decode)
  prompt    reset and a prompt whose last logits the caller takes (tf_hip_prefill)
  chat      reset, a prompt, then `gen` times tf_hip_sample at a temperature and a decode
  dropin    reset, a prompt, then `gen` decodes that copy their logits out, as Model::decode
            forwards them, the caller feeding back their first maximum
  attn      one decode attention over a cache on the device (tf_hip_attn_decode_noalloc)

Weights are N(0, 0.02) in the GGUF block formats, one set per (shape, format) as a user has one
model; the prompts, the draws and the attention's rows come from the seed. The output norm's
weights put the logits' deviation near 10, so that the next-token distribution is about as sharp
as a language model's: a few tokens hold most of it.
"""
import ctypes as C
import math

import numpy as np
import torch

from __graft_entry__ import load_package

DEV = "cuda"
F32, F16, Q4_0, Q4_1, Q8_0, Q6_K = 0, 1, 2, 3, 8, 14
BLOCK = {F32: (1, 4), F16: (1, 2), Q4_0: (32, 18), Q4_1: (32, 20), Q8_0: (32, 34), Q6_K: (256, 210)}

SHAPES = {
    # Llama-3.2-1B, Qwen2.5-0.5B and Qwen2.5-1.5B shapes
    "llama1b": dict(vocab=128256, d=2048, ff=8192, layers=16, heads=32, kv=8, theta=500000.0, eps=1e-5, bias=False),
    "qwen05b": dict(vocab=151936, d=896, ff=4864, layers=24, heads=14, kv=2, theta=1e6, eps=1e-6, bias=True),
    "qwen15b": dict(vocab=151936, d=1536, ff=8960, layers=28, heads=12, kv=2, theta=1e6, eps=1e-6, bias=True),
}
# the format mixes of each shape: mixq4 is Q4_0 layers, Q4_1 ffn_down in the first and last one, Q6_K embedding
FORMATS = {"llama1b": ("q8", "mixq4", "q6k", "f16"), "qwen05b": ("q8", "f16"), "qwen15b": ("q8", "f16")}

# kinds of layer slots (include/tf_hip.h): order of the 12 slots of a layer
L_NORM, L_Q, L_K, L_V, L_O, L_BQ, L_BK, L_BV, L_FNORM, L_GATE, L_UP, L_DOWN = range(12)


def listed():
    return [
        # Time to first token of a short question: six tokens, the shortest prompt in the benchmark.
        dict(name="prompt_llama1b_q8_6", kind="prompt", shape="llama1b", fmt="q8", prompt=6, max_seq=512, layout=0),
        # A page of context at an ordinary size: the benchmark's prefill-heavy prompt.
        dict(name="prompt_llama1b_q8_512", kind="prompt", shape="llama1b", fmt="q8", prompt=512, max_seq=1024, layout=0),
        # The headline: a short question answered greedily, decode-bound.
        dict(name="request_llama1b_q8_6", kind="request", shape="llama1b", fmt="q8", prompt=6, gen=31, max_seq=512,
             layout=0),
        # A sampled chat answer: temperature and nucleus over the whole vocabulary after every token.
        dict(name="chat_llama1b_q8_70", kind="chat", shape="llama1b", fmt="q8", prompt=70, gen=16, max_seq=2048,
             layout=0, temperature=0.8, top_p=0.95),
        # The 4-bit model's answer, and a ragged prompt on it.
        dict(name="request_llama1b_mixq4_6", kind="request", shape="llama1b", fmt="mixq4", prompt=6, gen=31, max_seq=512,
             layout=0),
        dict(name="prompt_llama1b_mixq4_333", kind="prompt", shape="llama1b", fmt="mixq4", prompt=333, max_seq=512,
             layout=0),
        # A 6-bit model's paragraph-long prompt.
        dict(name="prompt_llama1b_q6k_129", kind="prompt", shape="llama1b", fmt="q6k", prompt=129, max_seq=512, layout=1),
        # The small model with biases: a question of a sentence, a longer answer.
        dict(name="request_qwen05b_q8_16", kind="request", shape="qwen05b", fmt="q8", prompt=16, gen=63, max_seq=512,
             layout=0),
        # The unquantized small model behind Model::decode, logits on the host after every token.
        dict(name="dropin_qwen05b_f16_40", kind="dropin", shape="qwen05b", fmt="f16", prompt=40, gen=12, max_seq=1024,
             layout=0),
        # Long context: a ragged prompt of several thousand tokens, and decode over 4096 cached positions.
        dict(name="prompt_qwen15b_q8_2900", kind="prompt", shape="qwen15b", fmt="q8", prompt=2900, max_seq=8192, layout=1),
        dict(name="request_qwen15b_q8_4096", kind="request", shape="qwen15b", fmt="q8", prompt=4096, gen=63, max_seq=8192,
             layout=1),
        # One layer's decode attention in a serving loop with its own cache.
        dict(name="attn_32x64_1000", kind="attn", heads=32, kv=8, hd=64, n_pos=1000, max_seq=4096, layout=0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("prompt", "prompt", "prompt", "request", "request", "chat", "dropin", "attn"))
    layout = rng.choice((0, 1))
    if kind == "attn":
        heads, kv, hd = rng.choice(((32, 8, 64), (14, 2, 64), (12, 2, 128)))
        max_seq = rng.choice((512, 2048, 4096, 8192))
        return dict(kind=kind, heads=heads, kv=kv, hd=hd, n_pos=min(max_seq, _log_int(rng, 1, max_seq)), max_seq=max_seq,
                    layout=layout)
    shape = rng.choice(sorted(SHAPES))
    fmt = rng.choice(FORMATS[shape])
    # prompts over the whole range; the slower formats' and the per-token calls' ones are shorter
    top = {"prompt": 4096, "request": 2048, "chat": 512, "dropin": 512}[kind]
    prompt = _log_int(rng, 2, top if fmt in ("q8", "mixq4") else min(top, 512))
    gen = 0 if kind == "prompt" else rng.randint(4, 32 if kind == "request" else 12)
    need = prompt + gen + 1
    max_seq = rng.choice([m for m in (512, 1024, 2048, 4096, 8192) if m >= need][:3])
    c = dict(kind=kind, shape=shape, fmt=fmt, prompt=prompt, max_seq=max_seq, layout=layout)
    if kind != "prompt":
        c["gen"] = gen
    if kind == "chat":
        c["temperature"] = rng.choice((0.6, 0.8, 1.0))
        c["top_p"] = rng.choice((0.9, 0.95, 1.0))
    return c


# ---------------------------------------------------------------- weights in the GGUF block formats

def _f16_bytes(x):
    return x.half().contiguous().view(torch.uint8)


def _quantize(t, w):
    """w [n][k] float32 -> GGUF row bytes [n][row bytes] (uint8)."""
    n, k = w.shape
    if t == F32:
        return w.contiguous().view(torch.uint8)
    if t == F16:
        return w.half().contiguous().view(torch.uint8)
    if t == Q6_K:  # 16 sub-blocks of 16 with int8 scales, element e = 128 h + 32 j + l
        b = w.view(n, k // 256, 16, 16)
        sub = b.abs().amax(3) / 31.0
        d = (sub.amax(2, keepdim=True) / 127.0).half().float()
        sc = (sub / d.clamp_min(1e-20)).round().clamp(1, 127)
        q = (b / (d * sc).clamp_min(1e-20)[..., None]).round().clamp(-32, 31).to(torch.int32).view(n, -1, 2, 4, 32) + 32
        lo = torch.cat((q[:, :, :, 0] & 15 | (q[:, :, :, 2] & 15) << 4, q[:, :, :, 1] & 15 | (q[:, :, :, 3] & 15) << 4), 3)
        hi = (q[:, :, :, 0] >> 4) | (q[:, :, :, 1] >> 4) << 2 | (q[:, :, :, 2] >> 4) << 4 | (q[:, :, :, 3] >> 4) << 6
        return torch.cat((lo.to(torch.uint8).reshape(n, -1, 128), hi.to(torch.uint8).reshape(n, -1, 64),
                          sc.to(torch.int8).view(torch.uint8), _f16_bytes(d)), 2).reshape(n, -1)
    b = w.view(n, k // 32, 32)
    if t == Q8_0:
        d = (b.abs().amax(2, keepdim=True) / 127.0).half()
        q = (b / d.float().clamp_min(1e-20)).round().clamp(-127, 127).to(torch.int8).view(torch.uint8)
        return torch.cat((_f16_bytes(d), q), 2).reshape(n, -1)
    if t == Q4_0:
        d = (b.abs().amax(2, keepdim=True) / 8.0).half()
        head, q = _f16_bytes(d), (b / d.float().clamp_min(1e-20)).round().clamp(-8, 7).to(torch.int32) + 8
    else:  # Q4_1
        m = b.amin(2, keepdim=True).half()
        d = ((b.amax(2, keepdim=True) - m.float()) / 15.0).half()
        head = torch.cat((_f16_bytes(d), _f16_bytes(m)), 2)
        q = ((b - m.float()) / d.float().clamp_min(1e-20)).round().clamp(0, 15).to(torch.int32)
    return torch.cat((head, (q[:, :, :16] | q[:, :, 16:] << 4).to(torch.uint8)), 2).reshape(n, -1)


def _dequantize(t, raw, n, k):
    """GGUF row bytes on the GPU -> [n][k] float64."""
    if t == F32:
        return raw.view(torch.float32).view(n, k).double()
    if t == F16:
        return raw.view(torch.float16).view(n, k).double()
    b = raw.view(n, k // BLOCK[t][0], BLOCK[t][1])
    if t == Q6_K:
        ql, qh = b[:, :, :128].reshape(n, -1, 2, 64).to(torch.int16), b[:, :, 128:192].reshape(n, -1, 2, 32).to(torch.int16)
        sc = b[:, :, 192:208].contiguous().view(torch.int8).double()
        d = b[:, :, 208:210].contiguous().view(torch.float16).double()
        lo = torch.stack((ql[..., :32] & 15, ql[..., 32:] & 15, ql[..., :32] >> 4, ql[..., 32:] >> 4), 3)
        hi = torch.stack((qh & 3, qh >> 2 & 3, qh >> 4 & 3, qh >> 6 & 3), 3)
        q = (lo | hi << 4).double() - 32.0
        return (q.reshape(n, -1, 16, 16) * (sc * d)[..., None]).reshape(n, k)
    d = b[:, :, :2].contiguous().view(torch.float16).double()
    if t == Q8_0:
        return (b[:, :, 2:].contiguous().view(torch.int8).double() * d).reshape(n, k)
    h = 4 if t == Q4_1 else 2
    q = torch.cat((b[:, :, h:] & 15, b[:, :, h:] >> 4), 2).double()
    if t == Q4_0:
        return ((q - 8.0) * d).reshape(n, k)
    return (q * d + b[:, :, 2:4].contiguous().view(torch.float16).double()).reshape(n, k)


def _types(fmt, layer, layers, kind):
    if fmt == "mixq4":
        return Q4_1 if kind == L_DOWN and layer in (0, layers - 1) else Q4_0
    return {"q8": Q8_0, "q6k": Q6_K, "f16": F16}[fmt]


def _slot(layer, kind):
    return 16 + 12 * layer + kind


def _plan(shape, fmt):
    """(slot, type, row length, rows) of every matrix."""
    s = SHAPES[shape]
    hd = s["d"] // s["heads"]
    out = [(0, Q6_K if fmt == "mixq4" else _types(fmt, 0, s["layers"], L_Q), s["d"], s["vocab"])]
    dims = {L_Q: (s["d"], s["d"]), L_K: (s["d"], s["kv"] * hd), L_V: (s["d"], s["kv"] * hd), L_O: (s["d"], s["d"]),
            L_GATE: (s["d"], s["ff"]), L_UP: (s["d"], s["ff"]), L_DOWN: (s["ff"], s["d"])}
    for layer in range(s["layers"]):
        out += [(_slot(layer, k), _types(fmt, layer, s["layers"], k)) + dims[k] for k in dims]
    return out


_held = {}  # the last model's GGUF bytes on the host: what a program reads from its file


def _model(shape, fmt):
    if (shape, fmt) not in _held:
        _held.clear()
        s = SHAPES[shape]
        hd = s["d"] // s["heads"]
        g = torch.Generator(device=DEV).manual_seed(sum(map(ord, shape + fmt)))
        mats = []
        for slot, t, k, n in _plan(shape, fmt):
            raw = torch.cat([_quantize(t, 0.02 * torch.randn(min(16384, n - r), k, generator=g, device=DEV))
                             for r in range(0, n, 16384)])
            mats.append((slot, t, k, n, raw.cpu().numpy().reshape(-1)))
        vecs = []

        def vec(slot, n, mean, sigma):
            vecs.append((slot, (mean + sigma * torch.randn(n, generator=g, device=DEV)).cpu().numpy()))

        peak = 10.0 / (0.02 * math.sqrt(s["d"]))
        vec(1, s["d"], peak, 0.1 * peak)
        for layer in range(s["layers"]):
            vec(_slot(layer, L_NORM), s["d"], 1.0, 0.1)
            vec(_slot(layer, L_FNORM), s["d"], 1.0, 0.1)
            if s["bias"]:
                vec(_slot(layer, L_BQ), s["d"], 0.0, 0.01)
                vec(_slot(layer, L_BK), s["kv"] * hd, 0.0, 0.01)
                vec(_slot(layer, L_BV), s["kv"] * hd, 0.0, 0.01)
        _held[shape, fmt] = (mats, vecs)
    return _held[shape, fmt]


def _rope(shape, n):
    s = SHAPES[shape]
    hd = s["d"] // s["heads"]
    freq = (s["theta"] ** (-np.arange(0, hd, 2, dtype=np.float64) / hd)).astype(np.float32)
    ang = np.arange(n, dtype=np.float32)[:, None] * freq[None]
    return np.ascontiguousarray(np.cos(ang)), np.ascontiguousarray(np.sin(ang))


# ---------------------------------------------------------------- a program's side of the C ABI

def _ip(a):
    return a.ctypes.data_as(C.POINTER(C.c_int32))


def _fp(a):
    return None if a is None else a.ctypes.data_as(C.POINTER(C.c_float))


class Session:
    """One context of the C ABI with a model's weights on the GPU."""

    def __init__(self, shape, fmt, max_seq, layout):
        pkg = load_package()
        self.L, s = pkg.hip_lib(), SHAPES[shape]
        self.vocab = s["vocab"]
        hp = pkg.HParams(s["vocab"], s["d"], s["ff"], s["layers"], s["heads"], s["kv"], s["d"] // s["heads"], max_seq,
                         layout, s["eps"])
        self.h = C.c_void_p()
        self.ok(self.L.tf_hip_create(0, C.cast(C.byref(hp), C.c_void_p), C.byref(self.h)))
        mats, vecs = _model(shape, fmt)
        for slot, t, k, n, raw in mats:
            self.ok(self.L.tf_hip_upload_tensor(self.h, slot, t, k, n, raw.ctypes.data, raw.nbytes))
        for slot, v in vecs:
            self.ok(self.L.tf_hip_upload_tensor(self.h, slot, F32, len(v), 1, v.ctypes.data, v.nbytes))
        cos, sin = _rope(shape, max_seq)
        self.ok(self.L.tf_hip_set_rope_table(self.h, _fp(cos), _fp(sin), max_seq, cos.shape[1]))
        self.logits = np.zeros(s["vocab"], np.float32)
        self.am = C.c_int32(-1)

    def ok(self, rc):
        if rc != 0:
            raise RuntimeError("status %d: %s" % (rc, self.L.tf_hip_last_error(self.h).decode()))

    def __del__(self):
        if getattr(self, "h", None):
            self.L.tf_hip_destroy(self.h)
            self.h = None

    def reset(self):
        self.ok(self.L.tf_hip_reset(self.h))

    def prefill(self, tokens, logits=None):
        self.ok(self.L.tf_hip_prefill(self.h, _ip(tokens), len(tokens), _fp(logits), C.byref(self.am)))
        return self.am.value

    def decode(self, token, logits=None):
        self.ok(self.L.tf_hip_decode(self.h, int(token), _fp(logits), C.byref(self.am)))
        return self.am.value

    def generate(self, n):
        out = np.zeros(n, np.int32)
        self.ok(self.L.tf_hip_generate(self.h, n, _ip(out)))
        return out

    def sample(self, temperature, top_p, r):
        tok = np.zeros(1, np.int32)
        self.ok(self.L.tf_hip_sample(self.h, temperature, top_p, r, _ip(tok)))
        return int(tok[0])


def _inputs(case, seed):
    r = np.random.RandomState(seed % (1 << 31))
    tokens = r.randint(0, SHAPES[case["shape"]]["vocab"], case["prompt"] + 1).astype(np.int32)
    return tokens[:-1].copy(), int(tokens[-1]), r.random_sample(case.get("gen", 0)).astype(np.float32)


def _attn_inputs(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    q = torch.randn(case["heads"], case["hd"], generator=g, device=DEV)
    k = torch.randn(case["n_pos"], case["kv"], case["hd"], generator=g, device=DEV)
    v = torch.randn(case["n_pos"], case["kv"], case["hd"], generator=g, device=DEV)
    return q, k, v


def prepare(case, seed):
    if case["kind"] == "attn":
        q, k, v = _attn_inputs(case, seed)
        rows = (case["max_seq"], case["kv"], case["hd"])
        caches = []
        for x in (k, v):
            c = torch.zeros(rows, device=DEV)
            c[: case["n_pos"]] = x
            caches.append(c if case["layout"] == 0 else c.transpose(0, 1).contiguous())
        lib = load_package().hip_lib()
        return dict(case=case, lib=lib, q=q, k=caches[0], v=caches[1], out=torch.empty_like(q))
    tokens, extra, draws = _inputs(case, seed)
    session = Session(case["shape"], case["fmt"], case["max_seq"], case["layout"])
    return dict(case=case, m=session, tokens=tokens, extra=extra, draws=draws)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "attn":
        rc = state["lib"].tf_hip_attn_decode_noalloc(
            0, state["q"].data_ptr(), state["k"].data_ptr(), state["v"].data_ptr(), case["heads"], case["kv"], case["hd"],
            case["n_pos"], case["max_seq"], case["layout"], state["out"].data_ptr(), torch.cuda.current_stream().cuda_stream)
        if rc != 0:
            raise RuntimeError("tf_hip_attn_decode_noalloc: status %d" % rc)
        return state["out"]
    m = state["m"]
    m.reset()
    if kind == "prompt":
        logits = np.empty(m.vocab, np.float32)
        return {"next": m.prefill(state["tokens"], logits), "logits": logits}
    first = m.prefill(state["tokens"])
    if kind == "request":
        tokens = m.generate(case["gen"])
        logits = np.empty(m.vocab, np.float32)
        return {"tokens": tokens, "next": m.decode(state["extra"], logits), "logits": logits}
    if kind == "chat":
        tokens = []
        for r in state["draws"]:
            tokens.append(m.sample(case["temperature"], case["top_p"], float(r)))
            m.decode(tokens[-1])
        logits = np.empty(m.vocab, np.float32)
        return {"tokens": np.array(tokens, np.int32), "next": m.decode(state["extra"], logits), "logits": logits}
    tokens, rows, token = [], [], first
    for _ in range(case["gen"]):
        logits = np.empty(m.vocab, np.float32)
        tokens.append(token)
        token = m.decode(token, logits)
        rows.append(logits)
    return {"tokens": np.array(tokens, np.int32), "logits": rows}


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    if case["kind"] == "attn":
        kv = 2 * case["n_pos"] * case["kv"] * case["hd"] * 4
        return {"bytes": kv + 2 * case["heads"] * case["hd"] * 4, "flops": 4 * case["n_pos"] * case["heads"] * case["hd"]}
    s = SHAPES[case["shape"]]
    hd = s["d"] // s["heads"]
    plan = _plan(case["shape"], case["fmt"])
    nbytes = [n * (k // BLOCK[t][0]) * BLOCK[t][1] for _, t, k, n in plan]
    weights, head = sum(nbytes), plan[0][2] * plan[0][3]
    per_row = sum(k * n for _, _, k, n in plan[1:])
    kv_row = 2 * 4 * s["layers"] * s["kv"] * hd
    p = case["prompt"]
    # the prompt: every weight once, its K and V rows written, the next token's logits
    b = weights + p * kv_row + 4 * s["vocab"]
    f = 2 * (p * per_row + head) + 2 * p * (p + 1) * s["heads"] * hd * s["layers"]
    for i in range(case.get("gen", 0) + (case["kind"] in ("request", "chat"))):
        n_pos = p + i + 1
        b += weights + n_pos * kv_row
        f += 2 * (per_row + head) + 4 * n_pos * s["heads"] * hd * s["layers"]
        if case["kind"] == "dropin":
            b += 4 * s["vocab"]
    return {"bytes": b, "flops": f}


def tolerance(case):
    # fp32 sums in another order, measured against 64 bits over these ranges, times about four
    if case["kind"] == "attn":
        return {"rel": 1e-6, "max": 1e-5}
    return {"rel": 1.5e-5, "max": 1e-4, "differ": 0.0}


# ---------------------------------------------------------------- the same in 64 bits

class Exact:
    def __init__(self, case):
        self.s = s = SHAPES[case["shape"]]
        mats, vecs = _model(case["shape"], case["fmt"])
        self.w = {slot: _dequantize(t, torch.from_numpy(raw).to(DEV), n, k) for slot, t, k, n, raw in mats}
        self.v = {slot: torch.from_numpy(v).to(DEV).double() for slot, v in vecs}
        cos, sin = _rope(case["shape"], case["max_seq"])
        self.cos, self.sin = torch.from_numpy(cos).to(DEV).double(), torch.from_numpy(sin).to(DEV).double()
        self.hd = s["d"] // s["heads"]
        self.kc = [None] * s["layers"]
        self.vc = [None] * s["layers"]
        self.pos = 0

    def norm(self, x, slot):
        return x / (x.square().mean(-1, keepdim=True) + np.float32(self.s["eps"])).sqrt() * self.v[slot]

    def rope(self, x):
        c = self.cos[self.pos: self.pos + len(x), None]
        s = self.sin[self.pos: self.pos + len(x), None]
        a, b = x.chunk(2, -1)
        return torch.cat((a * c - b * s, a * s + b * c), -1)

    def attend(self, q, k, v):
        """Causal: the last query sees every key. q [n][heads][hd], k and v [m][kv][hd]."""
        n, m, rep = len(q), len(k), self.s["heads"] // self.s["kv"]
        out = torch.empty_like(q)
        for h in range(self.s["heads"]):
            kh, vh = k[:, h // rep].contiguous(), v[:, h // rep].contiguous()
            for r in range(0, n, 1024):
                sc = q[r: r + 1024, h].contiguous() @ kh.T.contiguous() / math.sqrt(self.hd)
                last = torch.arange(m - n + r, m - n + min(n, r + 1024), device=DEV)
                sc.masked_fill_(torch.arange(m, device=DEV)[None] > last[:, None], -math.inf)
                out[r: r + 1024, h] = sc.softmax(-1) @ vh
        return out

    def __call__(self, tokens):
        """The last token's logits, float64 [vocab]."""
        s, x = self.s, self.w[0][torch.as_tensor(np.asarray(tokens, np.int64), device=DEV)]
        n = len(x)
        for layer in range(s["layers"]):
            w, b = (lambda k: self.w[_slot(layer, k)].T), (lambda k: self.v.get(_slot(layer, k), 0.0))
            y = self.norm(x, _slot(layer, L_NORM))
            q = (y @ w(L_Q) + b(L_BQ)).view(n, s["heads"], self.hd)
            k = (y @ w(L_K) + b(L_BK)).view(n, s["kv"], self.hd)
            v = (y @ w(L_V) + b(L_BV)).view(n, s["kv"], self.hd)
            q, k = self.rope(q), self.rope(k)
            if self.pos:
                k, v = torch.cat((self.kc[layer], k)), torch.cat((self.vc[layer], v))
            self.kc[layer], self.vc[layer] = k, v
            x = x + self.attend(q, k, v).view(n, -1) @ w(L_O)
            y = self.norm(x, _slot(layer, L_FNORM))
            g = y @ w(L_GATE)
            x = x + (g / (1.0 + torch.exp(-g)) * (y @ w(L_UP))) @ w(L_DOWN)
        self.pos += n
        return self.w[0] @ self.norm(x[-1], 1)


def _sample(logits, temperature, top_p, r):
    p, order = (logits / temperature).softmax(0).sort(descending=True, stable=True)
    c = p.cumsum(0)
    last = int((c < top_p).sum()) + 1 if top_p < 1.0 else len(p)
    last = min(last, len(p))
    c = c[:last] / c[last - 1]
    return int(order[min(int((c < r).sum()), last - 1)])


@torch.no_grad()
def exact(case, seed):
    if case["kind"] == "attn":
        q, k, v = (x.double() for x in _attn_inputs(case, seed))
        rep = case["heads"] // case["kv"]
        out = torch.empty_like(q)
        for h in range(case["heads"]):
            p = (k[:, h // rep] @ q[h] / math.sqrt(case["hd"])).softmax(0)
            out[h] = p @ v[:, h // rep]
        return out
    tokens, extra, draws = _inputs(case, seed)
    m = Exact(case)
    logits = m(tokens)
    if case["kind"] == "prompt":
        return {"next": int(logits.argmax()), "logits": logits}
    out, rows = [], []
    for i in range(case["gen"]):
        out.append(_sample(logits, case["temperature"], case["top_p"], float(draws[i])) if case["kind"] == "chat"
                   else int(logits.argmax()))
        logits = m([out[-1]])
        rows.append(logits)
    out = np.array(out, np.int32)
    if case["kind"] == "dropin":
        return {"tokens": out, "logits": rows}
    logits = m([extra])
    return {"tokens": out, "next": int(logits.argmax()), "logits": logits}
