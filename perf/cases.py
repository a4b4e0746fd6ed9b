"""The work that a user of this framework has it do, as a list of timed cases.

A chat session is a prompt (``PagedEngine.forward`` in chunks of the performance mode's batch)
and a reply (``PagedEngine.decode``), over every weight mix and K/V ring type that the loader
takes in earnest; a host that drives single ops calls ``Compute``. The cases below cover both,
from the smallest call to the largest, at the widths of the repository's own model shapes.
Models keep those widths and vocabularies with fewer layers where the file would be large:
the layers of a decoder are alike, so four of them stand for thirty-two.

Weights are random blocks with the statistics of ``webgpu_amd.synth``, drawn on the GPU from the
seed. ``exact`` restates the same computation in float64 with plain torch.
"""
import dataclasses
import math
import struct

import numpy as np
import torch

from webgpu_amd import synth
from webgpu_amd.engine import LoadOptions, PagedEngine
from webgpu_amd.gpu import Compute

F32, F16, Q4_0, Q8_0, Q4_K, Q5_K, Q6_K = 0, 1, 2, 8, 12, 13, 14
BLOCK = {F32: (1, 4), F16: (1, 2), Q4_0: (32, 18), Q8_0: (32, 34), Q4_K: (256, 144), Q5_K: (256, 176), Q6_K: (256, 210)}
TYPES = {"f16": F16, "q4_0": Q4_0, "q8_0": Q8_0, "q4_k": Q4_K, "q5_k": Q5_K, "q6_k": Q6_K}
# the weight types of whole files, by role
MIXES = {
    "q4_k_m": None,  # the mix of the synthetic shapes
    "q5_k_m": {"embd": Q5_K, "output": Q6_K, "attn": Q5_K, "v": Q6_K, "ffn": Q5_K},
    "q8_0": {"embd": Q8_0, "output": Q8_0, "attn": Q8_0, "v": Q8_0, "ffn": Q8_0},
}


# ------------------------------------------------------------------------------- the cases

def listed():
    return [
        # a reply of the small model in a default session, shortly after a short prompt: every
        # launch is small, so the fixed cost of a step counts
        {"name": "reply_0.6b", "kind": "reply", "model": "qwen3-0.6b", "layers": 28, "mix": "q4_k_m", "kv": "f32",
         "batch": 16, "start": 64, "tokens": 16},
        # a reply deep in a long conversation with half-precision rings
        {"name": "reply_8b_long", "kind": "reply", "model": "llama3-8b", "layers": 4, "mix": "q4_k_m", "kv": "f16",
         "batch": 128, "start": 4000, "tokens": 24},
        # a first prompt in the default performance mode (batches of 16)
        {"name": "prompt_8b_default", "kind": "prompt", "model": "llama3-8b", "layers": 4, "mix": "q4_k_m", "kv": "f32",
         "batch": 16, "start": 0, "tokens": 250},
        # a short prompt in the lite mode (batches of 8)
        {"name": "prompt_0.6b_lite", "kind": "prompt", "model": "qwen3-0.6b", "layers": 28, "mix": "q4_k_m", "kv": "f32",
         "batch": 8, "start": 0, "tokens": 61},
        # a first prompt in the fast mode (batches of 128)
        {"name": "prompt_8b_fast", "kind": "prompt", "model": "llama3-8b", "layers": 4, "mix": "q4_k_m", "kv": "f32",
         "batch": 128, "start": 0, "tokens": 512},
        # the widest model: a prompt that wraps the local layers' rings
        {"name": "prompt_27b_fast", "kind": "prompt", "model": "gemma3-27b-6l", "layers": 6, "mix": "q4_k_m", "kv": "f32",
         "batch": 128, "start": 0, "tokens": 1280},
        # the next user message of a conversation: a short ragged prompt behind a cached prefix
        {"name": "turn_8b_q5", "kind": "prompt", "model": "llama3-8b", "layers": 4, "mix": "q5_k_m", "kv": "f32",
         "batch": 128, "start": 1500, "tokens": 21},
        # a file of 8-bit weights in batches of 64
        {"name": "prompt_8b_q8", "kind": "prompt", "model": "llama3-8b", "layers": 2, "mix": "q8_0", "kv": "f16",
         "batch": 64, "start": 0, "tokens": 200},
        # single ops, as a host drives them: one token's MLP on half-precision weights
        {"name": "mlp_f16_one", "kind": "mlp", "type": "f16", "hidden": 1024, "ffn": 3072, "batch": 1},
        # and a batch of 32 through Q6_K weights
        {"name": "mlp_q6_32", "kind": "mlp", "type": "q6_k", "hidden": 4096, "ffn": 14336, "batch": 32},
        # attention of a default prompt batch over a long ring
        {"name": "attention_8k", "kind": "attention", "heads": 32, "kv_heads": 16, "head_dim": 128, "start": 8191,
         "window": 8448, "batch": 16, "kv": "f32"},
        # the token pick of the default generation settings (temperature 0.7, top-k 40, top-p 0.9)
        {"name": "sample_128k", "kind": "sample", "vocab": 128256, "top_k": 40, "draws": 4},
    ]


def _spread(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["prompt", "prompt", "prompt", "reply", "mlp", "mlp", "attention", "sample"])
    if kind in ("prompt", "reply"):
        model = rng.choice(["qwen3-0.6b", "qwen3-0.6b", "llama3-8b"])
        c = {"kind": kind, "model": model, "layers": rng.randint(4, 28) if model == "qwen3-0.6b" else rng.randint(1, 4),
             "mix": rng.choice(["q4_k_m", "q4_k_m", "q5_k_m", "q8_0"]), "kv": rng.choice(["f32", "f16"])}
        if kind == "prompt":
            c["batch"] = rng.choice([8, 16, 16, 32, 64, 128])
            c["start"] = rng.choice([0, 0, _spread(rng, 16, 2000)])
            c["tokens"] = _spread(rng, 2, 400)
        else:
            c["batch"], c["start"], c["tokens"] = 128, _spread(rng, 8, 6000), _spread(rng, 4, 24)
        return c
    if kind == "mlp":
        t = rng.choice(sorted(TYPES))
        unit = 256 if t.endswith("_k") else 64
        return {"kind": "mlp", "type": t, "hidden": unit * _spread(rng, 512 // unit, 5376 // unit),
                "ffn": unit * _spread(rng, 512 // unit, 16384 // unit), "batch": _spread(rng, 1, 128)}
    if kind == "attention":
        kvh = rng.choice([2, 4, 8, 16])
        start = _spread(rng, 1, 12000)
        return {"kind": "attention", "heads": kvh * rng.choice([1, 2, 4, 8]), "kv_heads": kvh,
                "head_dim": rng.choice([64, 128, 128, 256]), "start": start,
                "window": rng.choice([start + 128, 1024]), "batch": _spread(rng, 1, 128), "kv": rng.choice(["f32", "f16"])}
    return {"kind": "sample", "vocab": _spread(rng, 4000, 262144), "top_k": _spread(rng, 1, 200), "draws": rng.randint(1, 6)}


# ------------------------------------------------------------------------------- weights

def _gen(seed, tag):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1_000_003 + tag * 7919 + 17) & 0x7FFFFFFFFFFF)


def _blocks(type_, n, gen, std):
    """n weights of a type as GGUF bytes on the GPU (uint8), standard deviation about ``std``."""
    if type_ in (F32, F16):
        v = torch.randn(n, generator=gen, device="cuda") * std
        return (v if type_ == F32 else v.half()).view(torch.uint8)
    per, size = BLOCK[type_]
    b = torch.randint(0, 256, (n // per, size), generator=gen, device="cuda", dtype=torch.uint8)
    u = torch.rand(n // per, generator=gen, device="cuda") * 0.5 + 0.75
    half = lambda d: d.half().view(torch.uint8).reshape(-1, 2)  # noqa: E731
    if type_ in (Q4_K, Q5_K):  # a centred block: dmin takes the mean of the quants away
        d = u * (std / (245.0 if type_ == Q4_K else 480.0))
        b[:, 0:2], b[:, 2:4] = half(d), half(d * (7.5 if type_ == Q4_K else 15.5))
    elif type_ == Q6_K:
        b[:, 208:210] = half(u * (std / 1365.0))
    else:
        b[:, 0:2] = half(u * (std / (73.9 if type_ == Q8_0 else 4.6)))
    return b.reshape(-1)


def _decode(type_, raw):
    """GGUF bytes (uint8, GPU) -> float64 weights."""
    if type_ == F32:
        return raw.view(torch.float32).double()
    if type_ == F16:
        return raw.view(torch.float16).double()
    b = raw.reshape(-1, BLOCK[type_][1])
    f16 = lambda i: b[:, i:i + 2].contiguous().view(torch.float16).double()  # noqa: E731
    if type_ == Q8_0:
        return (f16(0) * b[:, 2:].contiguous().view(torch.int8).double()).reshape(-1)
    if type_ == Q4_0:
        q = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double() - 8
        return (f16(0) * q).reshape(-1)
    if type_ == Q6_K:
        ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 32)
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        lo = torch.cat([ql & 15, ql >> 4], 2)  # [half][4][32] in element order
        hi = torch.stack([(qh >> (2 * k)) & 3 for k in range(4)], 2)
        q = (lo | (hi << 4)).double() - 32
        return (f16(208)[:, :, None] * sc[:, :, None] * q.reshape(-1, 16, 16)).reshape(-1)
    s = b[:, 4:16]
    sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
    qs = b[:, 16 if type_ == Q4_K else 48:].reshape(-1, 4, 1, 32)
    q = torch.cat([qs & 15, qs >> 4], 2).reshape(-1, 8, 32)
    if type_ == Q5_K:
        qh = b[:, 16:48]
        q = q | torch.stack([((qh >> j) & 1) << 4 for j in range(8)], 1)
    return (f16(0)[:, :, None] * sc[:, :, None] * q.double() - f16(2)[:, :, None] * mn[:, :, None]).reshape(-1)


# ------------------------------------------------------------------------------- models

def _spec(case):
    s = synth.SPECS[case["model"]]
    return dataclasses.replace(s, layers=case["layers"], types=MIXES[case["mix"]] or s.types)


def _tensors(spec, seed):
    """(name, dims, type, bytes on the GPU) of a model, in file order; one at a time."""
    for i, (name, dims, type_, role) in enumerate(synth.tensor_list(spec)):
        gen, n = _gen(seed, i), math.prod(dims)
        if role == "norm":
            v = 0.9 + 0.2 * torch.rand(n, generator=gen, device="cuda")
            if spec.signed_out_norm and name == "output_norm.weight":
                v = v * (torch.randint(0, 2, (n,), generator=gen, device="cuda") * 2 - 1)
            yield name, dims, type_, v.view(torch.uint8)
        else:
            std = spec.embd_std if role == "embd" and spec.embd_std is not None else spec.std
            yield name, dims, type_, _blocks(type_, n, gen, std)


def _gguf(spec, seed):
    """The model as a GGUF file in host memory."""
    text = lambda v: struct.pack("<Q", len(v.encode())) + v.encode()  # noqa: E731
    scalar = {4: lambda v: struct.pack("<I", v), 6: lambda v: struct.pack("<f", v), 8: text}
    meta, tensors = synth.metadata(spec), synth.tensor_list(spec)
    head = struct.pack("<IIQQ", synth.MAGIC, 3, len(tensors), len(meta))
    for key, kind, value in meta:
        head += text(key) + struct.pack("<I", kind) + scalar[kind](value)
    at, offsets = 0, []
    for name, dims, type_, _ in tensors:
        at = -(-at // 32) * 32
        offsets.append(at)
        head += text(name) + struct.pack("<I", len(dims)) + b"".join(struct.pack("<Q", d) for d in dims)
        head += struct.pack("<IQ", type_, at)
        at += synth.tensor_bytes(dims, type_)
    begin = -(-len(head) // 32) * 32
    file = torch.zeros(begin + at, dtype=torch.uint8, device="cuda")
    file[:len(head)] = torch.frombuffer(bytearray(head), dtype=torch.uint8).cuda()
    for off, (_, _, _, raw) in zip(offsets, _tensors(spec, seed)):
        file[begin + off:begin + off + raw.numel()] = raw
    return file.cpu().numpy()


def _ids(case, spec, seed):
    rng = np.random.default_rng(seed)
    return [int(v) for v in rng.integers(0, spec.vocab, case["start"] + (case["tokens"] if case["kind"] == "prompt" else 1))]


class _Session:
    """A loaded engine whose rings hold the case's cached prefix."""

    def __init__(self, case, seed):
        spec = _spec(case)
        self.case, self.ids, self.engine = case, _ids(case, spec, seed), PagedEngine()
        context = max(256, -(-(case["start"] + case["tokens"] + 2) // 128) * 128)
        self.engine.load(_gguf(spec, seed), LoadOptions(contextLength=context, batchSize=case["batch"], kvCacheType=case["kv"]))
        self.engine.source.close()
        for i in range(0, case["start"], case["batch"]):
            self.engine.forward(self.ids[i:min(i + case["batch"], case["start"])], i, False)

    def run(self):
        c, e, start = self.case, self.engine, self.case["start"]
        if c["kind"] == "prompt":
            end = len(self.ids)
            for i in range(start, end, c["batch"]):
                logits = e.forward(self.ids[i:i + c["batch"]], i, i + c["batch"] >= end)
            return {"logits": logits}
        tokens = e.decode(self.ids[start], start, c["tokens"])
        return {"logits": e.forward([tokens[-1]], start + c["tokens"], True), "tokens": np.array(tokens, np.int32)}

    def __del__(self):
        self.engine.dispose()


class _Exact:
    """The decoder in float64: every matrix decoded when it is used, K and V kept whole."""

    def __init__(self, case, seed):
        self.s, self.half = _spec(case), case["kv"] == "f16"
        self.t = {name: (dims, type_, raw) for name, dims, type_, raw in _tensors(self.s, seed)}
        self.k, self.v = [None] * self.s.layers, [None] * self.s.layers

    def mat(self, name, rows=None):
        dims, type_, raw = self.t[name]
        if rows is not None:
            raw = raw.reshape(dims[1], -1)[rows].reshape(-1)
        return _decode(type_, raw).reshape(-1, dims[0])

    def norm(self, x, name):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + self.s.eps) * _decode(F32, self.t[name][2])

    def rope(self, x, pos, theta):
        hd = x.shape[-1]
        a = pos.double()[:, None, None] * theta ** (-torch.arange(0, hd, 2, device="cuda").double() / hd)
        c, s = torch.cos(a), torch.sin(a)
        if self.s.arch == "llama":  # adjacent pairs
            l, r = x[..., 0::2], x[..., 1::2]
            return torch.stack([l * c - r * s, l * s + r * c], -1).reshape(x.shape)
        l, r = x[..., :hd // 2], x[..., hd // 2:]
        return torch.cat([l * c - r * s, l * s + r * c], -1)

    def attend(self, q, k, v, start, window):
        n, heads, hd = q.shape
        out, group = torch.empty_like(q), heads // k.shape[1]
        at = torch.arange(start, start + n, device="cuda")[:, None]
        key = torch.arange(k.shape[0], device="cuda")[None]
        mask = (key > at) | (key <= at - window)
        for h in range(heads):
            p = (q[:, h] @ k[:, h // group].t().contiguous()) / math.sqrt(hd)
            out[:, h] = torch.softmax(p.masked_fill(mask, -math.inf), -1) @ v[:, h // group].contiguous()
        return out.reshape(n, -1)

    def forward(self, ids, start):
        s, gemma = self.s, self.s.arch == "gemma3"
        pos = torch.arange(start, start + len(ids), device="cuda")
        x = self.mat("token_embd.weight", torch.tensor(ids, device="cuda")) * (math.sqrt(s.hidden) if gemma else 1.0)
        for l in range(s.layers):
            p = "blk.%d." % l
            local = gemma and l % 6 != 5
            h = self.norm(x, p + "attn_norm.weight")
            q, k, v = ((h @ self.mat(p + "attn_%s.weight" % m).t()).reshape(len(ids), -1, s.head_dim) for m in "qkv")
            if s.qk_norm:
                q, k = self.norm(q, p + "attn_q_norm.weight"), self.norm(k, p + "attn_k_norm.weight")
            theta = s.local_theta if local else s.theta
            q, k = self.rope(q, pos, theta), self.rope(k, pos, theta)
            if self.half:
                k, v = k.float().half().double(), v.float().half().double()
            self.k[l] = k if start == 0 else torch.cat([self.k[l], k])
            self.v[l] = v if start == 0 else torch.cat([self.v[l], v])
            o = self.attend(q, self.k[l], self.v[l], start, s.window if local else 1 << 30) @ self.mat(p + "attn_output.weight").t()
            x = x + (self.norm(o, p + "post_attention_norm.weight") if gemma else o)
            h = self.norm(x, p + "ffn_norm.weight")
            g, u = (h @ self.mat(p + "ffn_%s.weight" % m).t() for m in ("gate", "up"))
            g = 0.5 * g * (1 + torch.tanh(0.7978845608 * (g + 0.044715 * g ** 3))) if gemma else g * torch.sigmoid(g)
            d = (g * u) @ self.mat(p + "ffn_down.weight").t()
            x = x + (self.norm(d, p + "post_ffw_norm.weight") if gemma else d)
        h = self.norm(x[-1], "output_norm.weight")
        head = "token_embd.weight" if s.tied else "output.weight"
        rows = torch.arange(s.vocab, device="cuda").split(16384)
        return torch.cat([self.mat(head, r) @ h for r in rows])


# ------------------------------------------------------------------------------- single ops

def _mlp_inputs(case, seed):
    """x [batch][hidden], the norm weight, and gate, up and down as GGUF bytes."""
    H, F, t = case["hidden"], case["ffn"], TYPES[case["type"]]
    x = torch.randn(case["batch"], H, generator=_gen(seed, 0), device="cuda")
    w = 0.9 + 0.2 * torch.rand(H, generator=_gen(seed, 1), device="cuda")
    return x, w, [_blocks(t, H * F, _gen(seed, 2 + i), 0.02) for i in range(3)]


class _Mlp:
    """norm -> gate, up -> SiLU -> down -> residual, one op at a time on device buffers."""

    def __init__(self, case, seed):
        H, F, B, t = case["hidden"], case["ffn"], case["batch"], TYPES[case["type"]]
        x, w, mats = _mlp_inputs(case, seed)
        self.case, self.c = case, Compute().init()
        c = self.c
        self.x, self.w = c.upload(x.cpu().numpy(), "x"), c.upload(w.cpu().numpy(), "norm")
        shapes = ((H, F), (H, F), (F, H))
        self.m = [c.upload_weights(t, k, r, m.cpu().numpy()) for m, (k, r) in zip(mats, shapes)]
        self.state, self.normed, self.down = (c.buffer(4 * B * H, n) for n in ("state", "normed", "down"))
        self.gate, self.up, self.prod = (c.buffer(4 * B * F, n) for n in ("gate", "up", "product"))

    def run(self):
        c, H, F, B, t = self.c, self.case["hidden"], self.case["ffn"], self.case["batch"], TYPES[self.case["type"]]
        c.copy(self.x, self.state, 4 * B * H)
        c.norm(self.state, self.w, self.normed, H, 1e-5, B)
        c.matmul(t, self.m[0], self.normed, self.gate, H, F, F, 0, 0, B)
        c.matmul(t, self.m[1], self.normed, self.up, H, F, F, 0, 0, B)
        c.silu(self.gate, self.up, self.prod, B * F)
        c.matmul(t, self.m[2], self.prod, self.down, F, H, H, 0, 0, B)
        c.add(self.down, self.state, B * H)
        return {"state": c.read_f32(self.state, B * H)}

    def __del__(self):
        self.c.dispose()


def _attention_inputs(case, seed):
    """q of a batch, and K/V rings that hold every key up to its last query."""
    T = case["start"] + case["batch"]
    q = torch.randn(case["batch"], case["heads"], case["head_dim"], generator=_gen(seed, 0), device="cuda")
    kv = [torch.randn(T, case["kv_heads"], case["head_dim"], generator=_gen(seed, 1 + i), device="cuda") for i in range(2)]
    return (q, *kv) if case["kv"] == "f32" else (q, kv[0].half(), kv[1].half())


class _Attention:
    def __init__(self, case, seed):
        self.case, self.c = case, Compute().init()
        self.q, self.k, self.v = (self.c.upload(t.cpu().numpy()) for t in _attention_inputs(case, seed))
        self.n = case["batch"] * case["heads"] * case["head_dim"]
        self.y = self.c.buffer(4 * self.n, "attention")

    def run(self):
        a, c = self.case, self.c
        op = c.attention if a["kv"] == "f32" else c.attention_f16kv
        T = a["start"] + a["batch"]
        op(self.q, self.k, self.v, self.y, a["heads"], a["kv_heads"], a["head_dim"], a["start"],
           1 / math.sqrt(a["head_dim"]), a["window"], T, T, a["batch"])
        return {"y": c.read_f32(self.y, self.n)}

    def __del__(self):
        self.c.dispose()


class _Sample:
    """Draws of the next token from one row of logits with the default settings."""

    def __init__(self, case, seed):
        self.case, self.seed, self.c = case, seed, Compute().init()
        self.logits = self.c.upload(_logits(case, seed).cpu().numpy(), "logits")

    def run(self):
        a = self.case
        return [self.c.sample(self.logits, a["vocab"], 0.7, a["top_k"], 0.9, self.seed, i) for i in range(a["draws"])]

    def __del__(self):
        self.c.dispose()


def _logits(case, seed):
    return 2.5 * torch.randn(case["vocab"], generator=_gen(seed, 0), device="cuda")


# ------------------------------------------------------------------------------- the interface

def prepare(case, seed):
    if case["kind"] in ("prompt", "reply"):
        return _Session(case, seed)
    return {"mlp": _Mlp, "attention": _Attention, "sample": _Sample}[case["kind"]](case, seed)


def run(state):
    return state.run()


def work(case):
    kind = case["kind"]
    if kind == "sample":
        return {"bytes": 4.0 * case["vocab"] * case["draws"], "flops": 0.0}
    if kind == "attention":
        n, end, hd = case["batch"], case["start"] + case["batch"], case["head_dim"]
        pairs = sum(min(case["start"] + b + 1, case["window"]) for b in range(n))
        keys = min(end, case["window"] + n - 1)
        size = 4 if case["kv"] == "f32" else 2
        return {"bytes": 2.0 * keys * case["kv_heads"] * hd * size + 8.0 * n * case["heads"] * hd,
                "flops": 4.0 * pairs * case["heads"] * hd}
    if kind == "mlp":
        per, size = BLOCK[TYPES[case["type"]]]
        weights = 3.0 * case["hidden"] * case["ffn"]
        return {"bytes": weights / per * size + 8.0 * case["batch"] * case["hidden"], "flops": 2.0 * weights * case["batch"]}
    s = _spec(case)
    layer = head = weights = 0.0
    for name, dims, type_, role in synth.tensor_list(s):
        b = synth.tensor_bytes(dims, type_)
        if name.startswith("blk."):
            layer += b
            weights += math.prod(dims) if len(dims) == 2 else 0
        elif name == ("token_embd.weight" if s.tied else "output.weight"):
            head, vocab_weights = float(b), float(math.prod(dims))
    size = 4 if case["kv"] == "f32" else 2
    row, pair = 2.0 * s.kv_heads * s.head_dim * size, 4.0 * s.heads * s.head_dim
    start, n = case["start"], case["tokens"]
    seen = lambda l, pos: min(pos + 1, s.window) if s.arch == "gemma3" and l % 6 != 5 else pos + 1  # noqa: E731
    if kind == "reply":  # every step reads every weight and the keys behind it
        steps = range(start, start + n + 1)
        keys = float(sum(seen(l, p) for l in range(s.layers) for p in steps))
        return {"bytes": len(steps) * (layer + head) + keys * row, "flops": len(steps) * 2 * (weights + vocab_weights) + keys * pair}
    chunks = [(i, min(i + case["batch"], start + n)) for i in range(start, start + n, case["batch"])]
    # the mode's batch bounds the activations, so each chunk reads the layers' weights once
    keys = float(sum(min(e, seen(l, e - 1) + e - i - 1) for l in range(s.layers) for i, e in chunks))
    pairs = float(sum(seen(l, p) for l in range(s.layers) for p in range(start, start + n)))
    return {"bytes": len(chunks) * layer + head + keys * row, "flops": 2 * weights * n + 2 * vocab_weights + pairs * pair}


def tolerance(case):
    if case["kind"] == "sample":  # f64 probabilities of f32 logits: the draw is one token
        return "exact"
    if case["kind"] in ("prompt", "reply"):
        # measured against float64: 3e-5 (16-bit splits of both operands of a prompt's
        # products); with half-precision rings 2e-4, as a cached value next to the middle of
        # two halves may round either way
        return {"rel": 1.5e-4, "max": 1.5e-3} if case["kv"] == "f32" else {"rel": 8e-4, "max": 8e-3}
    if case["kind"] == "attention":  # measured 5e-7: f32 products and sums
        return {"rel": 4e-6, "max": 4e-5}
    return {"rel": 4e-5, "max": 4e-4}  # measured 7e-6: the same splits


def exact(case, seed):
    kind = case["kind"]
    if kind in ("prompt", "reply"):
        spec = _spec(case)
        m, ids, start = _Exact(case, seed), _ids(case, spec, seed), case["start"]
        logits = None
        end = len(ids) if kind == "prompt" else start
        for i in range(0, end, 2048):
            logits = m.forward(ids[i:min(i + 2048, end)], i)
        if kind == "prompt":
            return {"logits": logits}
        token = ids[start]
        for i in range(case["tokens"] + 1):
            logits = m.forward([token], start + i)
            token = int(logits.argmax())
        return {"logits": logits, "tokens": None}
    if kind == "mlp":
        x, w, mats = _mlp_inputs(case, seed)
        x, F = x.double(), case["ffn"]
        h = x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * w.double()
        t = TYPES[case["type"]]
        g, u = (h @ _decode(t, m).reshape(F, -1).t() for m in mats[:2])
        return {"state": (x + (g * torch.sigmoid(g) * u) @ _decode(t, mats[2]).reshape(-1, F).t()).reshape(-1)}
    if kind == "attention":
        q, k, v = (t.double() for t in _attention_inputs(case, seed))
        n, heads, hd = q.shape
        at = torch.arange(case["start"], case["start"] + n, device="cuda")[:, None]
        key = torch.arange(k.shape[0], device="cuda")[None]
        mask = (key > at) | (key <= at - case["window"])
        out, group = torch.empty_like(q), heads // case["kv_heads"]
        for h in range(heads):
            p = (q[:, h] @ k[:, h // group].t().contiguous()) / math.sqrt(hd)
            out[:, h] = torch.softmax(p.masked_fill(mask, -math.inf), -1) @ v[:, h // group].contiguous()
        return {"y": out.reshape(-1)}
    return None
