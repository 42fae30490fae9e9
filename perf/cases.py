"""Performance cases: forward passes of a server on this library, through the C ABI (transformer_batch over paged pools).

A case is one ragged batch: `prompts` prompt portions of `portion` tokens each, which begin at position `start` of their
sequences, and `rows` decoding sequences with one token each, whose cached contexts lie between half of `context` and
`context`.  What is cached has been through the library before (prepare), run() is the one pass, and its outputs are the
logits rows that transformer_batch leaves for the driver: one per sequence, the last token's.

Models have random weights in the shapes of this repository's benchmark and tests.  They are loaded once per process, as
a server does; a case's tokens come from the seed.
"""
import ctypes as C
import json
import math
import os
import struct
import tempfile
import zlib

import numpy as np
import torch

from nvllm_amd import capi, synth

BLOCK = 16
MAX_PASS = 2048   # tokens of one pass (the workspace that malloc_run_state lays out)
EPS = 1e-5

# ------------------------------------------------------------------------------------------------ cases


def case(name, model, weights, pool, prompts=0, portion=0, start=0, rows=0, context=0):
    c = dict(model=model, weights=weights, pool=pool, prompts=prompts, portion=portion, start=start, rows=rows, context=context)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one user, a trained llama2.c checkpoint as it is (fp32 values that fp16 cannot hold): the reference's demo.  The smallest call
        case("chat-15m-f32", "stories15M", "f32", "f32", rows=1, context=120),
        # a prompt of odd length on such a checkpoint
        case("prompt-42m-f32", "stories42M", "f32", "f32", prompts=1, portion=301),
        # a small fp16 model for a batch of users, the library's default pool
        case("decode-42m-b32", "stories42M", "f16", "f32", rows=32, context=220),
        # one user of a 1.1B model: latency of a token
        case("chat-1b", "tinyllama-1.1b", "f16", "f16", rows=1, context=700),
        # the benchmark's step: 64 users
        case("decode-1b-b64", "tinyllama-1.1b", "f16", "f16", rows=64, context=1088),
        # continuous batching: prompt chunks and the users that already decode
        case("prefill-1b", "tinyllama-1.1b", "f16", "f16", prompts=3, portion=512, start=512, rows=11, context=1050),
        # long contexts of few users, on the default pool
        case("long-1b", "tinyllama-1.1b", "f16", "f32", rows=9, context=3900),
        # the designs that come as folders, in bf16: a decoding batch, and prompt chunks
        case("decode-suselorn", "suselorn-1.2b", "bf16", "bf16", rows=64, context=1088),
        case("prefill-suselorn", "suselorn-1.2b", "bf16", "bf16", prompts=2, portion=512, start=512, rows=5, context=1050),
        case("decode-simivik", "simivik-1.2b", "bf16", "bf16", rows=64, context=1088),
        case("prefill-simivik", "simivik-1.2b", "bf16", "bf16", prompts=2, portion=512, start=512, rows=5, context=1050),
        # a replayed trace in 32 bits: a prompt beside decoding rows
        case("replay-simivik-f32", "simivik-0.4b", "f32", "f32", prompts=1, portion=77, rows=3, context=200),
    ]


def draw(rng):
    """Another ragged batch of the ranges above."""
    def spread(lo, hi):
        return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))

    kind = rng.choice(["small-f32", "small-f16", "1b", "1b", "suselorn", "simivik", "folder-f32"])
    c = dict(prompts=0, portion=0, start=0, rows=0, context=0)
    longest = {"small-f32": 240, "small-f16": 1000, "folder-f32": 300}.get(kind, 2000)
    if rng.random() < 0.55:
        c["rows"] = spread(1, 8 if kind == "folder-f32" else 64)
        c["context"] = spread(16, longest if c["rows"] <= 16 else min(longest, 1088))
    else:
        c["prompts"] = rng.choice([1, 1, 2, 3])
        c["portion"] = spread(8, (100 if kind == "folder-f32" else min(longest, 512)) // (2 if kind.startswith("small") else 1))
        c["start"] = rng.choice([0, 0, c["portion"]])
        if rng.random() < 0.5:
            c["rows"], c["context"] = spread(1, 8), spread(16, min(longest, 1050))
    if kind == "small-f32":
        return case(None, rng.choice(["stories15M", "stories42M"]), "f32", "f32", **c)
    if kind == "small-f16":
        return case(None, "stories42M", "f16", rng.choice(["f16", "f32"]), **c)
    if kind == "1b":
        return case(None, "tinyllama-1.1b", "f16", rng.choice(["f16", "f16", "f32"]), **c)
    if kind == "folder-f32":
        return case(None, rng.choice(["suselorn-0.4b", "simivik-0.4b"]), "f32", "f32", **c)
    return case(None, kind + rng.choice(["-0.4b", "-1.2b"]), "bf16", "bf16", **c)


def sequences(c):
    """(cached positions, new tokens) of each sequence of the batch."""
    out = [(c["start"], c["portion"])] * c["prompts"]
    for i in range(c["rows"]):   # contexts between a half of `context` and all of it, no two alike
        out.append((max(1, round(c["context"] * (1.0 - 0.5 * ((i * 0.6180339887) % 1.0)))), 1))
    return out


# ------------------------------------------------------------------------------------------------ models

FOLDERS = {   # sizes of the repository's benchmark of these designs
    "0.4b": dict(width=1024, ff=2816, layers=16, vocab=32000, heads=16, kv_heads=4, dim=64, rot=32, vdim=64, kv_rank=256, q_rank=512),
    "1.2b": dict(width=2048, ff=5632, layers=22, vocab=32000, heads=32, kv_heads=4, dim=64, rot=64, vdim=64, kv_rank=512, q_rank=1024),
}
MAX_LEN = {"stories15M": 256, "stories42M": 1024, "tinyllama-1.1b": 4096}


def llama_shape(model):
    return synth.ModelShape.named(model, max_seq_len=MAX_LEN[model])


def llama_tensors(s):
    """name -> shape, in file order."""
    D, F, V, QD, KD = s.dim, s.hidden_dim, s.vocab_size, s.n_heads * s.head_dim, s.n_kv_heads * s.head_dim
    out = {"embed": (V, D)}
    for name, shape in (("rms_att", (D,)), ("wq", (QD, D)), ("wk", (KD, D)), ("wv", (KD, D)), ("wo", (D, QD)),
                        ("rms_ffn", (D,)), ("gate", (F, D)), ("down", (D, F)), ("up", (F, D))):
        for i in range(s.n_layers):
            out["%s.%d" % (name, i)] = shape
    out["rms_final"] = (D,)
    return out


def folder_config(model):
    design, size = model.split("-")
    z = FOLDERS[size]
    if design == "suselorn":
        m = synth.latent_mixer(z["heads"], z["dim"], z["rot"], z["vdim"], z["kv_rank"], z["q_rank"])
        return synth.latent_config(z["width"], z["vocab"], [(m, z["ff"])] * z["layers"], streams=2)
    window = synth.window_mixer(z["heads"], z["kv_heads"], z["dim"], z["vdim"], size=512, keep_first=16)
    decay = [math.exp(-0.7 * 0.8 ** i) for i in range(z["heads"])]
    lightning, experts = synth.lightning_mixer(z["heads"], z["dim"], z["vdim"], decay), synth.expert_mlp(z["ff"] // 4, 16, 2, z["ff"] // 2)
    period = [(lightning, z["ff"]), (window, experts), (window, z["ff"]), (window, experts)]
    return synth.hybrid_config(z["width"], z["vocab"], [period[i % 4] for i in range(z["layers"])])


class Tensors:
    """The weights of a model, tensor by tensor on the GPU, each from its own seed: what the file holds and what exact() uses."""

    def __init__(self, model, weights):
        self.model, self.weights = model, weights
        if model in MAX_LEN:
            self.cfg, self.routed = None, 0
            self.shapes = {n: (s, None) for n, s in llama_tensors(llama_shape(model)).items()}
            if weights == "f16":   # fp16 files bring a classifier of their own
                self.shapes["head"] = (self.shapes["embed"][0], None)
        else:
            self.cfg = folder_config(model)
            self.shapes = synth.DESIGN_TENSORS[self.cfg["architecture"]](self.cfg)
            self.routed = max([x["mlp"]["router"]["experts"] for x in self.cfg["layers"] if x["mlp"] and x["mlp"]["kind"] == "moe"], default=0)

    def __call__(self, name):
        shape, kind = self.shapes[name]
        gen = torch.Generator("cuda").manual_seed(zlib.crc32(("%s %s" % (self.model, name)).encode()))

        def normal(std, mean=0.0):
            return torch.randn(shape, generator=gen, device="cuda") * std + mean

        fan = shape[-1] if shape else 1
        if kind is None:
            if name.startswith("rms"):
                v = normal(0.1, 1.0)
            elif name in ("embed", "head"):
                v = normal(1.0 if name == "embed" and "head" in self.shapes else 3.0 * fan ** -0.5)
            else:
                v = normal(fan ** -0.5)
            return v.half() if self.weights == "f16" else v
        if kind.endswith("embed"):
            v = normal(3.0 * fan ** -0.5)
            if self.routed:
                # the routers read dims of their own, which hold every token's order of the experts, well apart, and which no layer
                # writes: as with trained routers the choice does not hang on rounding
                order = torch.rand((shape[0], self.routed), generator=gen, device="cuda").argsort(1).float()
                v[:, :self.routed] = (order - (self.routed - 1) / 2) * 0.15
        elif kind in ("matrix", "sharp", "routed_out"):
            v = normal(fan ** -0.5)
        elif kind == "router":
            v = normal(0.002)
            at = torch.randperm(shape[0], generator=gen, device="cuda")
            v[torch.arange(shape[0], device="cuda"), at] += 4.0
        elif kind == "taps":
            v = normal(0.2)
            v[:, -1] += 1.0
        elif kind == "mix":
            v = normal(0.05) + 0.9 * torch.eye(fan, device="cuda")
        else:
            v = {"gain": lambda: normal(0.1, 1.0), "bias": lambda: normal(0.02), "alpha": lambda: normal(0.05, 0.7), "sink": lambda: normal(1.0, 0.5),
                 "weight": lambda: normal(0.1, 0.6), "zero_gain": lambda: normal(0.1), "routed_zero_gain": lambda: normal(0.1)}[kind]()
        if kind in ("routed_out", "routed_zero_gain"):
            v[:self.routed] = 0.0
        if name == "final.norm" and self.routed:
            v[:self.routed] = -1.0   # (weights of these norms lie around zero: the routers' dims have no part in the logits)
        return v.bfloat16()

    def exact(self, name):
        return self(name).double()

    def write(self, folder):
        """The model's file or folder; returns its path."""
        raw = lambda t: (t.view(torch.int16) if t.dtype == torch.bfloat16 else t).cpu().numpy()  # noqa: E731
        if self.cfg is None:
            path = os.path.join(folder, "model.bin")
            with open(path, "wb") as f:
                f.write(llama_shape(self.model).header())
                for name in self.shapes:
                    raw(self(name)).tofile(f)
            return path
        header, at = {}, 0
        for name, (shape, _) in self.shapes.items():
            header[name] = dict(dtype="BF16", shape=list(shape), data_offsets=[at, at + 2 * math.prod(shape)])
            at += 2 * math.prod(shape)
        text = json.dumps(header).encode()
        text += b" " * (-len(text) % 8)
        with open(os.path.join(folder, "model.safetensors"), "wb") as f:
            f.write(struct.pack("<Q", len(text)) + text)
            for name in self.shapes:
                raw(self(name)).tofile(f)
        with open(os.path.join(folder, "config.json"), "w") as f:
            json.dump(self.cfg, f)
        return folder


LIB = None
MODELS = {}


def library():
    global LIB
    if LIB is None:
        LIB = capi.load_hip()
        LIB.nvllm_set_logits_mode(0)   # logits rows come to the host, as the reference's driver reads them
        LIB.init_ops()
    return LIB


class Model:
    """A loaded model, its workspace and the numbers its sequences go by."""

    def __init__(self, model, weights):
        lib = library()
        self.folder_model = model not in MAX_LEN
        self.cfg, self.weights, self.state = capi.Config(), capi.Weights(), capi.RunState()
        lib.nvllm_set_compute_dtype(capi.COMPUTE_F32 if weights == "f32" else capi.COMPUTE_BF16)
        with tempfile.TemporaryDirectory() as d:
            path = Tensors(model, weights).write(d)
            lib.load_model(C.byref(self.weights), C.byref(self.cfg), path.encode())
        self.cfg.max_seq_len = max(MAX_PASS, MAX_LEN.get(model, 0))
        lib.malloc_run_state(C.byref(self.state), C.byref(self.cfg))
        self.free_ids = list(range(4 * 64 - 1, -1, -1))
        if self.folder_model:
            lib.nvllm_init_model_states(C.byref(self.weights), len(self.free_ids))


def model_of(c):
    key = (c["model"], c["weights"])
    if key not in MODELS:
        MODELS[key] = Model(*key)
    return MODELS[key]


# ------------------------------------------------------------------------------------------------ a batch


def token_lists(c, seed):
    """Every sequence's tokens, the cached ones and the new."""
    vocab = 32000
    rng = np.random.default_rng(seed)
    return [rng.integers(3, vocab, size=cached + new).astype(np.int32) for cached, new in sequences(c)]


class Batch:
    """The driver's side of one case: a block pool, block tables, and the arrays of the coming pass."""

    def __init__(self, c, seed):
        lib = library()
        self.model = m = model_of(c)
        tokens, seqs = token_lists(c, seed), sequences(c)
        self.pool = capi.KVCacheManager()
        blocks = [-(-len(t) // BLOCK) for t in tokens]
        lib.nvllm_set_kv_elem_bytes(4 if c["pool"] == "f32" else 2)
        lib.nvllm_init_model_kv(C.byref(self.pool), BLOCK, sum(blocks), C.byref(m.cfg), C.byref(m.weights))
        self.ids = [m.free_ids.pop() for _ in tokens]
        top = max(self.ids) + 1
        self.tables = (C.POINTER(capi.BlockTable) * top)()
        self.records = []
        for i, n in zip(self.ids, blocks):
            at = (C.c_int * n)(*[lib.alloc_block(C.byref(self.pool)) for _ in range(n)])
            self.records.append(capi.BlockTable(C.cast(at, capi.c_int_p), n))
            self.records.append(at)
            self.tables[i] = C.pointer(self.records[-2])
        # what is cached goes through the model in passes of whole sequences' portions
        todo = [(i, t[:cached], 0) for i, t, (cached, _) in zip(self.ids, tokens, seqs) if cached]
        while todo:
            part, room = [], MAX_PASS
            while todo and room:
                i, t, at = todo.pop(0)
                n = min(len(t) - at, room, 512)
                part.append((i, t[at:at + n], at))
                room -= n
                if at + n < len(t):
                    todo.insert(0, (i, t, at + n))
                    break
            self.lay_out(part)
            self.run()
        self.lay_out([(i, t[cached:], cached) for i, t, (cached, _) in zip(self.ids, tokens, seqs)])

    def lay_out(self, part):
        """part: (sequence, its next tokens, their first position); one output row per sequence."""
        ends = np.cumsum([len(t) for _, t, _ in part])
        self.n, self.outputs = int(ends[-1]), len(part)
        self.args = (capi.ints(np.concatenate([t for _, t, _ in part])), capi.ints(np.concatenate([np.arange(at, at + len(t)) for _, t, at in part])),
                     capi.ints(np.concatenate([np.full(len(t), i) for i, t, _ in part])), capi.ints(ends - 1))

    def run(self):
        lib, m = LIB, self.model
        C.memmove(C.addressof(capi.KVCacheManager.in_dll(lib.dll, "g_kv_manager")), C.addressof(self.pool), C.sizeof(self.pool))   # the driver's pool
        tokens, pos, ids, out = self.args
        lib.transformer_batch(tokens, self.n, pos, ids, out, self.outputs, C.byref(m.cfg), C.byref(m.state), C.byref(m.weights), self.tables)
        return np.ctypeslib.as_array(C.cast(m.state.logits, capi.c_float_p), shape=(self.outputs, m.cfg.vocab_size))

    def __del__(self):
        if getattr(self, "ids", None):
            LIB.free_kv_cache_manager(C.byref(self.pool))
            self.model.free_ids += self.ids


def prepare(c, seed):
    return Batch(c, seed)


def run(state):
    return state.run()


# ------------------------------------------------------------------------------------------------ what a pass needs


def work(c):
    """Every weight that the batch meets read once, every cached key and value it may see read once, new ones written, the
    logits written; multiply-adds of the products and of attention."""
    seqs = sequences(c)
    n, outputs = sum(new for _, new in seqs), len(seqs)
    size = {"f16": 2, "bf16": 2, "f32": 4}
    wb, kb = size[c["weights"]], size[c["pool"]]
    seen = sum(cached + new for cached, new in seqs)                                     # positions that attention reads
    pairs = sum(new * cached + new * (new + 1) // 2 for cached, new in seqs)             # (query, key) pairs

    def windowed(cached, new, size, keep):
        return sum(min(p + 1, size) + min(keep, max(0, p + 1 - size)) for p in range(cached, cached + new))
    weights, products, cache, attention, rows = 0.0, 0.0, 0.0, 0.0, 0
    if c["model"] in MAX_LEN:
        s = llama_shape(c["model"])
        QD, KD = s.n_heads * s.head_dim, s.n_kv_heads * s.head_dim
        layer = 2 * s.dim * QD + 2 * s.dim * KD + 3 * s.dim * s.hidden_dim
        weights, products = s.n_layers * layer, s.n_layers * layer * n
        cache, attention, D, V = s.n_layers * 2 * KD * (seen + n), s.n_layers * 2 * QD * pairs, s.dim, s.vocab_size
    else:
        cfg = folder_config(c["model"])
        D, V = cfg["width"], cfg["vocab"]
        for x in cfg["layers"]:
            m, f = x["mixer"], x["mlp"]
            H = m["heads"]
            if "kv_rank" in m:
                layer = D * (m["q_rank"] + m["kv_rank"] + m["rot_dim"]) + m["q_rank"] * H * (m["dim"] + m["rot_dim"])
                layer += H * m["kv_rank"] * (m["dim"] + m["vdim"]) + D * H * m["vdim"]
                cache += (m["kv_rank"] + m["rot_dim"]) * (seen + n)
                attention += H * (2 * m["kv_rank"] + m["rot_dim"]) * pairs
            elif "decay" in m:
                layer = D * H * (2 * m["dim"] + 3 * m["vdim"])
                cache += len(seqs) * H * m["dim"] * m["vdim"] * 2 * 4 / kb               # 32-bit states, read and written
                attention += 2 * n * H * m["dim"] * m["vdim"]
            else:
                per_position = m["kv_heads"] * (m["dim"] + m["vdim"])
                layer = D * (H * (m["dim"] + m["vdim"]) + per_position)
                w = m["mask"]
                cache += per_position * (sum(min(a + b, w["size"] + b + w["keep_first"]) for a, b in seqs) + n)
                attention += H * (m["dim"] + m["vdim"]) * sum(windowed(a, b, w["size"], w["keep_first"]) for a, b in seqs)
            weights, products = weights + layer, products + layer * n
            if f["kind"] == "dense":
                layer = (2 if cfg["architecture"] == "Simivik" else 3) * D * f["ff"]
                weights, products = weights + layer, products + layer * n
            else:
                E, top, one, shared = f["router"]["experts"], f["router"]["top"], 3 * D * f["expert"]["ff"], 3 * D * f["shared"]["ff"] + D * (f["router"]["experts"] + 1)
                weights += E * (1 - (1 - top / E) ** n) * one + shared
                products += n * (top * one + shared)
    weights, products = weights + V * D, products + V * D * outputs
    return dict(bytes=wb * (weights + n * D) + kb * cache + 4 * outputs * V, flops=2 * (products + attention))


def tolerance(c):
    """About four times what the library is off exact() over these ranges: sums of 32 bits; cached keys and values in fp16;
    activations, keys and values in bf16 (of which the latent design rounds the more)."""
    if c["pool"] == "f32":
        return dict(rel=1e-5)
    return dict(rel=1.5e-3 if c["pool"] == "f16" else 3e-2 if c["model"].startswith("suselorn") else 2e-2)


# ------------------------------------------------------------------------------------------------ the same in 64 bits


def rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def angles(n, base, dims):
    a = torch.arange(n, device="cuda", dtype=torch.float64)[:, None] * base ** (-2.0 * torch.arange(dims // 2, device="cuda", dtype=torch.float64) / dims)
    return a.cos()[:, None], a.sin()[:, None]


def turn_pairs(x, base, dims):
    """x [tokens, heads, dim]: entries (2i, 2i + 1) turn."""
    c, s = angles(len(x), base, dims)
    u, v = x[..., 0:dims:2], x[..., 1:dims:2]
    return torch.cat([torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2), x[..., dims:]], -1)


def turn_halves(x, base, dims):
    """Entries (i, i + dims/2) turn."""
    c, s = angles(len(x), base, dims)
    u, v = x[..., :dims // 2], x[..., dims // 2:dims]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., dims:]], -1)


def attend(q, k, v, scale, cap=None, window=None, sink=None):
    """q [tokens, heads, dim], k and v [tokens, groups, ..] -> [tokens, heads * vdim]; window: (size, kept first ones)."""
    n, H, G = len(q), q.shape[1], k.shape[1]
    s = torch.matmul(q.transpose(0, 1).reshape(G, H // G * n, -1), k.permute(1, 2, 0).contiguous()).reshape(H, n, n) * scale
    if cap:
        s = cap * torch.tanh(s / cap)
    i, j = torch.arange(n, device="cuda")[:, None], torch.arange(n, device="cuda")[None]
    hidden = j > i
    if window:
        hidden = hidden | ((i - j >= window[0]) & (j >= window[1]))
    s = s.masked_fill(hidden, -math.inf)
    if sink is not None:
        s = torch.cat([s, sink[:, None, None].expand(H, n, 1)], -1)
    p = torch.softmax(s, -1)[..., :n].reshape(G, H // G * n, n)
    return torch.matmul(p, v.transpose(0, 1).contiguous()).reshape(H, n, -1).transpose(0, 1).reshape(n, -1)


def silu(x):
    return x * torch.sigmoid(x)


def llama_exact(W, c, x, parts):
    s = llama_shape(c["model"])
    for i in range(s.n_layers):
        w = lambda name: W.exact("%s.%d" % (name, i))  # noqa: B023, E731
        h = rms(x, EPS) * w("rms_att")
        q, k, v = h @ w("wq").T, h @ w("wk").T, h @ w("wv").T
        o = torch.cat([attend(turn_pairs(a.reshape(len(a), s.n_heads, -1), 10000.0, s.head_dim), turn_pairs(b.reshape(len(b), s.n_kv_heads, -1), 10000.0, s.head_dim),
                              d.reshape(len(d), s.n_kv_heads, -1), s.head_dim ** -0.5) for a, b, d in zip(q.split(parts), k.split(parts), v.split(parts))])
        x = x + o @ w("wo").T
        h = rms(x, EPS) * w("rms_ffn")
        x = x + (silu(h @ w("gate").T) * (h @ w("up").T)) @ w("down").T
    ends = torch.tensor(np.cumsum(parts) - 1, device="cuda")
    return (rms(x[ends], EPS) * W.exact("rms_final")) @ W.exact("head" if "head" in W.shapes else "embed").T


def suselorn_exact(W, c, x, parts):
    cfg = W.cfg
    eps = cfg["norm"]["eps"]
    streams = torch.stack([x] * cfg["streams"])

    def mixer(h, m, w):
        H, dim, rank = m["heads"], m["dim"], m["kv_rank"]
        q = ((rms(h @ w("dq").T, eps) * w("dq.norm")) @ w("uq").T).reshape(len(h), H, -1)
        kv = h @ w("dkv").T
        latent = rms(kv[:, :rank], eps) * w("dkv.norm")
        k, v = (latent @ w("uk").T).reshape(len(h), H, dim), (latent @ w("uv").T).reshape(len(h), H, -1)
        sink, base, rot = w("sink"), m["rot"]["base"], m["rot"]["dims"]
        outs = []
        for a, b, d, r in zip(q.split(parts), k.split(parts), v.split(parts), kv[:, rank:].split(parts)):
            a = torch.cat([a[..., :dim], turn_pairs(a[..., dim:], base, rot)], -1)
            b = torch.cat([b, turn_pairs(r[:, None], base, rot).expand(-1, H, -1)], -1)
            outs.append(attend(a, b, d, m["scale"], sink=sink))
        return torch.cat(outs) @ w("o").T

    def feed_forward(h, w):
        return (silu(h @ w("gate").T + w("gate.b")) * (h @ w("up").T + w("up.b"))) @ w("down").T + w("down.b")

    for i, layer in enumerate(cfg["layers"]):
        p = "l%d." % i
        for part in ("1", "2"):
            u = (W.exact(p + "hc" + part + ".in")[:, None, None] * streams).sum(0)
            h = torch.tanh(W.exact(p + "norm" + part + ".alpha") * u) * W.exact(p + "norm" + part) + W.exact(p + "norm" + part + ".b")
            y = mixer(h, layer["mixer"], lambda n: W.exact(p + "mix." + n)) if part == "1" else feed_forward(h, lambda n: W.exact(p + "mlp." + n))  # noqa: B023
            y = y * W.exact(p + "ls" + part)
            mix, out = W.exact(p + "hc" + part + ".mix"), W.exact(p + "hc" + part + ".out")
            streams = torch.matmul(mix.T, streams.flatten(1)).reshape(streams.shape) + out[:, None, None] * y
    ends = torch.tensor(np.cumsum(parts) - 1, device="cuda")
    z = torch.tanh(W.exact("final.norm.alpha") * streams.sum(0)[ends]) * W.exact("final.norm") + W.exact("final.norm.b")
    cap = cfg["logit_softcap"]
    return cap * torch.tanh(z @ W.exact("embed").T / cap)


def simivik_exact(W, c, x, parts):
    cfg = W.cfg
    eps = cfg["norm"]["eps"]

    def convolved(u, taps):
        n = taps.shape[1]
        padded = torch.cat([u.new_zeros(n - 1, u.shape[1]), u])
        return sum(taps[:, j] * padded[j:j + len(u)] for j in range(n))

    def lightning(h, m, w):
        H = m["heads"]
        q, k, v = (silu(h @ w(t).T).reshape(len(h), H, -1) for t in "qkv")
        decay = torch.tensor(m["decay"], device="cuda", dtype=torch.float64).log()
        outs = []
        for a, b, d in zip(q.split(parts), k.split(parts), v.split(parts)):
            i = torch.arange(len(a), device="cuda", dtype=torch.float64)
            gap = i[:, None] - i[None]
            s = torch.matmul(a.transpose(0, 1).contiguous(), b.permute(1, 2, 0).contiguous()) * torch.exp(decay[:, None, None] * gap.clamp(min=0)) * (gap >= 0)
            outs.append(torch.matmul(s, d.transpose(0, 1).contiguous()).transpose(0, 1).reshape(len(a), -1))
        return (rms(torch.cat(outs), eps) * w("norm") * torch.sigmoid(h @ w("g").T)) @ w("o").T

    def window(h, m, w):
        raw = {t: (h @ w(t).T).split(parts) for t in "qkv"}
        taps = {t: w(t + ".conv") for t in "qkv"}
        base, dims, mask = m["rot"]["base"], m["rot"]["dims"], m["mask"]
        outs = []
        for a, b, d in zip(*(raw[t] for t in "qkv")):
            n = len(a)
            a, b, d = convolved(a, taps["q"]).reshape(n, m["heads"], -1), convolved(b, taps["k"]).reshape(n, m["kv_heads"], -1), convolved(d, taps["v"]).reshape(n, m["kv_heads"], -1)
            outs.append(attend(turn_halves(a, base, dims), turn_halves(b, base, dims), d, m["scale"], m["softcap"], (mask["size"], mask["keep_first"])))
        return torch.cat(outs) @ w("o").T

    def experts(h, f, w):
        score, chosen = torch.sigmoid(h @ w("router").T).topk(f["router"]["top"], 1)
        gated = lambda u, n: (silu(u @ w(n + ".gate").T) * (u @ w(n + ".up").T)) @ w(n + ".down").T  # noqa: E731
        out = torch.sigmoid(h @ w("shared.sg").T) * gated(h, "shared")
        for e in range(f["router"]["experts"]):
            t, place = (chosen == e).nonzero(as_tuple=True)
            if len(t):
                out[t] += gated(score[t, place][:, None] * h[t], "e%d" % e)
        return out

    for i, layer in enumerate(cfg["layers"]):
        p = "l%d." % i
        h = rms(x, eps) * (1 + W.exact(p + "norm1"))
        x = x + (lightning if layer["type"] == "lightning" else window)(h, layer["mixer"], lambda n: W.exact(p + "mix." + n))  # noqa: B023
        h, w = rms(x, eps) * (1 + W.exact(p + "norm2")), lambda n: W.exact(p + "mlp." + n)  # noqa: B023, E731
        x = x + (torch.relu(h @ w("up").T) ** 2 @ w("down").T if layer["mlp"]["kind"] == "dense" else experts(h, layer["mlp"], w))
    ends = torch.tensor(np.cumsum(parts) - 1, device="cuda")
    return (rms(x[ends], eps) * (1 + W.exact("final.norm"))) @ W.exact("embed").T


def exact(c, seed):
    """The whole sequences at once, in 64 bits: nothing is cached, cut or batched."""
    tokens = token_lists(c, seed)
    W = Tensors(c["model"], c["weights"] if c["model"] in MAX_LEN else "bf16")
    x = W("embed")[torch.from_numpy(np.concatenate(tokens)).long().cuda()].double()
    form = llama_exact if c["model"] in MAX_LEN else suselorn_exact if c["model"].startswith("suselorn") else simivik_exact
    return form(W, c, x, [len(t) for t in tokens])
