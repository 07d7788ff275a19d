"""What the performance of this package is measured on: the work its users have it do, through its public entry points.

  gemm      y = W x for x and y in device memory (HipGemv.gemm_device), the matrices of several layers in turn, as a
            model's layers follow each other: 1 token (decode), a few (continuous batching), hundreds (a prompt chunk)
  step      all weight products of one generated token of an 8B-shaped model, as a graph of batched calls
  moe       the routed feed-forward of a layer with experts, host rows to host rows (Llama.moe_ffn)
  dispatch  gemv_<t>_f32 / gemm_<t>_f32 on host arrays: the call that finds its matrix by the bytes it is given
  generate  requests to a model: prompt, then greedy tokens - one session with everything on the GPU, several
            sequences decoded together, or the host session whose every product is a call of its own

Weights have the block formats of GGUF files with codes drawn uniformly and scales that give them mean 0 and deviation
0.02, as model weights have; activations are N(0, 1).
"""
import importlib
import math
import struct

import numpy as np
import torch

pkg = importlib.import_module("llama-rust_amd")
hip = importlib.import_module("llama-rust_amd.hiprt")
llama = importlib.import_module("llama-rust_amd.llama")

TYPES = {name: ty for ty, name in pkg.TYPE_NAMES.items()}
BLOCK = {"f32": (1, 4), "f16": (1, 2), "q4_0": (32, 18), "q5_0": (32, 22), "q5_1": (32, 24), "q8_0": (32, 34),
         "q4_k": (256, 144), "q6_k": (256, 210)}  # columns and bytes of a block

# Most operations and bytes of one drawn pass: below the largest listed case's.
MOST_FLOPS, MOST_BYTES = 2.0e11, 1.0e9


def listed():
    return [
        # decode through a small model's projection: the smallest calls, where the launch and the call count
        {"name": "gemv_q8_0_4096", "kind": "gemm", "type": "q8_0", "rows": 4096, "cols": 4096, "tokens": 1, "layers": 16},
        # decode of a half-billion-parameter model: rows of 28 blocks, which are not whole 256-column units
        {"name": "gemv_q5_0_896", "kind": "gemm", "type": "q5_0", "rows": 4864, "cols": 896, "tokens": 1, "layers": 24},
        # eight sequences decoded together, gate / up projection of an 8B model
        {"name": "gemm_q4_0_8_tokens", "kind": "gemm", "type": "q4_0", "rows": 14336, "cols": 4096, "tokens": 8, "layers": 8},
        # a ragged prompt remainder: tokens that fill no tile, an odd number of rows
        {"name": "gemm_q4_k_100_tokens", "kind": "gemm", "type": "q4_k", "rows": 4099, "cols": 14336, "tokens": 100, "layers": 4},
        # a long prompt chunk, down projection: bound by the matrix cores
        {"name": "gemm_q4_0_512_tokens", "kind": "gemm", "type": "q4_0", "rows": 4096, "cols": 14336, "tokens": 512, "layers": 4},
        # an unquantized model's prompt chunk
        {"name": "gemm_f16_128_tokens", "kind": "gemm", "type": "f16", "rows": 4096, "cols": 14336, "tokens": 128, "layers": 2},
        # one token of an 8B model: every byte of its weights once
        {"name": "decode_step_8b", "kind": "step", "type": "q4_k", "head": "q6_k", "layers": 32, "width": 4096, "kv": 1024,
         "ff": 14336, "vocab": 128256},
        # a routed layer of 8 experts, two per token
        {"name": "moe_64_tokens", "kind": "moe", "type": "q4_k", "width": 4096, "ff": 14336, "experts": 8, "used": 2, "tokens": 64},
        # the call shape of the engine this executor is a drop-in for: host arrays, weights identified by content
        {"name": "dispatch_q4_k", "kind": "dispatch", "type": "q4_k", "rows": 4096, "cols": 4096, "tokens": 1, "layers": 4},
        # chat with one user: two requests to a resident session
        {"name": "generate_one", "kind": "generate", "session": "device", "type": "q4_k", "layers": 4, "width": 4096, "heads": 32,
         "heads_kv": 8, "ff": 14336, "vocab": 32000, "sequences": 1, "prompt": 128, "new": 64},
        # a server: eight sequences, prompts of different lengths
        {"name": "generate_8", "kind": "generate", "session": "batch", "type": "q4_k", "layers": 4, "width": 4096, "heads": 32,
         "heads_kv": 8, "ff": 14336, "vocab": 32000, "sequences": 8, "prompt": 128, "new": 32},
        # the host session: attention and element-wise steps on the host, every product through host buffers
        {"name": "generate_host", "kind": "generate", "session": "host", "type": "q4_k", "layers": 4, "width": 4096, "heads": 32,
         "heads_kv": 8, "ff": 14336, "vocab": 32000, "sequences": 1, "prompt": 96, "new": 16},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width_of(type_name, n):
    """The nearest positive row length of whole blocks."""
    qk = max(BLOCK[type_name][0], 4)
    return max(1, round(n / qk)) * qk


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "gemm", "gemm", "step", "moe", "dispatch", "generate", "generate"])
    if kind == "gemm":
        ty = rng.choice(list(BLOCK))
        c = {"kind": kind, "type": ty, "rows": _log(rng, 64, 16384), "cols": _width_of(ty, _log(rng, 256, 16384)),
             "tokens": _log(rng, 1, 512)}
        flops, size = 2.0 * c["rows"] * c["cols"] * c["tokens"], c["rows"] * _row_bytes(ty, c["cols"])
        c["layers"] = max(1, min(16, int(MOST_FLOPS / flops), int(MOST_BYTES / 4 / size)))
    elif kind == "step":
        width = rng.choice([1024, 2048, 4096])
        c = {"kind": kind, "type": rng.choice(["q4_k", "q8_0", "q4_0", "q5_0", "q5_1", "q6_k"]), "head": rng.choice(["q6_k", "q8_0"]),
             "layers": _log(rng, 2, 16), "width": width, "kv": width // rng.choice([1, 4]), "ff": 256 * _log(rng, width // 128, width // 64),
             "vocab": _log(rng, 4000, 64000)}
    elif kind == "moe":
        width = rng.choice([1024, 2048])
        c = {"kind": kind, "type": rng.choice(["q4_k", "q8_0", "q4_0", "q6_k"]), "width": width, "ff": 256 * _log(rng, width // 256, width // 64),
             "experts": rng.choice([4, 8, 16]), "used": rng.choice([1, 2, 3]), "tokens": _log(rng, 1, 256)}
    elif kind == "dispatch":
        ty = rng.choice(list(BLOCK))
        c = {"kind": kind, "type": ty, "rows": _log(rng, 64, 8192), "cols": _width_of(ty, _log(rng, 256, 8192)), "tokens": _log(rng, 1, 64)}
        c["layers"] = max(1, min(8, int(5e7 / (c["rows"] * _row_bytes(ty, c["cols"])))))
    else:
        width = rng.choice([1024, 2048, 4096])
        heads = width // rng.choice([64, 128])
        session = rng.choice(["device", "batch", "batch", "host"])
        c = {"kind": kind, "session": session, "type": rng.choice(["q4_k", "q8_0", "q4_0", "q5_1", "q6_k"]), "layers": rng.randint(1, 3),
             "width": width, "heads": heads, "heads_kv": heads // rng.choice([1, 4, 8]), "ff": 256 * _log(rng, width // 128, width // 64),
             "vocab": _log(rng, 2000, 32000), "sequences": _log(rng, 2, 32) if session == "batch" else 1, "prompt": _log(rng, 3, 160)}
        # two requests, or all sequences: no more prompt tokens and steps than the listed cases have
        c["new"] = _log(rng, 4, 12 if session == "host" else 32)
        if session == "host":
            c["prompt"] = min(c["prompt"], 96)
    return c


# ------------------------------------------------------------------ weights and inputs
def _row_bytes(type_name, cols):
    qk, bb = BLOCK[type_name]
    return cols // qk * bb


def _packed(type_name, rows, cols, gen, sigma=0.02):
    """Rows of GGUF blocks on the device, as bytes."""
    def normal(*shape):
        return torch.randn(shape, generator=gen, device="cuda")

    def halves(v):
        return v.to(torch.float16).contiguous().view(torch.uint8)

    if type_name in ("f16", "f32"):
        w = normal(rows, cols) * sigma
        return (w.to(torch.float16) if type_name == "f16" else w).contiguous().view(torch.uint8).reshape(-1)
    qk, bb = BLOCK[type_name]
    n = rows * (cols // qk)
    blk = torch.randint(-(2 ** 31), 2 ** 31 - 1, ((n * bb + 3) // 4,), dtype=torch.int32, generator=gen, device="cuda")
    blk = blk.view(torch.uint8)[:n * bb].view(n, bb)
    if type_name == "q8_0":
        blk[:, 0:2] = halves(normal(n, 1).abs() * (sigma / 73.3))
    elif type_name == "q4_0":
        blk[:, 0:2] = halves(normal(n, 1) * (sigma / 4.64))
    elif type_name == "q5_0":
        blk[:, 0:2] = halves(normal(n, 1) * (sigma / 9.25))
    elif type_name == "q5_1":
        d = normal(n, 1) * (sigma / 9.23)
        blk[:, 0:4] = halves(torch.cat([d, -15.5 * d], dim=1))
    elif type_name == "q4_k":
        d = normal(n, 1).abs() * (sigma / 258.0)
        blk[:, 0:4] = halves(torch.cat([d, 7.5 * d], dim=1))
    else:
        blk[:, 192:208] = torch.randint(-32, 32, (n, 16), dtype=torch.int8, generator=gen, device="cuda").view(torch.uint8)
        blk[:, 208:210] = halves(normal(n, 1).abs() * (sigma / 341.0))
    return blk.reshape(-1)


_gpu_handle = None


def _gpu():
    """The program's executor: one for all its matrices."""
    global _gpu_handle
    if _gpu_handle is None:
        _gpu_handle = pkg.HipGemv(0)
    return _gpu_handle


def _upload(type_name, rows, cols, gen, tokens):
    w = _packed(type_name, rows, cols, gen)
    torch.cuda.synchronize()  # the executor reads the bytes on a stream of its own
    m = _gpu().upload_packed_device(TYPES[type_name], rows, cols, w.data_ptr(), w.numel())
    _gpu().prepare(m, tokens)
    return m


def _gguf(c, gen):
    """A model file in memory: llama architecture, dense or routed feed-forward."""
    width, ff, layers, vocab = c["width"], c["ff"], c["layers"], c["vocab"]
    heads, kv = c["heads"], c["width"] // c["heads"] * c["heads_kv"]
    experts = c.get("experts", 0)
    tensors = []  # name, type, shape (columns first), bytes

    def mat(name, type_name, rows, cols, parts=1, sigma=0.02):
        tensors.append((name, TYPES[type_name], [cols, rows] + ([parts] if parts > 1 else []), _packed(type_name, rows * parts, cols, gen, sigma)))

    def norm(name):
        w = 1.0 + 0.05 * torch.randn(width, generator=gen, device="cuda")
        tensors.append((name, 0, [width], w.view(torch.uint8)))

    mat("token_embd.weight", c["type"], vocab, width)
    for i in range(layers):
        p = "blk.%d." % i
        norm(p + "attn_norm.weight")
        for name, rows in (("attn_q", width), ("attn_k", kv), ("attn_v", kv), ("attn_output", width)):
            mat(p + name + ".weight", c["type"], rows, width)
        norm(p + "ffn_norm.weight")
        if experts:
            mat(p + "ffn_gate_inp.weight", "f32", experts, width, sigma=1.0 / math.sqrt(width))
        tail = ("_exps", experts) if experts else ("", 1)
        for name, rows, cols in (("ffn_gate", ff, width), ("ffn_up", ff, width), ("ffn_down", width, ff)):
            mat(p + name + tail[0] + ".weight", c["type"], rows, cols, tail[1])
    norm("output_norm.weight")
    mat("output.weight", "q6_k", vocab, width)

    def text(s):
        return struct.pack("<Q", len(s)) + s.encode()

    numbers = [("block_count", layers), ("embedding_length", width), ("feed_forward_length", ff), ("attention.head_count", heads),
               ("attention.head_count_kv", c["heads_kv"])]
    if experts:
        numbers += [("expert_count", experts), ("expert_used_count", c["used"])]
    kvs = [text("general.architecture") + struct.pack("<I", 8) + text("llama")]
    kvs += [text("llama." + k) + struct.pack("<II", 4, v) for k, v in numbers]
    kvs += [text("llama.rope.freq_base") + struct.pack("<If", 6, 5e5)]
    head = b"GGUF" + struct.pack("<IQQ", 3, len(tensors), len(kvs)) + b"".join(kvs)
    at, places = 0, []
    for name, ty, shape, data in tensors:
        head += text(name) + struct.pack("<I", len(shape)) + struct.pack("<%dQ" % len(shape), *shape) + struct.pack("<IQ", ty, at)
        places.append(at)
        at += (data.numel() + 31) // 32 * 32
    start = (len(head) + 31) // 32 * 32
    blob = np.zeros(start + at, np.uint8)
    blob[:len(head)] = np.frombuffer(head, np.uint8)
    for (_, _, _, data), place in zip(tensors, places):
        torch.from_numpy(blob[start + place:start + place + data.numel()]).copy_(data)
    return blob


def _step_products(c):
    """(name, rows, cols, which vector it reads) of a layer."""
    d, kv, ff = c["width"], c["kv"], c["ff"]
    return [("q", d, d, "h1"), ("k", kv, d, "h1"), ("v", kv, d, "h1"), ("o", d, d, "attn"), ("gate", ff, d, "h2"),
            ("up", ff, d, "h2"), ("down", d, ff, "act")]


class _Step:
    """A token's products as one graph on a stream of its own."""

    def __init__(self, c, gen):
        x = {k: torch.randn(n, generator=gen, device="cuda") for k, n in (("h1", c["width"]), ("attn", c["width"]), ("h2", c["width"]), ("act", c["ff"]))}
        self.x, self.y, self.mats = x, {}, []
        xs, ys = [], []
        for name, rows, _, _ in _step_products(c):
            self.y[name] = torch.zeros(c["layers"], rows, device="cuda")
        self.y["head"] = torch.zeros(c["vocab"], device="cuda")
        for layer in range(c["layers"]):
            for name, rows, cols, src in _step_products(c):
                self.mats.append(_upload(c["type"], rows, cols, gen, 1))
                xs.append(x[src].data_ptr())
                ys.append(self.y[name][layer].data_ptr())
        self.mats.append(_upload(c["head"], c["vocab"], c["width"], gen, 1))
        xs.append(x["h1"].data_ptr())
        ys.append(self.y["head"].data_ptr())
        batch = _gpu().make_batch(self.mats, [1] * len(self.mats), xs, ys)
        torch.cuda.synchronize()
        self.stream = hip.Stream()
        _gpu().gemm_batch_device(batch, self.stream.ptr)
        self.stream.synchronize()
        self.graph = hip.Graph(self.stream, lambda s: _gpu().gemm_batch_device(batch, s.ptr))

    def __del__(self):
        if hasattr(self, "graph"):
            self.stream.synchronize()
            self.graph.destroy()
            self.stream.destroy()


def prepare(case, seed):
    c = case
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    rng = np.random.default_rng(seed)
    s = {"case": c}
    if c["kind"] == "gemm":
        s["mats"] = [_upload(c["type"], c["rows"], c["cols"], gen, c["tokens"]) for _ in range(c["layers"])]
        s["x"] = torch.randn(c["layers"], c["tokens"], c["cols"], generator=gen, device="cuda")
        s["y"] = torch.zeros(c["layers"], c["tokens"], c["rows"], device="cuda")
        s["calls"] = [(m, x.data_ptr(), y.data_ptr()) for m, x, y in zip(s["mats"], s["x"], s["y"])]
    elif c["kind"] == "step":
        s["step"] = _Step(c, gen)
    elif c["kind"] == "moe":
        blob = _gguf(dict(c, layers=1, heads=c["width"] // 128, heads_kv=c["width"] // 512, vocab=256), gen)
        s["model"] = llama.Llama(blob=blob)
        s["x"] = rng.standard_normal((c["tokens"], c["width"]), np.float32)
        s["model"].moe_ffn(0, rng.standard_normal((max(64, c["tokens"]), c["width"]), np.float32))  # every expert resident
    elif c["kind"] == "dispatch":
        s["w"] = [_packed(c["type"], c["rows"], c["cols"], gen).cpu().numpy() for _ in range(c["layers"])]
        s["x"] = rng.standard_normal((c["layers"], c["tokens"] * c["cols"]), np.float32)
        s["y"] = np.zeros((c["layers"], c["tokens"] * c["rows"]), np.float32)
    else:
        s["model"] = llama.Llama(blob=_gguf(c, gen))
        n, positions = c["sequences"], c["prompt"] + c["new"] + 1
        if c["session"] == "batch":
            lengths = rng.integers((c["prompt"] + 1) // 2, c["prompt"] + 1, n)
            s["prompts"] = [rng.integers(0, c["vocab"], k).astype(np.uint32) for k in lengths]
            s["session"] = s["model"].batch_session(n, positions)
        else:
            first = rng.integers(0, c["vocab"])
            s["prompts"] = [rng.integers(0, c["vocab"], c["prompt"]).astype(np.uint32) for _ in range(2)]
            s["prompts"][0][0], s["prompts"][1][0] = first, (first + 1) % c["vocab"]  # different requests from their first token on
            s["session"] = s["model"].session(device_positions=positions if c["session"] == "device" else None)
            if c["session"] == "host":  # uploads what is not resident yet
                s["session"].forward(rng.integers(0, c["vocab"], 4))
    return s


def run(state):
    s, c = state, state["case"]
    if c["kind"] == "gemm":
        gpu, tokens = _gpu(), c["tokens"]
        for m, x, y in s["calls"]:
            gpu.gemm_device(m, tokens, x, y)
        return s["y"]
    if c["kind"] == "step":
        s["step"].graph.launch()
        return s["step"].y
    if c["kind"] == "moe":
        return s["model"].moe_ffn(0, s["x"])
    if c["kind"] == "dispatch":
        for w, x, y in zip(s["w"], s["x"], s["y"]):
            if c["tokens"] == 1:
                pkg.gemv(TYPES[c["type"]], c["cols"], w, x, y)
            else:
                pkg.gemm(TYPES[c["type"]], c["cols"], c["tokens"], w, x, y)
        return s["y"]
    if c["session"] == "batch":
        tokens, _, _ = s["session"].generate_greedy(s["prompts"], c["new"])
        return tokens.astype(np.int64)
    out = []
    for prompt in s["prompts"]:
        logits, _ = s["session"].prompt(prompt)
        tokens, _, _ = s["session"].generate_greedy([llama.argmax(logits)], c["new"])
        out.append((logits, tokens.astype(np.int64)))
    return out


def work(case):
    c = case

    def weights(type_name, *shapes):
        return sum(r * _row_bytes(type_name, k) for r, k in shapes), sum(r * k for r, k in shapes)

    if c["kind"] in ("gemm", "dispatch"):
        size, n = weights(c["type"], (c["rows"], c["cols"]))
        return {"bytes": c["layers"] * (size + 4 * c["tokens"] * (c["rows"] + c["cols"])), "flops": 2 * c["layers"] * c["tokens"] * n}
    if c["kind"] == "step":
        size, n = weights(c["type"], *[(r, k) for _, r, k, _ in _step_products(c)])
        head, n_head = weights(c["head"], (c["vocab"], c["width"]))
        vectors = sum(4 * (r + k) for _, r, k, _ in _step_products(c))
        return {"bytes": c["layers"] * (size + vectors) + head + 4 * (c["vocab"] + c["width"]), "flops": 2 * (c["layers"] * n + n_head)}
    if c["kind"] == "moe":
        size, n = weights(c["type"], (c["ff"], c["width"]), (c["ff"], c["width"]), (c["width"], c["ff"]))
        pairs = c["tokens"] * c["used"]
        return {"bytes": min(c["experts"], pairs) * size + 4 * c["experts"] * c["width"] + 8 * c["tokens"] * c["width"],
                "flops": 2 * pairs * n + 2 * c["tokens"] * c["experts"] * c["width"]}
    kv = c["width"] // c["heads"] * c["heads_kv"]
    d, ff = c["width"], c["ff"]
    size, n = weights(c["type"], (d, d), (kv, d), (kv, d), (d, d), (ff, d), (ff, d), (d, ff))
    head, n_head = weights("q6_k", (c["vocab"], d))
    if c["session"] == "batch":  # every weight once for all prompts together, then once per step
        passes, steps, rows = 1, c["new"], c["sequences"]
        prompts = rows * 3 * c["prompt"] // 4
        cache = 8 * kv * c["layers"] * rows * steps * 3 * c["prompt"] // 4
    else:  # the prompt's logits, then `new` steps, twice
        passes, steps, rows = 2, 2 * (c["new"] + 1), 1
        prompts = 2 * c["prompt"]
        cache = 8 * kv * c["layers"] * steps * c["prompt"]
    return {"bytes": (passes + steps) * c["layers"] * size + steps * head + cache,
            "flops": 2 * c["layers"] * n * (prompts + rows * steps) + 2 * n_head * rows * steps}


def tolerance(case):
    c = case
    if c["kind"] == "generate":  # f32 logits behind several layers; a token may fall to the other side of a tie
        return {"rel": 1e-4, "max": 1e-3, "differ": 0.01}
    if c["kind"] == "moe":  # three products in a row
        return {"rel": 3e-5, "max": 1e-3}
    return {"rel": 1e-5, "max": 4e-4}  # f32 sums of up to 16384 terms in another order
