"""What is timed: the work a bc-infer stage gives this library, one public call or one
block of them a case, over the shapes the repository's configurations, tests and benchmark
name (Qwen2.5-0.5B, Llama-3-8B, Qwen2.5-7B, the Llama-3-70B share) and the sizes between.

A case's `kind` says which part of a stage it is:
  step    one token's attention through `layers` layers (bchip_rope_append_attention): the
          decode loop, at short and long contexts, over both cache types.
  prompt  one layer's causal attention of a whole prompt, or of a later piece of one
          (bchip_attention with rows >= 16).
  verify  a speculative verify pass of a line of draft rows through `layers` layers
          (bchip_rope_append_attention_rows).
  tree    the same of a tree of draft tokens (bchip_rope_append, bchip_attention with masks).
  ragged  one decode step of several conversations in one cache pool
          (bchip_rope_append_attention_ragged).
  mlp     a layer's feed-forward block over ggml weights: norm, gate and up products,
          SiLU-mul, down product, residual add; n = 1 is decode, 2 .. 16 a verify pass,
          more a prompt.
  sample  the pick of the next token from a batch of score rows (bchip_sample).
  model   GpuLayers.forward and logits, host states in, scores out: a stage as the host
          program drives it.

Inputs come from torch on the GPU; a torch tensor's address is a device pointer like any
other to the library. Calls run on the context's stream, as a caller of the C ABI has it."""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.getcwd(), "borrowed-compute_amd"))
import bchip  # noqa: E402
from layers import Config, GpuLayers, Matrix, inv_freq  # noqa: E402

# (query heads, KV heads, head dim, neox pairs, rope base) of the attention shapes.
SHAPES = {"qwen05b": (14, 2, 64, True, 1e6), "llama8b": (32, 8, 128, False, 5e5),
          "qwen7b": (28, 4, 128, True, 1e6), "llama70b": (64, 8, 128, False, 5e5)}
# (hidden, feed-forward) of the same models.
FFN = {"qwen05b": (896, 4864), "llama8b": (4096, 14336), "qwen7b": (3584, 18944), "llama70b": (8192, 28672)}
# ggml types: number, weights a block, bytes a block.
TYPES = {"F16": (1, 1, 2), "Q4_0": (2, 32, 18), "Q8_0": (8, 32, 34), "Q4K": (12, 256, 144), "Q5K": (13, 256, 176),
         "Q6K": (14, 256, 210), "BF16": (30, 1, 2)}
MODEL_VOCAB = 32768

_ctx = None


def ctx():
    """The program's one context, made once."""
    global _ctx
    if _ctx is None:
        _ctx = bchip.Ctx(0)
    return _ctx


def listed():
    return [
        # The decode loop at the longest context, f16 cache.
        {"name": "step_llama8b_f16_32768", "kind": "step", "shape": "llama8b", "kv": "f16", "slots": 32768, "layers": 8},
        # The same over the reference's f32 cache (what an unmodified binding runs), an ordinary context.
        {"name": "step_llama8b_f32_6001", "kind": "step", "shape": "llama8b", "kv": "f32", "slots": 6001, "layers": 8},
        # A long prompt at once.
        {"name": "prompt_llama8b_f16_4096", "kind": "prompt", "shape": "llama8b", "kv": "f16", "rows": 4096, "pos": 0},
        # A piece of a prompt after some history, f32 cache, odd sizes.
        {"name": "prompt_llama8b_f32_777", "kind": "prompt", "shape": "llama8b", "kv": "f32", "rows": 777, "pos": 300},
        # Eight draft tokens verified by the 70B share.
        {"name": "verify_llama70b_f16_8", "kind": "verify", "shape": "llama70b", "kv": "f16", "rows": 8, "pos": 5003, "layers": 8},
        # A tree of draft tokens.
        {"name": "tree_llama70b_f16_33", "kind": "tree", "shape": "llama70b", "kv": "f16", "rows": 33, "pos": 3001, "layers": 4},
        # Sixteen conversations of ragged lengths, one step.
        {"name": "ragged_qwen7b_16", "kind": "ragged", "shape": "qwen7b", "kv": "f16", "seqs": 16, "longest": 24000, "layers": 4},
        # A decode step's feed-forward block in the common 4-bit mix.
        {"name": "mlp_llama8b_q4k_1", "kind": "mlp", "ffn": "llama8b", "up": "Q4K", "down": "Q6K", "n": 1},
        # The same of a prompt.
        {"name": "mlp_llama8b_q4k_512", "kind": "mlp", "ffn": "llama8b", "up": "Q4K", "down": "Q6K", "n": 512},
        # Next tokens of a verify pass, nucleus sampling over the largest vocabulary.
        {"name": "sample_151936_4", "kind": "sample", "vocab": 151936, "rows": 4, "temperature": 0.8, "top_p": 0.95},
        # A stage as the host program drives it: one token, and a short prompt.
        {"name": "model_qwen05b_1", "kind": "model", "rows": 1, "pos": 511, "layers": 6, "type": "Q8_0"},
        {"name": "model_qwen05b_67", "kind": "model", "rows": 67, "pos": 130, "layers": 6, "type": "Q8_0"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "prompt", "prompt", "verify", "tree", "ragged", "mlp", "mlp", "mlp", "sample", "model"])
    if kind == "step":
        shape = rng.choice(list(SHAPES))
        slots = _log(rng, 64, 32768)
        return {"kind": kind, "shape": shape, "kv": rng.choice(["f16", "f32"]), "slots": slots,
                "layers": rng.randint(2, 8 if slots > 8192 else 24)}
    if kind == "prompt":
        kv = rng.choice(["f16", "f16", "f32"])
        shape = rng.choice(["qwen05b", "llama8b", "qwen7b"] if kv == "f32" else list(SHAPES))
        return {"kind": kind, "shape": shape, "kv": kv, "rows": _log(rng, 17, 3500 if kv == "f16" else 777),
                "pos": rng.choice([0, _log(rng, 10, 2000 if kv == "f16" else 300)])}
    if kind == "verify":
        return {"kind": kind, "shape": rng.choice(list(SHAPES)), "kv": rng.choice(["f16", "f16", "f32"]),
                "rows": rng.randint(2, 16), "pos": _log(rng, 100, 6100), "layers": rng.randint(2, 8)}
    if kind == "tree":
        return {"kind": kind, "shape": rng.choice(list(SHAPES)), "kv": rng.choice(["f16", "f16", "f32"]),
                "rows": rng.randint(3, 33), "pos": _log(rng, 50, 3000), "layers": rng.randint(1, 4)}
    if kind == "ragged":
        return {"kind": kind, "shape": rng.choice(["qwen7b", "llama8b"]), "kv": "f16", "seqs": rng.randint(2, 24),
                "longest": _log(rng, 200, 15000), "layers": rng.randint(2, 4)}
    if kind == "mlp":
        ffn = rng.choice(["qwen05b", "llama8b", "llama8b", "qwen7b", "llama70b"])
        n = rng.choice([1, rng.randint(2, 16), _log(rng, 17, 48 if ffn == "llama70b" else 350)])
        up = rng.choice(["F16", "Q4_0", "Q8_0", "BF16"] if ffn == "qwen05b" else list(TYPES))
        if up == "BF16":
            n = min(n, 32)
        return {"kind": kind, "ffn": ffn, "up": up,
                "down": "Q6K" if up in ("Q4K", "Q5K") and rng.random() < 0.6 else up, "n": n}
    if kind == "sample":
        return {"kind": kind, "vocab": rng.choice([32000, 128256, 151936, _log(rng, 1000, 150000)]), "rows": rng.randint(1, 4),
                "temperature": rng.choice([0.0, 0.3, 0.7, 0.8, 1.0, 1.3]), "top_p": rng.choice([0.5, 0.8, 0.9, 0.95, 1.0])}
    return {"kind": kind, "rows": rng.choice([1, _log(rng, 2, 67)]), "pos": _log(rng, 20, 511), "layers": rng.randint(2, 6),
            "type": rng.choice(["Q8_0", "Q4_0", "F16"])}


# ---- inputs, made from the seed alone -----------------------------------------------------


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1000003 + 17)
    return g


def _randn(g, *shape, scale=1.0, dtype=torch.float32):
    t = torch.empty(*shape, device="cuda", dtype=dtype)
    t.normal_(0.0, scale, generator=g)
    return t


def _kv(kv):
    return (torch.float16, bchip.F16) if kv == "f16" else (torch.float32, bchip.F32)


def _freq(hd, base):
    # The frequencies a stage keeps on the device: base^(-2i / hd), f32.
    i = np.arange(hd // 2, dtype=np.float64)
    return torch.from_numpy((base ** (-2.0 * i / hd)).astype(np.float32)).cuda()


def _weights(g, type_name, rows, cols):
    """Random ggml blocks of a matrix [rows][cols], its weights about 0.02 in size: random
    quants and 6-bit scales, the f16 scales set so."""
    _, bw, bb = TYPES[type_name]
    if type_name == "F16":
        return _randn(g, rows, cols, scale=0.02).half().view(torch.uint8).reshape(-1)
    if type_name == "BF16":
        return _randn(g, rows, cols, scale=0.02).bfloat16().view(torch.uint8).reshape(-1)
    nb = rows * (cols // bw)
    w = torch.randint(0, 256, (nb, bb), device="cuda", dtype=torch.uint8, generator=g)
    d = 0.5 + torch.rand(nb, 1, device="cuda", generator=g)

    def put(at, v):
        w[:, at:at + 2] = v.half().view(torch.uint8)

    if type_name == "Q4_0":
        put(0, d * 0.004)
    elif type_name == "Q8_0":
        put(0, d * 0.0003)
    elif type_name in ("Q4K", "Q5K"):
        put(0, d * (1.2e-4 if type_name == "Q4K" else 6e-5))
        put(2, d * (9e-4 if type_name == "Q4K" else 9e-4))
    else:  # Q6K: int8 scales 192 .. 207, d at 208
        put(208, d * 1.5e-5)
    return w.reshape(-1)


def _dequant(w, type_name, rows, cols):
    """The weights of _weights' bytes in 64 bits, by ggml's block formats."""
    if type_name == "F16":
        return w.view(torch.float16).view(rows, cols).double()
    if type_name == "BF16":
        return w.view(torch.bfloat16).view(rows, cols).double()
    _, bw, bb = TYPES[type_name]
    b = w.view(-1, bb)

    def half(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).double()

    if type_name == "Q8_0":
        v = b[:, 2:].contiguous().view(torch.int8).double() * half(0)
    elif type_name == "Q4_0":
        q = b[:, 2:18]
        v = (torch.cat([q & 15, q >> 4], 1).double() - 8.0) * half(0)
    elif type_name in ("Q4K", "Q5K"):
        s = b[:, 4:16].int()
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        qs = b[:, bb - 128:].view(-1, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32)
        if type_name == "Q5K":
            qh = b[:, 16:48].view(-1, 1, 32)
            bit = torch.arange(8, device=w.device, dtype=torch.uint8).view(1, 8, 1)
            q = q + (((qh >> bit) & 1) << 4)
        v = (q.double() * (half(0) * sc).unsqueeze(2) - (half(2) * mn).unsqueeze(2)).reshape(-1, 256)
    else:
        ql, qh, out = b[:, :128].view(-1, 2, 2, 32), b[:, 128:192].view(-1, 2, 32), []
        for h in range(2):
            for k in range(4):
                lo = (ql[:, h, k & 1] >> (4 if k >= 2 else 0)) & 15
                out.append((lo | (((qh[:, h] >> (2 * k)) & 3) << 4)).double() - 32.0)
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        v = torch.stack(out, 1).view(-1, 16, 16) * (half(208) * sc).unsqueeze(2)
    return v.reshape(rows, cols)


def _attention_inputs(case, seed):
    """q, k, v of the new rows, the caches, and what goes with them, for step, verify, tree."""
    g = _gen(seed)
    nh, nkv, hd, neox, base = SHAPES[case["shape"]]
    rows = case.get("rows", 1)
    pos = case["slots"] - 1 if case["kind"] == "step" else case["pos"]
    dt, kv_type = _kv(case["kv"])
    L, slots = case["layers"], pos + (64 if case["kind"] == "tree" else rows)
    s = {"case": case, "nh": nh, "nkv": nkv, "hd": hd, "neox": neox, "rows": rows, "pos": pos, "kv_type": kv_type,
         # Queries are larger than keys in earnest: the softmax has its peaks.
         "q0": _randn(g, L, rows, nh, hd, scale=2.0), "k": _randn(g, L, rows, nkv, hd), "v": _randn(g, L, rows, nkv, hd),
         "kc": _randn(g, L, slots, nkv * hd, dtype=dt), "vc": _randn(g, L, slots, nkv * hd, dtype=dt),
         "freq": _freq(hd, base)}
    s["q"], s["out"] = torch.empty_like(s["q0"]), torch.empty_like(s["q0"])
    if case["kind"] == "tree":
        # Each node's parent is the root or an earlier node; a row sees its ancestors and itself.
        r = np.random.default_rng(int(seed))
        depth, seen = [], []
        for i in range(rows):
            parent = int(r.integers(-1, i)) if i else -1
            seen.append((0 if parent < 0 else seen[parent]) | (1 << i))
            depth.append(0 if parent < 0 else depth[parent] + 1)
        s["seen"] = seen
        s["masks"] = torch.from_numpy(bchip.masks_words(np.array(seen, np.uint64)).view(np.int32)).cuda()
        s["positions"] = torch.tensor([pos + d for d in depth], device="cuda", dtype=torch.int32)
    else:
        s["positions"] = torch.arange(pos, pos + rows, device="cuda", dtype=torch.int32)
    return s


def _ragged_lens(case, seed):
    r = np.random.default_rng(int(seed) + 5)
    longest = case["longest"]
    lens = np.exp(r.uniform(math.log(max(32, longest // 8)), math.log(longest), case["seqs"])).astype(np.uint32)
    lens[0] = longest
    return lens


class _Model:
    """A stage's layers and head over random weights, and its cache with `pos` tokens in it."""

    def __init__(self, case, seed):
        g = _gen(seed)
        ty, (nh, nkv, hd, neox, base), (e, ff) = case["type"], SHAPES["qwen05b"], FFN["qwen05b"]
        self.cfg = Config(e, case["layers"], nh, nkv, hd, hd, base, neox, 1e-6, MODEL_VOCAB)
        num = TYPES[ty][0]
        self.norms, self.mats, layers = [], [], []

        def matrix(rows, cols):
            w = _weights(g, ty, rows, cols)
            self.mats.append((w, rows, cols))
            return Matrix(num, w.cpu().numpy().tobytes(), rows, cols)

        def vector(n, mean, scale):
            v = mean + _randn(g, n, scale=scale)
            self.norms.append(v)
            return v.cpu().numpy()

        for _ in range(case["layers"]):
            layers.append({"attn_norm": vector(e, 1.0, 0.1), "ffn_norm": vector(e, 1.0, 0.1),
                           "bq": vector(nh * hd, 0.0, 0.3), "bk": vector(nkv * hd, 0.0, 0.3), "bv": vector(nkv * hd, 0.0, 0.1),
                           "wq": matrix(nh * hd, e), "wk": matrix(nkv * hd, e), "wv": matrix(nkv * hd, e),
                           "wo": matrix(e, nh * hd), "gate": matrix(ff, e), "up": matrix(ff, e), "down": matrix(e, ff)})
        head = (vector(e, 1.0, 0.1), matrix(MODEL_VOCAB, e))
        rows, pos = case["rows"], case["pos"]
        self.x = _randn(g, rows, e).cpu().numpy()
        self.k0 = [_randn(g, pos, nkv * hd) for _ in range(case["layers"])]
        self.v0 = [_randn(g, pos, nkv * hd) for _ in range(case["layers"])]
        self.positions = np.arange(pos, pos + rows, dtype=np.uint32)
        self.layers, self.head = layers, head
        self.g = self.cache = None

    def start(self):
        c = ctx()
        self.g = GpuLayers(c, self.cfg, self.layers, self.head)
        self.cache = self.g.new_cache()
        self.cache.reserve(len(self.positions) + len(self.k0[0]), 0, self.cfg.context)
        for buf, t in zip(self.cache.k + self.cache.v, self.k0 + self.v0):
            c.copy(t.data_ptr(), bchip.F32, buf, bchip.F32, 0, t.numel())
        c.sync()
        self.layers = self.head = None
        return self

    def __del__(self):
        try:
            if self.g is not None:
                self.cache.free()
                self.g.free()
        except Exception:  # the process is ending
            pass


def _make(case, seed):
    """A case's inputs; nothing of the library is called."""
    kind = case["kind"]
    if kind in ("step", "verify", "tree"):
        return _attention_inputs(case, seed)
    g = _gen(seed)
    if kind == "prompt":
        nh, nkv, hd, _, _ = SHAPES[case["shape"]]
        dt, kv_type = _kv(case["kv"])
        rows, slots = case["rows"], case["pos"] + case["rows"]
        q = _randn(g, rows, nh, hd, scale=2.0)
        return {"case": case, "q": q, "out": torch.empty_like(q), "kc": _randn(g, slots, nkv * hd, dtype=dt),
                "vc": _randn(g, slots, nkv * hd, dtype=dt), "kv_type": kv_type, "nh": nh, "nkv": nkv, "hd": hd}
    if kind == "ragged":
        nh, nkv, hd, neox, base = SHAPES[case["shape"]]
        dt, kv_type = _kv(case["kv"])
        lens, L, n = _ragged_lens(case, seed), case["layers"], case["seqs"]
        offs = np.concatenate([[0], np.cumsum(lens.astype(np.uint64))])[:-1].astype(np.uint64)
        total = int(lens.sum())
        s = {"case": case, "nh": nh, "nkv": nkv, "hd": hd, "neox": neox, "kv_type": kv_type, "lens": lens, "offs": offs,
             "q0": _randn(g, L, n, nh, hd, scale=2.0), "k": _randn(g, L, n, nkv, hd), "v": _randn(g, L, n, nkv, hd),
             "kc": _randn(g, L, total, nkv * hd, dtype=dt), "vc": _randn(g, L, total, nkv * hd, dtype=dt),
             "freq": _freq(hd, base), "positions": torch.from_numpy(lens.astype(np.int32) - 1).cuda()}
        s["q"], s["out"] = torch.empty_like(s["q0"]), torch.empty_like(s["q0"])
        return s
    if kind == "mlp":
        (e, ff), n = FFN[case["ffn"]], case["n"]
        f = lambda *d: torch.empty(*d, device="cuda")
        return {"case": case, "x": _randn(g, n, e), "norm": 1.0 + _randn(g, e, scale=0.1),
                "gate": _weights(g, case["up"], ff, e), "up": _weights(g, case["up"], ff, e),
                "down": _weights(g, case["down"], e, ff), "n": f(n, e), "g": f(n, ff), "u": f(n, ff), "o": f(n, e)}
    if kind == "sample":
        # Most of a vocabulary is unlikely; a few dozen tokens hold most of the mass.
        s = _randn(g, case["rows"], case["vocab"], scale=2.0)
        top = torch.randint(0, case["vocab"], (case["rows"], 32), device="cuda", generator=g)
        s.scatter_add_(1, top, 4.0 + 8.0 * torch.rand(case["rows"], 32, device="cuda", generator=g))
        return {"case": case, "scores": s, "ids": torch.empty(case["rows"], device="cuda", dtype=torch.int32), "seed": int(seed)}
    return _Model(case, seed)


def prepare(case, seed):
    c = ctx()
    s = _make(case, seed)
    torch.cuda.synchronize()  # the library's stream does not wait for torch's
    if case["kind"] == "model":
        return s.start()
    s["ctx"] = c
    return s


# ---- one pass -----------------------------------------------------------------------------


def run(s):
    if isinstance(s, _Model):
        x = s.g.forward(s.x, len(s.k0[0]), s.positions, None, s.cache)
        return {"states": x, "logits": s.g.logits(x, len(s.positions))}
    return _RUN[s["case"]["kind"]](s, s["ctx"])


def _run_step(s, c):
    p, nh, nkv, hd = s["q"].data_ptr, s["nh"], s["nkv"], s["hd"]
    c.copy(s["q0"].data_ptr(), bchip.F32, p(), bchip.F32, 0, s["q0"].numel())  # the layers' q products' place
    scale, rows, pos, kind = 1.0 / math.sqrt(hd), s["rows"], s["pos"], s["case"]["kind"]
    freq, positions = s["freq"].data_ptr(), s["positions"].data_ptr()
    a = [s[k] for k in ("q", "k", "v", "kc", "vc", "out")]
    at, by = [t.data_ptr() for t in a], [t.stride(0) * t.element_size() for t in a]
    for l in range(s["case"]["layers"]):
        q, k, v, kc, vc, out = [x + l * y for x, y in zip(at, by)]
        if kind == "step":
            c.rope_append_attention(q, k, v, kc, vc, s["kv_type"], freq, positions, nh, nkv, hd, hd, s["neox"], pos, scale, out)
        elif kind == "verify":
            c.rope_append_attention_rows(q, k, v, kc, vc, s["kv_type"], freq, positions, rows, nh, nkv, hd, hd, s["neox"], pos,
                                         scale, out)
        else:
            c.rope_append(q, k, v, kc, vc, s["kv_type"], freq, positions, rows, nh, nkv, hd, hd, s["neox"], pos)
            c.attention(q, kc, vc, s["kv_type"], out, s["masks"].data_ptr(), True, rows, nh, nkv, hd, pos, scale)
    # The caches are left as they were but for the new rows.
    return {"out": s["out"], "q": s["q"], "k": s["kc"][:, pos:pos + rows], "v": s["vc"][:, pos:pos + rows]}


def _run_prompt(s, c):
    c.attention(s["q"].data_ptr(), s["kc"].data_ptr(), s["vc"].data_ptr(), s["kv_type"], s["out"].data_ptr(), None, False,
                s["case"]["rows"], s["nh"], s["nkv"], s["hd"], s["case"]["pos"], 1.0 / math.sqrt(s["hd"]))
    return {"out": s["out"]}


def _run_ragged(s, c):
    c.copy(s["q0"].data_ptr(), bchip.F32, s["q"].data_ptr(), bchip.F32, 0, s["q0"].numel())
    a = [s[k] for k in ("q", "k", "v", "kc", "vc", "out")]
    at, by = [t.data_ptr() for t in a], [t.stride(0) * t.element_size() for t in a]
    for l in range(s["case"]["layers"]):
        q, k, v, kc, vc, out = [x + l * y for x, y in zip(at, by)]
        c.rope_append_attention_ragged(q, k, v, kc, vc, s["kv_type"], s["freq"].data_ptr(), s["positions"].data_ptr(), s["lens"],
                                       s["offs"], s["nh"], s["nkv"], s["hd"], s["hd"], s["neox"], 1.0 / math.sqrt(s["hd"]), out)
    return {"out": s["out"], "q": s["q"]}


def _run_mlp(s, c):
    case = s["case"]
    (e, ff), n = FFN[case["ffn"]], case["n"]
    up, down = TYPES[case["up"]][0], TYPES[case["down"]][0]
    x, nb, g, u, o = (s[k].data_ptr() for k in ("x", "n", "g", "u", "o"))
    c.rms_norm(x, s["norm"].data_ptr(), nb, n, e, 1e-5)
    c.matmul(s["gate"].data_ptr(), up, nb, g, ff, e, n)
    c.matmul(s["up"].data_ptr(), up, nb, u, ff, e, n)
    c.silu_mul(g, u, n * ff)
    c.matmul(s["down"].data_ptr(), down, g, o, e, ff, n)
    c.add(o, x, n * e)
    return {"x": s["o"], "hidden": s["g"]}


def _run_sample(s, c):
    case = s["case"]
    c.sample(s["scores"].data_ptr(), case["rows"], case["vocab"], case["temperature"], case["top_p"], s["seed"], 100,
             s["ids"].data_ptr())
    return {"ids": s["ids"]}


_RUN = {"step": _run_step, "verify": _run_step, "tree": _run_step, "prompt": _run_prompt, "ragged": _run_ragged, "mlp": _run_mlp,
        "sample": _run_sample}


# ---- what a pass cannot do without --------------------------------------------------------


def _attn_work(nh, nkv, hd, eb, rows, slots, pairs):
    """One layer: q read and left rotated, the cache read once, the new rows written, out;
    scores and weighted values of every visible pair."""
    kvd = nkv * hd
    return {"bytes": 2.0 * slots * kvd * eb + rows * (3 * nh * hd * 4 + 2 * kvd * (4 + eb)), "flops": 4.0 * nh * hd * pairs}


def _mat_bytes(type_name, rows, cols):
    _, bw, bb = TYPES[type_name]
    return float(rows) * cols / bw * bb


def work(case):
    kind = case["kind"]
    if kind in ("step", "verify", "tree"):
        nh, nkv, hd, _, _ = SHAPES[case["shape"]]
        rows = case.get("rows", 1)
        pos = case["slots"] - 1 if kind == "step" else case["pos"]
        # (A tree row sees a few of the tree's rows: about half of a line's here.)
        pairs = rows * pos + rows * (rows + 1) / (4.0 if kind == "tree" else 2.0)
        w = _attn_work(nh, nkv, hd, 2 if case["kv"] == "f16" else 4, rows, pos + rows, pairs)
        return {k: v * case["layers"] for k, v in w.items()}
    if kind == "prompt":
        nh, nkv, hd, _, _ = SHAPES[case["shape"]]
        rows, pos = case["rows"], case["pos"]
        eb = 2 if case["kv"] == "f16" else 4
        return {"bytes": 2.0 * (pos + rows) * nkv * hd * eb + 2.0 * rows * nh * hd * 4,
                "flops": 4.0 * nh * hd * (rows * pos + rows * (rows + 1) / 2.0)}
    if kind == "ragged":
        nh, nkv, hd, _, _ = SHAPES[case["shape"]]
        # The lengths spread evenly over their logarithm from longest / 8 to longest.
        total = case["longest"] + (case["seqs"] - 1) * case["longest"] * (7.0 / 8.0) / math.log(8.0)
        w = _attn_work(nh, nkv, hd, 2, case["seqs"], total, total)
        return {k: v * case["layers"] for k, v in w.items()}
    if kind == "mlp":
        (e, ff), n = FFN[case["ffn"]], case["n"]
        wb = 2 * _mat_bytes(case["up"], ff, e) + _mat_bytes(case["down"], e, ff)
        return {"bytes": wb + 4.0 * n * (3 * e) + 4.0 * n * ff, "flops": 6.0 * n * e * ff}
    if kind == "sample":
        return {"bytes": 4.0 * case["rows"] * case["vocab"], "flops": 2.0 * case["rows"] * case["vocab"]}
    (nh, nkv, hd, _, _), (e, ff), n, L = SHAPES["qwen05b"], FFN["qwen05b"], case["rows"], case["layers"]
    layer = _mat_bytes(case["type"], nh * hd + 2 * nkv * hd, e) + _mat_bytes(case["type"], e, nh * hd) + 3 * _mat_bytes(case["type"], ff, e)
    slots = case["pos"] + n
    mac = L * (e * (nh + 2 * nkv) * hd + e * nh * hd + 3 * e * ff) + MODEL_VOCAB * e
    return {"bytes": L * (layer + 2.0 * slots * nkv * hd * 4) + _mat_bytes(case["type"], MODEL_VOCAB, e) + 4.0 * n * (3 * e + MODEL_VOCAB),
            "flops": 2.0 * n * mac + L * 4.0 * nh * hd * n * (case["pos"] + n / 2.0)}


def tolerance(case):
    kind = case["kind"]
    if kind == "sample":
        return "exact"
    if kind == "mlp":
        return {"rel": 1.5e-6}  # f32 sums over weights exact in their format, twice over
    if kind == "model":
        return {"rel": 2e-6}  # f32 throughout, several layers
    if case["kv"] == "f32":
        return {"rel": 2.5e-6}
    return {"rel": 2e-3}  # q, K, V and the softmax weights are f16 operands


# ---- the same in 64 bits ------------------------------------------------------------------


def _rotate(t, positions, freq, neox):
    """t [..., rows, heads, hd] turned by the f32 angle the operation is defined by."""
    theta = (positions.float()[:, None] * freq[None, :]).double()[:, None, :]
    cos, sin, out = theta.cos(), theta.sin(), t.double().clone()
    half = freq.numel()
    a, b = (slice(0, half), slice(half, 2 * half)) if neox else (slice(0, 2 * half, 2), slice(1, 2 * half, 2))
    x, y = t[..., a].double(), t[..., b].double()
    out[..., a], out[..., b] = x * cos - y * sin, x * sin + y * cos
    return out


def _attend(q, kc, vc, nkv, visible):
    """q [rows, nh, hd]; kc, vc [slots, nkv * hd]; visible(r0, r1) -> mask [r1 - r0, slots]."""
    rows, nh, hd = q.shape
    G, slots = nh // nkv, kc.shape[0]
    out = torch.empty(rows, nh, hd, device=q.device, dtype=torch.float64)
    step = max(1, (1 << 27) // (G * slots))
    for h in range(nkv):
        k = kc[:, h * hd:(h + 1) * hd].double()
        v = vc[:, h * hd:(h + 1) * hd].double()
        kt = k.t().contiguous()
        for r0 in range(0, rows, step):
            r1 = min(rows, r0 + step)
            x = q[r0:r1, h * G:(h + 1) * G].double().reshape(-1, hd) @ kt / math.sqrt(hd)
            x = x.view(r1 - r0, G, slots).masked_fill(~visible(r0, r1)[:, None, :], -math.inf)
            out[r0:r1, h * G:(h + 1) * G] = (torch.softmax(x, 2).view(-1, slots) @ v).view(r1 - r0, G, hd)
    return out


def _line(pos, slots):
    j = torch.arange(slots, device="cuda")
    return lambda r0, r1: j[None, :] <= (pos + torch.arange(r0, r1, device="cuda"))[:, None]


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":
        return None  # a pick by the f32 sums' own rounding, or an argmax
    s = _make(case, seed)
    if kind == "model":
        return _exact_model(case, s)
    if kind == "mlp":
        (e, ff) = FFN[case["ffn"]]
        x = s["x"].double()
        n = x / torch.sqrt((x * x).mean(1, keepdim=True) + 1e-5) * s["norm"].double()
        g = n @ _dequant(s["gate"], case["up"], ff, e).t().contiguous()
        u = n @ _dequant(s["up"], case["up"], ff, e).t().contiguous()
        h = g * torch.sigmoid(g) * u
        return {"x": x + h @ _dequant(s["down"], case["down"], e, ff).t().contiguous(), "hidden": h}
    if kind == "prompt":
        return {"out": _attend(s["q"], s["kc"], s["vc"], s["nkv"], _line(case["pos"], s["kc"].shape[0]))}
    nkv, hd, L = s["nkv"], s["hd"], case["layers"]
    q = torch.stack([_rotate(s["q0"][l], s["positions"], s["freq"], s["neox"]) for l in range(L)])
    k = torch.stack([_rotate(s["k"][l], s["positions"], s["freq"], s["neox"]) for l in range(L)])
    out = torch.empty_like(q)
    if kind == "ragged":
        for l in range(L):
            for i, (o, n) in enumerate(zip(s["offs"].astype(int), s["lens"].astype(int))):
                kc, vc = s["kc"][l, o:o + n], s["vc"][l, o:o + n]
                kc[n - 1], vc[n - 1] = k[l, i].reshape(-1).to(kc.dtype), s["v"][l, i].reshape(-1).to(vc.dtype)
                out[l, i:i + 1] = _attend(q[l, i:i + 1], kc, vc, nkv, _line(n - 1, n))
        return {"out": out, "q": q}
    rows, pos = s["rows"], s["pos"]
    if kind == "tree":
        see = torch.tensor([[(m >> j) & 1 for j in range(rows)] for m in s["seen"]], device="cuda", dtype=torch.bool)
        seen = torch.cat([torch.ones(rows, pos, device="cuda", dtype=torch.bool), see], 1)
        visible = lambda r0, r1: seen[r0:r1]
    else:
        visible = _line(pos, pos + rows)
    kn, vn = k.reshape(L, rows, -1).to(s["kc"].dtype), s["v"].reshape(L, rows, -1).to(s["vc"].dtype)
    for l in range(L):
        kc, vc = s["kc"][l, :pos + rows], s["vc"][l, :pos + rows]
        kc[pos:], vc[pos:] = kn[l], vn[l]
        out[l] = _attend(q[l], kc, vc, nkv, visible)
    keep = (lambda t: t.double()) if case["kv"] == "f16" else (lambda t: t)
    return {"out": out, "q": q, "k": keep(kn) if case["kv"] == "f16" else k.reshape(L, rows, -1),
            "v": vn.double()}


def _exact_model(case, m):
    c, pos, n = m.cfg, case["pos"], case["rows"]
    nh, nkv, hd = c.n_head, c.n_head_kv, c.head_dim
    freq = torch.from_numpy(inv_freq(c)).cuda()
    positions = torch.arange(pos, pos + n, device="cuda", dtype=torch.int32)
    mats = iter([_dequant(w, case["type"], r, k) for w, r, k in m.mats])
    vecs = iter([v.double() for v in m.norms])
    norm = lambda x, w: x / torch.sqrt((x * x).mean(1, keepdim=True) + c.eps) * w
    mul = lambda x, w: x @ w.t().contiguous()
    x = torch.from_numpy(m.x).cuda().double()
    for l in range(case["layers"]):
        an, fn, bq, bk, bv = (next(vecs) for _ in range(5))
        wq, wk, wv, wo, gate, up, down = (next(mats) for _ in range(7))
        h = norm(x, an)
        q = _rotate((mul(h, wq) + bq).view(n, nh, hd), positions, freq, c.rope_neox)
        k = _rotate((mul(h, wk) + bk).view(n, nkv, hd), positions, freq, c.rope_neox)
        kc = torch.cat([m.k0[l].double(), k.view(n, -1)])
        vc = torch.cat([m.v0[l].double(), mul(h, wv) + bv])
        x = x + mul(_attend(q, kc, vc, nkv, _line(pos, pos + n)).view(n, -1), wo)
        h = norm(x, fn)
        g = mul(h, gate)
        x = x + mul(g * torch.sigmoid(g) * mul(h, up), down)
    return {"states": x, "logits": mul(norm(x, next(vecs)), next(mats))}
