"""Performance cases: the calls a program makes on this library, timed and checked.

Two levels are covered, as users reach them:

  generate      a whole greedy generation through a Session (prompt in, ids and
                the last step's logits out) on a GGUF file of a named shape;
  proj          one projection of a decode step (M = 1) through the kernel layer:
                plain, with the RMSNorm of its input, added into a residual, or
                the SwiGLU pair of an FFN;
  proj_rows     the same four for the rows of a prompt (M > 1);
  attn_decode   attention of one query over a KV cache, f16 or f32;
  attn_prompt   causal attention of a run of prompt positions over an f16 cache.

Weights are GGUF blocks in the formats that model files are stored in: Q4_0 and
Q8_0, the K-quants that the usual mixes are made of (Q4_K, Q5_K, Q6_K) and F16.
"""
from __future__ import annotations

import ctypes
import dataclasses
import math
import os
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "universal-ai-inference_amd"))
import uaii_amd  # noqa: E402
from uaii_amd import synth  # noqa: E402

GGUF_TYPE = {"q4_0": uaii_amd.Q4_0, "q8_0": uaii_amd.Q8_0, "q4_k": uaii_amd.Q4_K, "q5_k": uaii_amd.Q5_K,
             "q6_k": uaii_amd.Q6_K, "f16": uaii_amd.F16}
# values per block and bytes per block of the file format
BLOCK = {"q4_0": (32, 18), "q8_0": (32, 34), "q4_k": (256, 144), "q5_k": (256, 176), "q6_k": (256, 210),
         "f16": (1, 2)}
EPS = 1e-5


# ---- the cases ---------------------------------------------------------------------------


def listed():
    return [
        # gate and up of the smallest configured model: little more than the call and the launch
        {"name": "proj_small_q8_0", "kind": "proj", "fmt": "q8_0", "op": "swiglu", "n": 1408, "k": 512},
        # the gate and up projections of an 8B layer, the largest weights of a decode step's layer
        {"name": "proj_gate_up_q4_0", "kind": "proj", "fmt": "q4_0", "op": "swiglu", "n": 14336, "k": 4096},
        # the down projection of an 8B layer in a 5-bit file
        {"name": "proj_down_q5_k", "kind": "proj", "fmt": "q5_k", "op": "add", "n": 4096, "k": 14336},
        # the LM head of a 1B model: tied embeddings are stored in Q6_K
        {"name": "proj_head_q6_k", "kind": "proj", "fmt": "q6_k", "op": "rmsnorm", "n": 128256, "k": 2048},
        # a prompt of a few words
        {"name": "rows_short_q8_0", "kind": "proj_rows", "fmt": "q8_0", "op": "plain", "m": 9, "n": 4096, "k": 4096},
        # a chat turn's rows on a 5-bit file
        {"name": "rows_chat_q5_k", "kind": "proj_rows", "fmt": "q5_k", "op": "rmsnorm", "m": 100, "n": 4096, "k": 4096},
        # the down projection over a batch of prompt rows
        {"name": "rows_down_q4_0", "kind": "proj_rows", "fmt": "q4_0", "op": "add", "m": 512, "n": 4096, "k": 14336},
        # gate and up of a 1B layer over a document's rows, not a multiple of any tile
        {"name": "rows_gate_up_q4_k", "kind": "proj_rows", "fmt": "q4_k", "op": "swiglu", "m": 1003, "n": 8192, "k": 2048},
        # one decode step's attention at a long context
        {"name": "attn_decode_f16", "kind": "attn_decode", "f16": True, "heads": 32, "kv": 8, "hd": 128, "keys": 4037},
        # the second thousand positions of a long prompt
        {"name": "attn_prompt", "kind": "attn_prompt", "heads": 32, "kv": 8, "hd": 128, "p0": 1024, "m": 1024},
        # a whole answer with the session's defaults (f32 cache) on a 4-bit K-quant file
        {"name": "generate_1b", "kind": "generate", "shape": "1b", "fmt": "q4_k", "f16": False, "prompt": 1000, "new": 8},
        # the same on layers of the 8B shape with the f16 cache
        {"name": "generate_8b_layers", "kind": "generate", "shape": "8b4", "fmt": "q4_0", "f16": True, "prompt": 1111, "new": 8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["proj", "proj", "proj_rows", "proj_rows", "attn_decode", "attn_prompt", "generate"])
    if kind in ("proj", "proj_rows"):
        fmt = rng.choice(sorted(BLOCK))
        # row lengths are what widths of models are: multiples of 64, of 256 in the K-quants
        unit = 256 if fmt.endswith("_k") else 64
        k = unit * max(2, round(_log(rng, 512, 14336) / unit))
        c = {"kind": kind, "fmt": fmt, "op": rng.choice(["plain", "rmsnorm", "add", "swiglu"]), "k": k}
        if kind == "proj":
            c["n"] = _log(rng, 256, min(128256, 4e8 / k))
            return c
        c["m"] = _log(rng, 2, 2048)
        c["n"] = _log(rng, 256, max(1024, min(16384, 1.6e10 / (c["m"] * k))))
        return c
    heads, kv, hd = rng.choice([(8, 8, 64), (32, 8, 64), (32, 8, 128), (32, 32, 128), (64, 8, 128)])
    if kind == "attn_decode":
        return {"kind": kind, "f16": rng.random() < 0.6, "heads": heads, "kv": kv, "hd": hd, "keys": _log(rng, 1, 16384)}
    if kind == "attn_prompt":
        m = _log(rng, 2, 2048)
        return {"kind": kind, "heads": heads, "kv": kv, "hd": hd, "p0": rng.choice([0, _log(rng, 1, 4096)]), "m": m}
    shape = rng.choice(["tiny", "1b", "8b4"])
    fmt = {"tiny": ["q8_0"], "1b": ["q4_k", "q5_k"], "8b4": ["q4_0", "q8_0"]}[shape]
    return {"kind": kind, "shape": shape, "fmt": rng.choice(fmt), "f16": rng.random() < 0.5,
            "prompt": _log(rng, 2, 1000), "new": rng.randint(1, 8)}


# ---- weights in the file format -------------------------------------------------------------


def _rand_q(gen, shape, center, sd, lo, hi):
    """Quantized values as a Gaussian weight matrix has them, as bytes."""
    x = torch.randn(shape, generator=gen, device="cuda").mul_(sd).add_(center).round_().clamp_(lo, hi)
    return x.to(torch.int16).bitwise_and_(255).to(torch.uint8)


def _rand_d(gen, shape, scale):
    """Block scales (f16 bits as two bytes each): blocks of Gaussian values differ by some 10 %."""
    d = torch.randn(shape, generator=gen, device="cuda").mul_(0.1).exp_().mul_(scale).half()
    return d.view(torch.uint8).reshape(*shape, 2)


def _rand_sc6(gen, nb, center):
    """Eight 6-bit values of each super-block."""
    return torch.randn(nb, 8, generator=gen, device="cuda").mul_(5).add_(center).round_().clamp_(0, 63).to(torch.uint8)


def _pack_sc6(sc, mn):
    """The 12 bytes that hold eight 6-bit scales and eight 6-bit minimums."""
    lo = torch.cat([sc[:, :4] | ((sc[:, 4:] >> 4) << 6), mn[:, :4] | ((mn[:, 4:] >> 4) << 6)], 1)
    return torch.cat([lo, (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], 1)


def make_packed(fmt, n, k, gen):
    """n rows of k values in the file's blocks; the values are about N(0, 0.02)."""
    be, bb = BLOCK[fmt]
    nb = n * k // be
    if fmt == "f16":
        w = torch.randn(n, k, generator=gen, device="cuda").mul_(0.02).half().view(torch.uint8)
    elif fmt == "q4_0":
        q = _rand_q(gen, (nb, 32), 8, 2.6, 0, 15)
        w = torch.cat([_rand_d(gen, (nb,), 0.0077), q[:, :16] | (q[:, 16:] << 4)], 1)
    elif fmt == "q8_0":
        w = torch.cat([_rand_d(gen, (nb,), 0.0004), _rand_q(gen, (nb, 32), 0, 50, -127, 127)], 1)
    elif fmt in ("q4_k", "q5_k"):
        top = 15 if fmt == "q4_k" else 31
        q = _rand_q(gen, (nb, 4, 2, 32), top / 2, top / 6, 0, top)  # 64 values: 32 low, 32 high
        sc, mn = _rand_sc6(gen, nb, 48), _rand_sc6(gen, nb, 48)
        d = 0.02 / (48 * top / 6)
        parts = [_rand_d(gen, (nb,), d), _rand_d(gen, (nb,), d * top / 2), _pack_sc6(sc, mn)]
        if fmt == "q5_k":
            bits = (q >> 4).reshape(nb, 8, 32)
            qh = torch.zeros(nb, 32, dtype=torch.uint8, device="cuda")
            for j in range(8):
                qh |= bits[:, j] << j
            parts.append(qh)
        lo = q & 15
        parts.append((lo[:, :, 0] | (lo[:, :, 1] << 4)).reshape(nb, 128))
        w = torch.cat(parts, 1)
    else:  # q6_k
        q = _rand_q(gen, (nb, 2, 4, 32), 32, 10, 0, 63)  # halves of 128 values, four runs of 32
        ql = torch.cat([(q[:, :, 0] & 15) | ((q[:, :, 2] & 15) << 4), (q[:, :, 1] & 15) | ((q[:, :, 3] & 15) << 4)], 2)
        qh = (q[:, :, 0] >> 4) | ((q[:, :, 1] >> 4) << 2) | ((q[:, :, 2] >> 4) << 4) | ((q[:, :, 3] >> 4) << 6)
        sc = _rand_q(gen, (nb, 16), 0, 60, -127, 127)
        w = torch.cat([ql.reshape(nb, 128), qh.reshape(nb, 64), sc, _rand_d(gen, (nb,), 0.02 / (60 * 10))], 1)
    return w.contiguous().reshape(n, k // be * bb)


def decode(fmt, w):
    """The values of packed rows, in 64 bits (the file format's definition)."""
    be, bb = BLOCK[fmt]
    n = w.shape[0]
    if fmt == "f16":
        return w.contiguous().view(torch.float16).double()
    b = w.reshape(-1, bb)

    def f16(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).double()

    if fmt == "q4_0":
        q = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double().sub_(8)
        return q.mul_(f16(0)).reshape(n, -1)
    if fmt == "q8_0":
        return b[:, 2:].contiguous().view(torch.int8).double().mul_(f16(0)).reshape(n, -1)
    if fmt in ("q4_k", "q5_k"):
        s = b[:, 4:16]
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double() * f16(0)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double() * f16(2)
        qs = b[:, bb - 128:].reshape(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(-1, 8, 32)
        if fmt == "q5_k":
            bit = torch.arange(8, device=b.device, dtype=torch.uint8).reshape(1, 8, 1)
            q = q | (((b[:, 16:48].reshape(-1, 1, 32) >> bit) & 1) << 4)
        return q.double().mul_(sc[:, :, None]).sub_(mn[:, :, None]).reshape(n, -1)
    ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 32)
    q = torch.stack([(ql[:, :, 0] & 15) | ((qh & 3) << 4), (ql[:, :, 1] & 15) | (((qh >> 2) & 3) << 4),
                     (ql[:, :, 0] >> 4) | (((qh >> 4) & 3) << 4), (ql[:, :, 1] >> 4) | ((qh >> 6) << 4)], 2)
    sc = b[:, 192:208].contiguous().view(torch.int8).double() * f16(208)
    return (q.double() - 32).reshape(-1, 16, 16).mul_(sc[:, :, None]).reshape(n, -1)


# ---- inputs ---------------------------------------------------------------------------------


def _gen(seed, stream):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 64 + stream)
    return g


def _rows(gen, m, k):
    """Residual-stream rows: channels of unlike size, a few of them large."""
    size = torch.randn(k, generator=gen, device="cuda").mul_(0.6).exp_()
    return torch.randn(m, k, generator=gen, device="cuda").mul_(size)


def _proj_inputs(case, seed):
    n, k, m = case["n"], case["k"], case.get("m", 1)
    out = {"w": make_packed(case["fmt"], n, k, _gen(seed, 1)), "x": _rows(_gen(seed, 2), m, k)}
    if case["op"] == "swiglu":
        out["w2"] = make_packed(case["fmt"], n, k, _gen(seed, 3))
    if case["op"] in ("rmsnorm", "swiglu"):
        out["norm"] = torch.randn(k, generator=_gen(seed, 4), device="cuda").mul_(0.2).add_(1)
    out["y"] = torch.zeros(m, n, device="cuda")
    if case["op"] == "add":
        out["y"].normal_(generator=_gen(seed, 5))
    return out


def _attn_inputs(case, seed):
    m, p0 = (1, case["keys"] - 1) if case["kind"] == "attn_decode" else (case["m"], case["p0"])
    half = case.get("f16", True)
    max_seq = (p0 + m + 511) // 512 * 512
    shape = (case["kv"], max_seq, case["hd"])
    kc = torch.zeros(shape, device="cuda", dtype=torch.float16 if half else torch.float32)
    vc = torch.zeros_like(kc)
    g = _gen(seed, 6)
    kc[:, :p0 + m] = torch.randn(shape[0], p0 + m, shape[2], generator=g, device="cuda").to(kc.dtype)
    vc[:, :p0 + m] = torch.randn(shape[0], p0 + m, shape[2], generator=g, device="cuda").to(kc.dtype)
    q = torch.randn(m, case["heads"] * case["hd"], generator=g, device="cuda").mul_(1.5)
    return q, kc, vc, max_seq, p0, m


def _model(case):
    """The GGUF file of a generate case: a configured shape in the asked format."""
    base = synth.PRESETS[{"8b4": "8b"}.get(case["shape"], case["shape"])]
    t = GGUF_TYPE[case["fmt"]]
    if case["shape"] == "1b":  # the mixes that such files are: Q6_K value and down projections
        base = dataclasses.replace(base, type_default=t, type_embd=uaii_amd.Q6_K)
    else:
        base = dataclasses.replace(base, type_default=t)
    if case["shape"] == "8b4":  # four layers; the smaller of the configured vocabularies
        base = dataclasses.replace(base, n_layers=4, vocab=synth.PRESETS["mx"].vocab)
    return synth.cached_model(base, os.path.join("/tmp", "uaii_models_%d" % os.getuid())), base


def _prompt(case, seed, vocab):
    return np.random.default_rng(seed).integers(0, vocab, case["prompt"], dtype=np.int64)


# ---- the passes ------------------------------------------------------------------------------

_ready = []


def _lib():
    L = uaii_amd.lib()
    if not _ready:
        uaii_amd.check_hip(L.uaii_hip_init(torch.cuda.current_device()), "init")
        _ready.append(True)
    return L


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def prepare(case, seed):
    L = _lib()
    if case["kind"] == "generate":
        path, cfg = _model(case)
        return {"session": uaii_amd.Session(path, kv_f16=case["f16"]), "prompt": _prompt(case, seed, cfg.vocab),
                "new": case["new"]}
    if case["kind"] in ("proj", "proj_rows"):
        t = _proj_inputs(case, seed)
        w = [uaii_amd.DeviceWeight(GGUF_TYPE[case["fmt"]], t[x].cpu().numpy(), case["n"], case["k"])
             for x in ("w", "w2") if x in t]
        rows = [ctypes.c_int64(case["m"])] if case["kind"] == "proj_rows" else []
        args = [x.h for x in w] + [_p(t["x"])] + rows
        norm, eps = _p(t["norm"]) if "norm" in t else None, ctypes.c_float(EPS)
        args += [] if case["op"] == "plain" else [norm, eps]
        name = ("uaii_hip_gemm" if rows else "uaii_hip_gemv") + ("" if case["op"] == "plain" else "_" + case["op"])
        torch.cuda.synchronize()
        return {"call": getattr(L, name), "args": args + [_p(t["y"]), None], "out": t["y"],
                "keep": (w, t["x"], t.get("norm"))}
    q, kc, vc, max_seq, p0, m = _attn_inputs(case, seed)
    out = torch.zeros_like(q)
    i64 = ctypes.c_int64
    heads = [case["heads"], case["kv"], case["hd"]]
    if case["kind"] == "attn_decode":
        call, args = L.uaii_hip_attention_decode, [int(case["f16"]), i64(max_seq), *heads, i64(case["keys"])]
    else:
        call, args = L.uaii_hip_attention_prefill, [i64(max_seq), *heads, i64(p0), i64(m)]
    return {"call": call, "args": [_p(q), _p(kc), _p(vc), *args, _p(out), None], "out": out, "keep": (q, kc, vc)}


def run(state):
    if "session" in state:
        ids = state["session"].generate(state["prompt"], state["new"])
        return {"ids": ids, "logits": state["session"].get("logits")}
    rc = state["call"](*state["args"])
    if rc:
        uaii_amd.check_hip(rc, "run")
    return state["out"]


# ---- what a pass cannot do without -------------------------------------------------------------


def _weight_bytes(fmt, n, k):
    be, bb = BLOCK[fmt]
    return n * k // be * bb


def work(case):
    if case["kind"] in ("proj", "proj_rows"):
        n, k, m = case["n"], case["k"], case.get("m", 1)
        mats = 2 if case["op"] == "swiglu" else 1
        out = m * n * 4 * (2 if case["op"] == "add" else 1)
        return {"bytes": mats * _weight_bytes(case["fmt"], n, k) + 4 * m * k + out, "flops": 2 * mats * m * n * k}
    if case["kind"] in ("attn_decode", "attn_prompt"):
        m, p0 = (1, case["keys"] - 1) if case["kind"] == "attn_decode" else (case["m"], case["p0"])
        pairs = m * p0 + m * (m + 1) // 2
        kv = 2 * (p0 + m) * case["kv"] * case["hd"] * (2 if case.get("f16", True) else 4)
        return {"bytes": kv + 8 * m * case["heads"] * case["hd"], "flops": 4 * pairs * case["heads"] * case["hd"]}
    cfg = _config(case)
    kvd = cfg.n_kv_heads * (cfg.dim // cfg.n_heads)
    mats = {case["fmt"]: 2 * cfg.dim * cfg.dim + cfg.dim * kvd + 2 * cfg.dim * cfg.ffn}
    mixed = "q6_k" if case["shape"] == "1b" else case["fmt"]
    mats[mixed] = mats.get(mixed, 0) + cfg.dim * kvd + cfg.dim * cfg.ffn
    layer = sum(_weight_bytes(f, 1, c) for f, c in mats.items())
    head = _weight_bytes(mixed, cfg.vocab, cfg.dim)
    tokens = case["prompt"] + case["new"] - 1
    kv = 2 * kvd * (2 if case["f16"] else 4)  # bytes of one position of a layer's cache
    step_kv = sum(range(case["prompt"], tokens + 1)) * kv
    params = sum(mats.values())
    pairs = tokens * (tokens + 1) // 2
    # the prompt reads the layers once (its last position may ride along), each later step once more
    return {"bytes": case["new"] * (cfg.n_layers * layer + head) + cfg.n_layers * (step_kv + tokens * kv) + 4 * cfg.vocab,
            "flops": 2 * tokens * cfg.n_layers * params + 2 * case["new"] * cfg.vocab * cfg.dim
            + 4 * cfg.n_layers * pairs * cfg.dim}


def _config(case):
    base = synth.PRESETS[{"8b4": "8b"}.get(case["shape"], case["shape"])]
    return dataclasses.replace(base, n_layers=4, vocab=synth.PRESETS["mx"].vocab) if case["shape"] == "8b4" else base


def tolerance(case):
    if case["kind"] == "generate":
        # f32 activations and sums throughout; an f16 cache rounds keys and values, and a
        # last-bit difference before that rounding becomes one of 5e-4 in that element
        # (measured against 64 bits: 3.8e-5 with the f16 cache, 2.1e-6 with the f32 one)
        return {"rel": 1.5e-4 if case["f16"] else 1e-5, "max": 1e-2 if case["f16"] else 1e-4, "differ": 0.01}
    # 32-bit inputs and sums: up to 5.6e-7 from the 64-bit result over all of these
    return {"rel": 2.5e-6, "max": 5e-5}


# ---- the same in 64 bits -----------------------------------------------------------------------


def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + float(np.float32(EPS))) * w


def _attend(q, k, v, first):
    """q [m, heads, hd] at positions first.. over k, v [keys, kv, hd], causal."""
    m, heads, hd = q.shape
    g = heads // k.shape[1]
    out = torch.empty_like(q)
    mask = torch.arange(k.shape[0], device=q.device)[None, :] > torch.arange(m, device=q.device)[:, None] + first
    for h in range(heads):
        s = (q[:, h] @ k[:, h // g].T) / math.sqrt(hd)
        out[:, h] = torch.softmax(s.masked_fill_(mask, -math.inf), -1) @ v[:, h // g]
    return out


def exact(case, seed):
    if case["kind"] == "generate":
        return _exact_generate(case, seed)
    if case["kind"] in ("proj", "proj_rows"):
        t = _proj_inputs(case, seed)
        x = t["x"].double()
        if "norm" in t:
            x = _rms(x, t["norm"].double())
        y = x @ decode(case["fmt"], t["w"]).T
        if case["op"] == "swiglu":
            y = torch.nn.functional.silu(y) * (x @ decode(case["fmt"], t["w2"]).T)
        return y + t["y"].double() if case["op"] == "add" else y
    q, kc, vc, _, p0, m = _attn_inputs(case, seed)
    kc, vc = (c[:, :p0 + m].double().transpose(0, 1) for c in (kc, vc))
    return _attend(q.double().view(m, case["heads"], case["hd"]), kc, vc, p0).reshape(m, -1)


def _read_gguf(path):
    """{name: (format, rows, the packed bytes of its rows)} of a GGUF file's tensors."""
    data = np.memmap(path, dtype=np.uint8, mode="r")
    at = 8

    def num(kind, size):
        nonlocal at
        v = data[at:at + size].view(kind)[0]
        at += size
        return int(v)

    def text():
        nonlocal at
        n = num("<u8", 8)
        at += n
        return bytes(data[at - n:at]).decode()

    tensors, keys = num("<u8", 8), num("<u8", 8)
    for _ in range(keys):
        text()
        kind = num("<u4", 4)
        if kind == 8:
            text()
        else:  # the other kinds that these files hold are 32-bit numbers
            num("<u4", 4)
    infos = []
    for _ in range(tensors):
        name = text()
        dims = [num("<u8", 8) for _ in range(num("<u4", 4))]
        infos.append((name, dims, num("<u4", 4), num("<u8", 8)))
    base = (at + 31) // 32 * 32
    names = {v: f for f, v in GGUF_TYPE.items()}
    out = {}
    for name, dims, kind, offset in infos:
        rows = int(np.prod(dims[1:])) if len(dims) > 1 else 1
        fmt = names.get(kind, "f32")
        be, bb = BLOCK.get(fmt, (1, 4))
        nbytes = rows * (dims[0] // be * bb)
        out[name] = (fmt, rows, data[base + offset:base + offset + nbytes])
    return out


def _exact_generate(case, seed):
    path, cfg = _model(case)
    file = _read_gguf(path)
    hd = cfg.dim // cfg.n_heads

    def weight(name, rows=None):
        fmt, n, raw = file[name]
        if fmt == "f32":
            return torch.from_numpy(raw.view("<f4").copy()).cuda().double()
        raw = raw.reshape(n, -1)
        return decode(fmt, torch.from_numpy(np.ascontiguousarray(raw if rows is None else raw[rows])).cuda())

    # rotation angles in 32 bits, as the reference defines them
    freq = np.float32(1) / np.power(float(np.float32(cfg.rope_theta)),
                                    (np.arange(0, hd, 2, dtype=np.float32) / np.float32(hd)).astype(np.float64)
                                    ).astype(np.float32)

    def rope(x, first):
        ang = np.arange(first, first + x.shape[0], dtype=np.float32)[:, None] * freq[None, :]
        ang = torch.from_numpy(ang).cuda().double()[:, None, :]
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * ang.cos() - b * ang.sin(), a * ang.sin() + b * ang.cos()], -1).flatten(-2)

    def cached(x):
        return x.float().half().double() if case["f16"] else x

    layers = []
    for i in range(cfg.n_layers):
        layers.append({n: weight("blk.%d.%s.weight" % (i, n)) for n in
                       ("attn_norm", "attn_q", "attn_k", "attn_v", "attn_output", "ffn_norm", "ffn_gate", "ffn_up",
                        "ffn_down")})
    norm, head = weight("output_norm.weight"), weight("token_embd.weight" if cfg.tied else "output.weight")
    cache = [[None, None] for _ in layers]
    tokens, first, logits = _prompt(case, seed, cfg.vocab), 0, None
    for _ in range(case["new"]):
        x = weight("token_embd.weight", tokens)
        m = x.shape[0]
        for w, kv in zip(layers, cache):
            h = _rms(x, w["attn_norm"])
            q = rope((h @ w["attn_q"].T).view(m, -1, hd), first)
            new = (cached(rope((h @ w["attn_k"].T).view(m, -1, hd), first)), cached((h @ w["attn_v"].T).view(m, -1, hd)))
            for j in range(2):
                kv[j] = new[j] if kv[j] is None else torch.cat([kv[j], new[j]])
            x = x + _attend(q, kv[0], kv[1], first).reshape(m, -1) @ w["attn_output"].T
            h = _rms(x, w["ffn_norm"])
            x = x + (torch.nn.functional.silu(h @ w["ffn_gate"].T) * (h @ w["ffn_up"].T)) @ w["ffn_down"].T
        first += m
        logits = _rms(x[-1:], norm) @ head.T
        tokens = logits.argmax(-1).cpu().numpy()
    return {"ids": None, "logits": logits.reshape(-1)}
