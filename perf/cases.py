"""What a program that uses this package has it compute, as measurable cases.

Each case is one call (or, for the model cases, one request batch) through a
public entry point: ``NativeOps`` (torch-facing binding of the v2 ABI), the
``ti_amd_*`` C entry points, and ``NativeModel``.  ``listed()`` gives the cases,
``draw(rng)`` another one of the same ranges, ``prepare`` its inputs, ``run`` one
pass, ``work`` the bytes and operations it cannot do without, ``tolerance`` what
another correct implementation may differ by, and ``exact`` the same outputs in
64-bit arithmetic.
"""
import ctypes
import math
import random
import tempfile

import numpy as np
import torch

from tinyinfer_amd import BACKEND_LIB, LLM_LIB
from tinyinfer_amd.artifact import GPT2_SMALL, GPT2_XL, load_tensors, write_synthetic
from tinyinfer_amd.native_ops import NativeOps
from tinyinfer_amd.runtime import NativeModel

DEV = "cuda"
VOCAB = 50257

# Model cases: GPT-2 small (12 layers), and GPT-2 XL's width (1600, 25 heads,
# MLP 6400) at two layers, which is what a layer of XL costs without writing 48.
ARCHS = {"small": dict(GPT2_SMALL), "wide": dict(GPT2_XL, layers=2)}
SLOTS = {"small": 32, "wide": 8}

EPILOGUES = {"bias": 0, "gelu": 1, "residual": 2}


def listed():
    return [
        # One token's attention input projection, weights as the reference ABI
        # keeps them: the smallest call a decode loop makes.
        {"name": "linear int8 decode b1", "op": "linear8", "m": 1, "k": 768, "n": 2304, "bias": True, "out": "f16",
         "config": 0},
        # GPT-2's tied head over a full decode batch, fp32 logits, an odd N.
        {"name": "lm head int8 b32", "op": "linear8", "m": 32, "k": 768, "n": VOCAB, "bias": False, "out": "f32",
         "config": 0},
        # GPT-2 XL's first MLP linear over a long prefill batch.
        {"name": "linear int8 prefill xl", "op": "linear8", "m": 8192, "k": 1600, "n": 6400, "bias": True,
         "out": "f16", "config": 0},
        # GPT-2 small's first MLP linear with fp16 weights over a prefill batch.
        {"name": "linear fp16 prefill", "op": "linear16", "m": 2048, "k": 768, "n": 3072, "bias": True, "out": "f16",
         "config": 0},
        # The same linear over packed weights with its GELU fused, a ragged row count.
        {"name": "packed mlp gelu", "op": "packed", "m": 500, "k": 768, "n": 3072, "epilogue": "gelu"},
        # One decode step's attention of 32 requests with ragged caches.
        {"name": "attention decode b32", "op": "attention", "batch": 32, "heads": 12, "q": 1, "kv": 1024, "dim": 64,
         "low": 128, "causal": True},
        # Prefill attention of eight full-length GPT-2 XL prompts.
        {"name": "attention prefill xl", "op": "attention", "batch": 8, "heads": 25, "q": 1024, "kv": 1024, "dim": 64,
         "low": 1024, "causal": True},
        # 128-wide heads, no causal mask, ragged and odd lengths.
        {"name": "attention d128 ragged", "op": "attention", "batch": 4, "heads": 16, "q": 333, "kv": 1500, "dim": 128,
         "low": 700, "causal": False},
        # The FP32 GEMM of the legacy ABI at the square size it is benchmarked at.
        {"name": "gemm fp32 1024", "op": "gemm32", "m": 1024, "k": 1024, "n": 1024},
        # LayerNorm of a prefill batch's residual stream at GPT-2 XL's width.
        {"name": "layernorm fp16", "op": "layernorm16", "rows": 8192, "cols": 1600},
        # A served batch: 32 ragged prompts, then token-by-token decode in which
        # the caller picks the tokens and asks for the last step's logits.
        {"name": "serve small b32", "op": "model", "arch": "small", "precision": "int8", "batch": 32, "low": 16,
         "high": 64, "steps": 12},
        # The prefill of eight long prompts at GPT-2 XL's width.
        {"name": "prefill wide b8", "op": "model", "arch": "wide", "precision": "int8", "batch": 8, "low": 128,
         "high": 512, "steps": 0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    """A case of the listed ones' ranges: the same operations over row counts from
    one token to a long prefill batch, the models' widths and odd ones."""
    op = rng.choice(("linear8", "linear8", "linear16", "linear16", "packed", "attention", "attention", "attention",
                     "gemm32", "rows", "rows", "model"))
    if op in ("linear8", "linear16", "packed"):
        m = _log(rng, 1, 8192)
        widths = (768, 1600, 2304, 3072, 4800, 6400)
        if op == "packed":  # its weights come in K chunks of 64
            k, n = rng.choice(((768, 2304), (768, 768), (768, 3072), (3072, 768), (1600, 4800), (1600, 1600),
                               (1600, 6400), (6400, 1600)))
            return {"op": op, "m": m, "k": k, "n": n if rng.random() < 0.7 else n + rng.randint(1, 63),
                    "epilogue": rng.choice(tuple(EPILOGUES))}
        k = rng.choice(widths) if rng.random() < 0.7 else _log(rng, 64, 6400)
        n = rng.choice(widths) if rng.random() < 0.7 else _log(rng, 64, 6400)
        if m <= 64 and rng.random() < 0.25:
            k, n = rng.choice((768, 1600)), VOCAB
        m = max(1, min(m, 80_000_000_000 // (k * n)))
        return {"op": op, "m": m, "k": k, "n": n, "bias": rng.random() < 0.7, "out": rng.choice(("f16", "f16", "f32")),
                "config": rng.choice((0, 0, 1, 2, 3, 6))}
    if op == "attention":
        dim, heads = rng.choice((64, 64, 128)), rng.choice((4, 12, 16, 25))
        if rng.random() < 0.4:  # decode
            batch, kv = _log(rng, 1, 64), _log(rng, 16, 4096)
            q = 1
        else:
            batch, q = _log(rng, 1, 32), _log(rng, 2, 2048)
            kv = q if rng.random() < 0.6 else min(4096, q + _log(rng, 1, 1024))
            batch = max(1, min(batch, 210_000_000 // (heads * q * kv)))
        return {"op": op, "batch": batch, "heads": heads, "q": q, "kv": kv, "dim": dim,
                "low": max(1, int(kv * rng.choice((0.1, 0.5, 1.0)))), "causal": rng.random() < 0.7}
    if op == "gemm32":
        return {"op": op, "m": _log(rng, 16, 2048), "k": _log(rng, 16, 2048), "n": _log(rng, 16, 2048)}
    if op == "rows":
        op = rng.choice(("layernorm16", "softmax16", "gelu16", "layernorm_softmax32"))
        return {"op": op, "rows": _log(rng, 1, 16384), "cols": rng.choice((768, 1024, 1600, 3072, _log(rng, 16, 4096)))}
    arch = rng.choice(("small", "small", "wide"))
    batch = _log(rng, 1, SLOTS[arch])
    high = min(_log(rng, 2, 512), (1600 if arch == "small" else 2560) // batch)
    return {"op": "model", "arch": arch, "precision": "int8", "batch": batch, "low": max(1, int(high * rng.random())),
            "high": high, "steps": rng.randint(0, 8)}


# -- what a user's program keeps ------------------------------------------------------
_kept = {}


def _keep(key, make):
    if key not in _kept:
        _kept[key] = make()
    return _kept[key]


def _ops():
    return _keep("ops", NativeOps)


def _lib():
    def make():
        lib = ctypes.CDLL(str(BACKEND_LIB))
        p, i, f, s, d = ctypes.c_void_p, ctypes.c_int, ctypes.c_float, ctypes.c_size_t, ctypes.c_int
        lib.ti_amd_packed_w8_bytes.argtypes, lib.ti_amd_packed_w8_bytes.restype = [i, i], ctypes.c_int64
        lib.ti_amd_pack_w8.argtypes = [p, i, i, p, s, d]
        lib.ti_amd_gemm_w8p_fused.argtypes = [p] * 6 + [i] * 4 + [s, d]
        lib.ti_amd_layernorm_softmax_f32.argtypes = [p] * 4 + [i, i, f, s, d]
        return lib
    return _keep("lib", make)


def _artifact(name, precision, use):
    """`use(manifest path)` on a synthetic artifact of that architecture."""
    with tempfile.TemporaryDirectory() as d:
        return use(write_synthetic(d, ARCHS[name], seed=42, precision=precision))


def _model(case):
    """One loaded model serves every request batch, as a server keeps it."""
    name, precision = case["arch"], case["precision"]
    return _keep(("model", name, precision), lambda: _artifact(
        name, precision, lambda path: NativeModel(LLM_LIB, path, max_batch=SLOTS[name], cache_slots=SLOTS[name])))


def _check(status):
    if status != 0:
        raise RuntimeError(f"status {status}")


# -- inputs ---------------------------------------------------------------------------
class _Draw:
    """Tensors of a seed: activations as a LayerNorm leaves them, weights and
    biases as GPT-2 initialises them."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed))

    def normal(self, shape, std=1.0, dtype=torch.float16, mean=0.0):
        return (torch.randn(shape, generator=self.g, device=DEV) * std + mean).to(dtype)

    def int8(self, k, n):
        """q and the scales of N(0, 0.02) columns whose largest value maps to 127."""
        q = (torch.randn((k, n), generator=self.g, device=DEV) * 38.0).round_().clamp_(-127, 127).to(torch.int8)
        scales = torch.rand(n, generator=self.g, device=DEV) * 1e-4 + 4.8e-4
        return q, scales


def _spread(count, low, high):
    """`count` lengths from `low` to `high`, evenly."""
    if count == 1:
        return [high]
    return [low + (high - low) * i // (count - 1) for i in range(count)]


def _shuffled(seed, count, low, high):
    values = _spread(count, low, high)
    random.Random(seed).shuffle(values)
    return values


def _attention_lengths(case, seed):
    """Per request: queries, visible keys and the first query's position.  Decode
    and causal prefill put the queries at the end of the keys."""
    kv = _shuffled(seed, case["batch"], case["low"], case["kv"])
    q = [min(case["q"], v) for v in kv]
    return q, kv, [v - n for v, n in zip(kv, q)]


def prepare(case, seed):
    op, d = case["op"], _Draw(seed)
    s = {"case": case}
    if op in ("linear8", "linear16", "packed"):
        m, k, n = case["m"], case["k"], case["n"]
        s["a"] = d.normal((m, k))
        if op == "linear16":
            s["w"] = d.normal((k, n), 0.02)
        else:
            s["w"], s["scales"] = d.int8(k, n)
        s["bias"] = d.normal((n,), 0.02) if op == "packed" or case["bias"] else None
        if op == "packed":
            lib = _lib()
            s["residual"] = d.normal((m, n)) if case["epilogue"] == "residual" else None
            s["packed"] = torch.empty(lib.ti_amd_packed_w8_bytes(k, n), dtype=torch.uint8, device=DEV)
            s["y"] = torch.empty((m, n), dtype=torch.float16, device=DEV)
            _check(lib.ti_amd_pack_w8(s["w"].data_ptr(), k, n, s["packed"].data_ptr(),
                                      torch.cuda.current_stream().cuda_stream, torch.cuda.current_device()))
    elif op == "attention":
        b, h, dim = case["batch"], case["heads"], case["dim"]
        s["q"] = d.normal((b, h, case["q"], dim))
        s["k"], s["v"] = d.normal((b, h, case["kv"], dim)), d.normal((b, h, case["kv"], dim))
        s["ql"], s["kvl"], s["off"] = _attention_lengths(case, seed)
    elif op == "gemm32":
        s["a"] = d.normal((case["m"], case["k"]), dtype=torch.float32)
        s["b"] = d.normal((case["k"], case["n"]), dtype=torch.float32)
    elif op == "model":
        _model(case)
        lens = _shuffled(seed, case["batch"], case["low"], case["high"])
        r = np.random.default_rng(seed)
        s["prompts"] = [r.integers(0, VOCAB, n).tolist() for n in lens]
        s["forced"] = [[[int(t)] for t in r.integers(0, VOCAB, case["batch"])] for _ in range(case["steps"])]
    else:
        rows, cols = case["rows"], case["cols"]
        dtype = torch.float32 if op.endswith("32") else torch.float16
        s["x"] = d.normal((rows, cols), 2.0, dtype)
        if op.startswith("layernorm"):
            s["gamma"], s["beta"] = d.normal((cols,), 0.02, dtype, 1.0), d.normal((cols,), 0.02, dtype)
        if op == "layernorm_softmax32":
            s["y"] = torch.empty_like(s["x"])
    return s


def run(s):
    case = s["case"]
    op = case["op"]
    if op in ("linear8", "linear16"):
        out = torch.float32 if case["out"] == "f32" else torch.float16
        if op == "linear8":
            return _ops().gemm_int8(s["a"], s["w"], s["scales"], bias=s["bias"], config=case["config"],
                                    output_dtype=out)
        return _ops().gemm(s["a"], s["w"], bias=s["bias"], config=case["config"], output_dtype=out)
    if op == "packed":
        res = s["residual"]
        _check(_lib().ti_amd_gemm_w8p_fused(
            s["a"].data_ptr(), s["packed"].data_ptr(), s["scales"].data_ptr(), s["bias"].data_ptr(),
            s["y"].data_ptr(), None if res is None else res.data_ptr(), case["m"], case["n"], case["k"],
            EPILOGUES[case["epilogue"]], torch.cuda.current_stream().cuda_stream, torch.cuda.current_device()))
        return s["y"]
    if op == "attention":
        return _ops().attention(s["q"], s["k"], s["v"], q_lengths=s["ql"], kv_lengths=s["kvl"],
                                query_offsets=s["off"], causal=case["causal"])
    if op == "gemm32":
        return _ops().legacy_gemm(s["a"], s["b"])
    if op == "layernorm16":
        return _ops().layernorm(s["x"], s["gamma"], s["beta"])
    if op == "softmax16":
        return _ops().softmax(s["x"])
    if op == "gelu16":
        return _ops().gelu_new(s["x"])
    if op == "layernorm_softmax32":
        _check(_lib().ti_amd_layernorm_softmax_f32(
            s["x"].data_ptr(), s["gamma"].data_ptr(), s["beta"].data_ptr(), s["y"].data_ptr(), case["rows"],
            case["cols"], 1e-5, torch.cuda.current_stream().cuda_stream, torch.cuda.current_device()))
        return s["y"]
    model, slots = _model(case), list(range(case["batch"]))
    for slot in slots:
        model.reset(slot)
    first = model.forward(slots, s["prompts"])
    last = first
    for i, rows in enumerate(s["forced"]):
        last = model.forward(slots, rows, return_logits=i + 1 == len(s["forced"]))
    outs = [first] if last is first else [first, last]
    return [np.frombuffer(r["logits"], dtype=np.float32).reshape(r["shape"]) for r in outs]


# -- what a pass cannot do without ------------------------------------------------------
def _pairs(case):
    """(query, key) pairs that attention sees, and the live queries and keys."""
    kv = _spread(case["batch"], case["low"], case["kv"])
    pairs = live_q = 0
    for v in kv:
        q = min(case["q"], v)
        live_q += q
        pairs += q * v - (q * (q - 1) // 2 if case["causal"] else 0)
    return pairs, live_q, sum(kv)


def work(case):
    op = case["op"]
    if op in ("linear8", "linear16", "packed"):
        m, k, n = case["m"], case["k"], case["n"]
        wide = 2 if op == "linear16" else 1
        out = 4 if case.get("out") == "f32" else 2
        res = 2 * m * n if case.get("epilogue") == "residual" else 0
        return {"bytes": 2 * m * k + wide * k * n + (0 if wide == 2 else 4 * n) + 2 * n + out * m * n + res,
                "flops": 2 * m * k * n}
    if op == "attention":
        pairs, live_q, live_kv = _pairs(case)
        h, dim = case["heads"], case["dim"]
        return {"bytes": h * dim * 2 * (live_q + case["batch"] * case["q"] + 2 * live_kv), "flops": 4 * dim * h * pairs}
    if op == "gemm32":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": 4 * (m * k + k * n + m * n), "flops": 2 * m * k * n}
    if op == "model":
        arch = ARCHS[case["arch"]]
        hid, layers = arch["hidden"], arch["layers"]
        lens = _spread(case["batch"], case["low"], case["high"])
        linear = 12 * hid * hid * layers
        passes = 1 + case["steps"]
        tokens = sum(lens) + case["batch"] * case["steps"]
        attended = sum(n * (n + 1) // 2 + sum(n + 1 + i for i in range(case["steps"])) for n in lens)
        read = sum(n * case["steps"] + case["steps"] * (case["steps"] + 1) // 2 for n in lens) + sum(lens)
        logits = case["batch"] * VOCAB * 4 * (2 if case["steps"] else 1)
        return {"bytes": passes * (linear + hid * VOCAB) + layers * 4 * hid * read + logits,
                "flops": 2 * linear * tokens + 2 * hid * VOCAB * case["batch"] * passes + 4 * hid * layers * attended}
    rows, cols = case["rows"], case["cols"]
    size = 4 if op.endswith("32") else 2
    return {"bytes": 2 * rows * cols * size + (2 * cols * size if op.startswith("layernorm") else 0),
            "flops": 8 * rows * cols}


# -- tolerances ---------------------------------------------------------------------------
def tolerance(case):
    """About four times the distance from 64-bit arithmetic measured on the listed
    cases: fp16 results carry their rounding (about 2e-4), fp32 ones their sums'
    order, the models the fp16 activations of every layer."""
    op = case["op"]
    if op == "model":
        return {"rel": 5e-3}
    if op in ("gemm32", "layernorm_softmax32") or case.get("out") == "f32":
        return {"rel": 3e-6}
    return {"rel": 1.3e-3}


# -- the same in 64 bits ------------------------------------------------------------------
def _gelu(z):
    return 0.5 * z * (1 + torch.tanh(math.sqrt(2 / math.pi) * (z + 0.044715 * z ** 3)))


def _softmax_attention(q, k, v, off, causal):
    """q [h, n, d] against k, v [h, t, d] in 64 bits; query i sits at off + i."""
    score = q @ k.transpose(1, 2) / math.sqrt(q.shape[-1])
    if causal:
        at = torch.arange(q.shape[1], device=q.device)[:, None] + off
        score.masked_fill_(torch.arange(k.shape[1], device=q.device)[None] > at, -math.inf)
    return torch.softmax(score, -1) @ v


def _weights(case):
    """The artifact's weights in 64 bits on the GPU, int8 ones as the 16-bit values they stand for."""
    def read(path):
        _, t = load_tensors(path)
        out = {}
        for name, v in t.items():
            if name.endswith(".scales"):
                continue
            if v.dtype == np.int8:
                f = torch.from_numpy(np.array(v)).to(DEV).float() * torch.from_numpy(np.array(t[name + ".scales"])).to(DEV)
                out[name] = f.half().double()
            else:
                out[name] = torch.from_numpy(np.array(v).view(np.float16)).to(DEV).double()
        return out
    return _keep(("weights", case["arch"], case["precision"]),
                 lambda: _artifact(case["arch"], case["precision"], read))


def _last_hidden(w, arch, ids, at):
    """ln_f of the rows `at` of one request's tokens."""
    hid, heads = arch["hidden"], arch["heads"]
    norm = lambda x, p: torch.nn.functional.layer_norm(x, (hid,), w[p + ".weight"], w[p + ".bias"], 1e-5)  # noqa: E731
    lin = lambda x, p: x @ w[p + ".weight"] + w[p + ".bias"]  # noqa: E731
    x = w["transformer.wte.weight"][ids] + w["transformer.wpe.weight"][:len(ids)]
    for layer in range(arch["layers"]):
        p = f"transformer.h.{layer}."
        q, k, v = (t.reshape(len(ids), heads, -1).transpose(0, 1).contiguous()
                   for t in lin(norm(x, p + "ln_1"), p + "attn.c_attn").split(hid, 1))
        x = x + lin(_softmax_attention(q, k, v, 0, True).transpose(0, 1).reshape(len(ids), hid), p + "attn.c_proj")
        x = x + lin(_gelu(lin(norm(x, p + "ln_2"), p + "mlp.c_fc")), p + "mlp.c_proj")
    return norm(x[at], "transformer.ln_f")


def exact(case, seed):
    op, s = case["op"], prepare(case, seed) if case["op"] != "model" else None
    if op in ("linear8", "linear16", "packed"):
        w = s["w"] if op == "linear16" else (s["w"].float() * s["scales"]).half()
        y = s["a"].double() @ w.double()
        if s["bias"] is not None:
            y += s["bias"].double()
        if case.get("epilogue") == "gelu":
            y = _gelu(y)
        elif case.get("epilogue") == "residual":
            y += s["residual"].double()
        return y
    if op == "attention":
        y = torch.zeros(s["q"].shape, dtype=torch.float64, device=DEV)
        for b, (nq, nk, off) in enumerate(zip(s["ql"], s["kvl"], s["off"])):
            y[b, :, :nq] = _softmax_attention(s["q"][b, :, :nq].double(), s["k"][b, :, :nk].double(),
                                              s["v"][b, :, :nk].double(), off, case["causal"])
        return y
    if op == "gemm32":
        return s["a"].double() @ s["b"].double()
    if op == "gelu16":
        return _gelu(s["x"].double())
    if op != "model":
        x = s["x"].double()
        if op.startswith("layernorm"):
            x = torch.nn.functional.layer_norm(x, (case["cols"],), s["gamma"].double(), s["beta"].double(), 1e-5)
        return torch.softmax(x, -1) if "softmax" in op else x
    arch, w = ARCHS[case["arch"]], _weights(case)
    lens = _shuffled(seed, case["batch"], case["low"], case["high"])
    r = np.random.default_rng(seed)
    prompts = [r.integers(0, VOCAB, n).tolist() for n in lens]
    forced = [r.integers(0, VOCAB, case["batch"]).tolist() for _ in range(case["steps"])]
    rows = [[], []]
    for b, prompt in enumerate(prompts):
        ids = prompt + [f[b] for f in forced]
        h = _last_hidden(w, arch, ids, [len(prompt) - 1, len(ids) - 1])
        rows[0].append(h[0])
        rows[1].append(h[1])
    logits = [torch.stack(x) @ w["lm_head.weight"] for x in rows]
    return logits if case["steps"] else logits[:1]
