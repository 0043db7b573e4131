"""Workloads of this framework as a user's program makes them, for timing and comparing builds.

Two kinds of case:

* "requant": one fused int8 GEMM + fold + requant funnel on device buffers
  (sslm_hip_gemm_requant_noalloc on the caller's stream, or the synchronous
  sslm_hip_gemm_requant), the primitive a host calls for its own layers.
* "serve": one burst of requests against a mapped model, through superslm_amd.sslm: open the
  sessions, prefill every prompt (in chunks), decode greedily or damped greedily over the whole
  batch at a layer budget, save the last session's blob (its KV block and stream state, what a
  program keeps to resume it), close the sessions.  The model, its adapter and the KV pool are in
  hand before.  Returned are all tokens of all calls and the saved blob.

The framework computes in integers throughout and promises the same bits on every path, so every
case is compared exactly.
"""
import ctypes
import dataclasses
import os

import numpy as np
import torch

from superslm_amd.sslm import Model, SslmLib
from superslm_amd.sslm_artifact import CONFIGS, build_adapter, build_synthetic

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

IN_SCALE = (1 << 30, -37)
SITE = (1518500250, -45)


def _requant(name, m, n, k, stream):
    return {"name": name, "kind": "requant", "m": m, "n": n, "k": k, "stream": stream}


def _serve(name, model, batch, lo, hi, chunk, calls, budget, damped=False, lora=False):
    return {"name": name, "kind": "serve", "model": model, "batch": batch, "prompt_lo": lo, "prompt_hi": hi,
            "chunk": chunk, "calls": calls, "budget": budget, "damped": damped, "lora": lora}


def listed():
    return [
        # the smallest call: one 0.9B-class gate projection of 32 rows, asynchronous on a stream
        _requant("requant_32x4864x896", 32, 4864, 896, True),
        # ragged rows, columns and depth (none a multiple of a tile) through the synchronous entry
        _requant("requant_203x4880x1552", 203, 4880, 1552, False),
        # the largest rows, columns that the entry takes, at a 7B model's depth
        _requant("requant_512x8192x3584", 512, 8192, 3584, False),
        # one user: a short prompt, then a sentence; latency of single-sequence decode
        _serve("chat_1", "1.5b", 1, 24, 24, 512, 32, 28),
        # the benchmark's batch: 16 sequences with 32-token prompts, decoded together
        _serve("batch_16", "1.5b", 16, 32, 32, 512, 32, 28),
        # an ordinary serving batch: ragged short prompts, an odd number of sequences
        _serve("batch_50", "1.5b", 50, 5, 40, 512, 24, 28),
        # a large batch of very short prompts
        _serve("batch_100", "1.5b", 100, 4, 12, 512, 24, 28),
        # prompt processing: full 512-token chunks, then each first token
        _serve("prompt_512", "1.5b", 4, 512, 512, 512, 1, 28),
        # ragged documents in chunks of 256 (remainders included), then each first token
        _serve("prompt_ragged", "1.5b", 4, 97, 731, 256, 1, 28),
        # an interactive client with a frame budget: 4 layers a call, damped greedy sampling
        _serve("sliced_damped_3", "1.5b", 3, 40, 90, 64, 57, 4, damped=True),
        # a rank-16 adapter on q and v: 64-token prompts, then decoding
        _serve("lora_8", "1.5b", 8, 64, 64, 512, 16, 28, lora=True),
        # long contexts at the 7B shape (four of its 28 layers): 32 sequences of 2048 tokens
        _serve("long_7b", "7b", 32, 2048, 2048, 2048, 192, 4),
    ]


# ---- shapes ----
# "7b" keeps the 7B configuration's widths and heads with 4 of its 28 identical layers, so that a
# process can make and map it in seconds.
def _config(model):
    if model == "7b":
        return dataclasses.replace(CONFIGS["qwen7b"], layers=4)
    return CONFIGS["qwen1.5b"]


def _lengths(case):
    """The prompts' lengths, spread over [prompt_lo, prompt_hi] the same way for every seed."""
    lo, hi = case["prompt_lo"], case["prompt_hi"]
    return [lo + (i * 7919 + (hi - lo)) % (hi - lo + 1) for i in range(case["batch"])]


def _layer_elems(c):
    kvh = c.kv_heads * c.head_dim
    return c.hidden * (2 * c.hidden + 2 * kvh + 3 * c.inter)


def _plan(case):
    """(prefill calls as (context, tokens), decode steps as context sums, head rows) of one pass."""
    c = _config(case["model"])
    lens = _lengths(case)
    pre = []
    for n in lens:
        done = 0
        while done < n:
            t = min(case["chunk"], n - done)
            pre.append((done, t))
            done += t
    # the first call after a prefill takes logits only; then layers / budget calls make a token
    per = -(-c.layers // case["budget"])
    layer_calls = case["calls"] - 1
    return c, lens, pre, per, layer_calls


def work(case):
    if case["kind"] == "requant":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": m * k + n * k + 12 * n + m * n + 20 * m, "flops": 2 * m * n * k}
    c, lens, pre, per, layer_calls = _plan(case)
    le, head = _layer_elems(c), c.vocab * c.hidden
    kv_row = 2 * c.kv_heads * c.head_dim  # bytes of one position's K and V in one layer
    by = fl = 0
    for ctx, t in pre:
        by += c.layers * (le + kv_row * (ctx + t)) + t * c.hidden
        fl += c.layers * (2 * t * le + 4 * c.hidden * (t * ctx + t * (t + 1) // 2))
    tokens = layer_calls // per  # whole tokens' worth of layers
    for s in range(tokens):
        widths = sum(n + s + 1 for n in lens)
        by += c.layers * (le + kv_row * widths)
        fl += c.layers * (2 * len(lens) * le + 4 * c.hidden * widths)
    heads = 1 + tokens
    by += heads * head + c.layers * c.context_cap * kv_row
    fl += heads * 2 * len(lens) * head
    return {"bytes": by, "flops": fl}


def draw(rng):
    def log(lo, hi):
        return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))

    if rng.random() < 0.3:
        stream = rng.random() < 0.5
        return {"kind": "requant", "m": log(1, 128 if stream else 512), "n": 16 * log(1, 512), "k": 16 * log(4, 224),
                "stream": stream}
    most = work(listed()[-1])
    while True:
        model = "1.5b" if rng.random() < 0.8 else "7b"
        c = _config(model)
        hi = log(4, 900 if model == "1.5b" else 2048)
        lo = max(1, hi - rng.randrange(0, hi))
        budget = c.layers if rng.random() < 0.7 else rng.choice([1, 2, 4] if model == "7b" else [1, 4, 7, 13])
        per = -(-c.layers // budget)
        case = {"kind": "serve", "model": model, "batch": log(1, 112), "prompt_lo": lo, "prompt_hi": hi,
                "chunk": rng.choice([64, 200, 512, 2048]), "calls": 1 + per * log(1, 48), "budget": budget,
                "damped": model == "1.5b" and rng.random() < 0.2, "lora": model == "1.5b" and rng.random() < 0.2}
        # latency counts beside bytes: a bound on the launches as well as on the work
        _, lens, pre, _, layer_calls = _plan(case)
        layers = len(pre) * c.layers + layer_calls * budget
        w = work(case)
        if layers <= 6000 and w["bytes"] <= most["bytes"] and w["flops"] <= most["flops"] and \
                hi + case["calls"] // per < c.context_cap:
            return case


def tolerance(case):
    return "exact"  # integer arithmetic throughout: the same bits on every path


# ---- what a program holds ----
class _Library:
    lib = None
    models = {}
    adapters = {}


def _lib():
    if _Library.lib is None:
        lib = SslmLib(os.path.join(ROOT, "superslm_amd", "libsslm_hip.so"))
        vp, i32, i64 = ctypes.c_void_p, ctypes.c_int32, ctypes.c_int64
        lib.lib.sslm_hip_gemm_requant.restype = ctypes.c_int
        lib.lib.sslm_hip_gemm_requant.argtypes = [vp] * 3 + [i32] * 3 + [i64] * 4 + [vp] * 3
        lib.lib.sslm_hip_gemm_requant_noalloc.restype = ctypes.c_int
        lib.lib.sslm_hip_gemm_requant_noalloc.argtypes = [vp] * 3 + [i32] * 3 + [i64] * 4 + [vp] * 4
        _Library.lib = lib
    return _Library.lib


def _model(kind):
    """The mapped model of a shape: a program maps its artifact once and keeps it."""
    if kind not in _Library.models:
        sm = build_synthetic(_config(kind), seed=1515 if kind == "1.5b" else 7007,
                             damped_logit_scale=1.0 / 20000 if kind == "1.5b" else None)
        _Library.models[kind] = (Model(_lib(), sm.to_array()), sm)
    return _Library.models[kind]


def _adapter(kind):
    if kind not in _Library.adapters:
        model, sm = _model(kind)
        _Library.adapters[kind] = model.adapter(build_adapter(sm, rank=16, targets=("q_proj", "v_proj"), seed=31))
    return _Library.adapters[kind]


class _Serve:
    """One client's holdings: a KV pool, its prompts, and a buffer for a saved session."""

    def __init__(self, case, seed):
        self.case = case
        self.model, _ = _model(case["model"])
        self.adapter = _adapter(case["model"]) if case["lora"] else None
        self.pool = self.model.pool(case["batch"])
        c = _config(case["model"])
        rng = np.random.default_rng(seed)
        self.prompts = [rng.integers(0, c.vocab, size=n, dtype=np.int32) for n in _lengths(case)]
        self.params = self.model.decode_params(case["budget"], 1) if case["damped"] else None
        self.history = c.context_cap if case["damped"] else 0  # a damped session's blob carries its tokens
        self.blob = np.zeros(self.model.block_size + c.hidden + 4 * self.history + 256, dtype=np.uint8)

    def __del__(self):
        if getattr(self, "pool", None) is not None:
            self.pool.close()


def _requant_host(case, seed):
    """Activations and weights uniform in [-127, 127], per-column multipliers in [2^30, 2^31) with
    right shifts in [8, 20]."""
    rng = np.random.default_rng(seed)
    m, n, k = case["m"], case["n"], case["k"]
    a = rng.integers(-127, 128, size=(m, k), dtype=np.int8)
    w = rng.integers(-127, 128, size=(n, k), dtype=np.int8)
    fold = np.zeros((n, 3), dtype=np.int32)
    fold[:, 1] = rng.integers(1 << 30, 1 << 31, size=n, dtype=np.int64).astype(np.int32)
    fold[:, 2] = rng.integers(8, 21, size=n, dtype=np.int32)
    return a, w, fold


def prepare(case, seed):
    if case["kind"] == "serve":
        return _Serve(case, seed)
    a, w, fold = (torch.from_numpy(x).cuda() for x in _requant_host(case, seed))
    m, n = case["m"], case["n"]
    return {"case": case, "a": a, "w": w, "fold": fold, "codes": torch.zeros((m, n), dtype=torch.int8, device="cuda"),
            "scales": torch.zeros((m, 2), dtype=torch.int64, device="cuda"),
            "status": torch.zeros((m,), dtype=torch.int32, device="cuda")}


def _run_requant(s):
    case, L = s["case"], _lib().lib
    args = (s["a"].data_ptr(), s["w"].data_ptr(), s["fold"].data_ptr(), case["m"], case["n"], case["k"], *IN_SCALE,
            *SITE, s["codes"].data_ptr(), s["scales"].data_ptr(), s["status"].data_ptr())
    if case["stream"]:
        st = L.sslm_hip_gemm_requant_noalloc(*args, torch.cuda.current_stream().cuda_stream)
    else:
        st = L.sslm_hip_gemm_requant(*args)
    _lib().check("gemm_requant", st)
    return {"codes": s["codes"], "scales": s["scales"], "status": s["status"]}


def run(state):
    if isinstance(state, dict):
        return _run_requant(state)
    case, model = state.case, state.model
    seqs = [state.pool.seq() for _ in range(case["batch"])]
    for s, p in zip(seqs, state.prompts):
        if state.adapter is not None:
            s.set_adapter(state.adapter)
        done = 0
        while done < len(p):
            done += s.prefill(p[done:], chunk_budget=case["chunk"])
    tokens = np.array([model.decode_step(seqs, case["budget"], params=state.params) for _ in range(case["calls"])],
                      dtype=np.int32)
    n = ctypes.c_size_t(state.blob.nbytes)
    lib = model.lib
    lib.check("sslm_seq_save", lib.lib.sslm_seq_save(seqs[-1].handle, state.blob.ctypes.data, ctypes.byref(n)))
    for s in seqs:
        if state.adapter is not None:
            s.set_adapter(None)
        s.release()
    return {"tokens": tokens, "session": state.blob[:n.value]}


# ---- the same in plain integers ----
def _combine(a, b):
    """Product of two carried scales (mantissa in [2^30, 2^31), exponent), rounded to a mantissa."""
    m = (a[0] * b[0] + (1 << 30)) >> 31
    e = a[1] + b[1] + 31
    return (m << 1, e - 1) if m < (1 << 30) else (m, e)


def exact(case, seed):
    """The requant cases in 64-bit integers.  A "serve" case has none: 64-bit integers through 28
    layers of 1.3 billion weights take minutes a token."""
    if case["kind"] != "requant":
        return None
    a, w, fold = _requant_host(case, seed)
    acc = (a.astype(np.float64) @ w.astype(np.float64).T).astype(np.int64)  # exact: |sums| < 2^53
    hi = (acc * fold[:, 1].astype(np.int64) + (1 << 30)) >> 31
    sh = fold[:, 2].astype(np.int64)
    x = np.sign(hi) * ((np.abs(hi) + (np.int64(1) << (sh - 1))) >> sh)  # ties away from zero
    codes = np.zeros(x.shape, dtype=np.int8)
    scales = np.zeros((case["m"], 2), dtype=np.int64)
    for t in range(case["m"]):
        d = max(1, int(np.abs(x[t]).max()))
        s = 30 - (d.bit_length() - 1)
        dn = d << s if s >= 0 else d >> 1
        r = ((1 << 63) + dn) // (2 * dn)
        f, e, ax = 127 * r, 62 - s, np.abs(x[t])
        high = ax * (f >> 16) + ((ax * (f & 0xffff)) >> 16)  # |x| f / 2^16
        mag = np.minimum((high + (1 << (e - 17))) >> (e - 16), 127)
        codes[t] = (np.sign(x[t]) * mag).astype(np.int8)
        scales[t] = _combine(_combine(IN_SCALE, SITE), (dn, -s))
    return {"codes": codes, "scales": scales, "status": np.zeros(case["m"], dtype=np.int32)}
