"""The work whose speed is watched: what a user of this framework has it do.

Families (``kind``), each through a public entry point:

  q4_linear    ``KernelTable.linear`` with a 4-bit group-64 weight
  bf16_linear  ``KernelTable.linear`` with a bf16 weight
  attention    ``PrefixKVCache.attention`` over a filled cache
  layer        one decoder layer composed of the kernel table's ops and the cache
  lm_head      ``drt_op_lm_head_score``: vocabulary softmax scores and tokens
  step         ``DeviceSession.propose_device``: one BD3 denoise step over a committed prefix
  window       ``start_device`` + ``execute_window``: a new BD3 request's prompt up to its
               first block's logits
  canvas       ``propose_device`` on a fixed-quota Dream session: the whole canvas, no cache

Shapes are the two architectures' of ``diffusorrt_amd.synthetic``; weights are random
(seeded on the device) with the scales the benchmarks use, norm weights near one.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from diffusorrt_amd import _lib
from diffusorrt_amd import synthetic as syn
from diffusorrt_amd.kernels import DeviceBF16Weight, DeviceQ4Weight, KernelTable, PrefixKVCache
from diffusorrt_amd.runtime import (Runtime, bd3_session_config, fixed_quota_session_config,
                                    rope_tables)

BLOCK = 32  # BD3's block, and the d2f_hybrid mask's
GEOMETRY = {"bd3": syn.BD3_QWEN3_06B, "dream": syn.DREAM_QWEN25_7B}
SHAPES = [(1024, 1024), (2048, 1024), (3072, 1024), (1024, 2048), (1024, 3072),
          (512, 3584), (3584, 3584), (18944, 3584), (3584, 18944)]  # (N, K) of both models
KERNELS = KernelTable()


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # a 32-token block through a small projection: the smallest call, all latency
        {"name": "q4_linear_block", "kind": "q4_linear", "m": 32, "n": 3072, "k": 1024,
         "x": "f32", "bias": False},
        # an 8-token block and its feeder row through a 7B projection: weight streaming
        {"name": "q4_linear_rows9", "kind": "q4_linear", "m": 9, "n": 18944, "k": 3584,
         "x": "bf16", "bias": False},
        # a 512-token canvas through a 7B projection
        {"name": "q4_linear_canvas", "kind": "q4_linear", "m": 512, "n": 18944, "k": 3584,
         "x": "f32", "bias": False},
        # the same with unquantized weights: one block of the small model ...
        {"name": "bf16_linear_block", "kind": "bf16_linear", "m": 32, "n": 1024, "k": 3072,
         "x": "f32", "bias": False},
        # ... and a 1000-token prompt of the large one
        {"name": "bf16_linear_prompt", "kind": "bf16_linear", "m": 1000, "n": 18944, "k": 3584,
         "x": "f32", "bias": False},
        # a block over an 8192-token prefix
        {"name": "attention_block_8k", "kind": "attention", "arch": "bd3", "rows": 32,
         "keys": 8224, "dtype": "f16", "mask": "d2f"},
        # the second 2048-token chunk of a prompt
        {"name": "attention_prompt", "kind": "attention", "arch": "bd3", "rows": 2048,
         "keys": 4096, "dtype": "bf16", "mask": "d2f"},
        # a decoder layer over a 2048-token prompt chunk, quantized
        {"name": "layer_prompt", "kind": "layer", "arch": "bd3", "weights": "q4", "rows": 2048,
         "prefix": 0},
        # scoring a block over the whole vocabulary
        {"name": "lm_head_block", "kind": "lm_head", "arch": "bd3", "weights": "q4", "rows": 32,
         "temperature": 0.0},
        # one denoise step of the small model at the longest prefix served
        {"name": "step_8k", "kind": "step", "prefix": 8192, "frontier": 32},
        # a 1000-token request to the unquantized small model, up to its first logits
        {"name": "window_bf16", "kind": "window", "weights": "bf16", "tokens": 1000, "scope": 8},
        # one step of the large model over prompt and canvas, half of it still masked
        {"name": "canvas_512", "kind": "canvas", "tokens": 512, "frontier": 256},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["q4_linear", "q4_linear", "bf16_linear", "bf16_linear", "attention",
                       "attention", "layer", "layer", "lm_head", "step", "window", "canvas"])
    if kind in ("q4_linear", "bf16_linear"):
        n, k = rng.choice(SHAPES)
        return {"kind": kind, "m": _log_int(rng, 1, 2048), "n": n, "k": k,
                "x": rng.choice(["f32", "bf16"]), "bias": rng.random() < 0.3}
    if kind == "attention":
        mask = rng.choice(["d2f", "full"])
        rows = _log_int(rng, 1, 2048)
        if mask == "full":  # a canvas attends itself
            return {"kind": kind, "arch": rng.choice(["bd3", "dream"]), "rows": rows,
                    "keys": rows, "dtype": rng.choice(["f16", "bf16"]), "mask": mask}
        return {"kind": kind, "arch": rng.choice(["bd3", "dream"]), "rows": rows,
                "keys": rows + BLOCK * rng.randint(0, 192), "dtype": rng.choice(["f16", "bf16"]),
                "mask": mask}
    if kind == "layer":
        rows = _log_int(rng, 8, 2048)
        return {"kind": kind, "arch": rng.choice(["bd3", "bd3", "dream"]),
                "weights": rng.choice(["q4", "bf16"]), "rows": rows,
                "prefix": BLOCK * rng.randint(0, 64)}
    if kind == "lm_head":
        return {"kind": kind, "arch": rng.choice(["bd3", "dream"]),
                "weights": rng.choice(["q4", "bf16"]), "rows": _log_int(rng, 1, 256),
                "temperature": rng.choice([0.0, 0.0, 0.8])}
    if kind == "step":
        return {"kind": kind, "prefix": BLOCK * _log_int(rng, 1, 256),
                "frontier": rng.choice([4, 8, 12, 16, 20, 24, 28, 32])}
    if kind == "window":
        return {"kind": kind, "weights": rng.choice(["q4", "bf16"]),
                "tokens": _log_int(rng, 40, 1600), "scope": rng.randint(1, 8)}
    tokens = rng.randint(64, 512)
    return {"kind": kind, "tokens": tokens, "frontier": rng.randint(4, tokens // 2)}


# ---------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(gen, *shape):
    return torch.randn(shape, generator=gen, device="cuda")


def _q4(gen, n, k):
    words = torch.randint(-2**31, 2**31, (n, k // 8), generator=gen, device="cuda",
                          dtype=torch.int64).to(torch.int32)
    scales = (0.003 + 0.003 * torch.rand((n, k // 64), generator=gen, device="cuda")).bfloat16()
    jitter = 0.004 * torch.rand((n, k // 64), generator=gen, device="cuda") - 0.002
    return syn.Q4Tensor(words, scales, (-7.5 * scales.float() + jitter).bfloat16())


def _bf16(gen, n, k):
    return (0.02 * _randn(gen, n, k)).bfloat16()


def _norm_weight(gen, d):
    return (1.0 + 0.1 * _randn(gen, d)).bfloat16()


def _weight(gen, weights, n, k):
    return _q4(gen, n, k) if weights == "q4" else _bf16(gen, n, k)


def _on_device(w):
    if isinstance(w, syn.Q4Tensor):
        return DeviceQ4Weight(w.w_q, w.scales, w.biases)
    return DeviceBF16Weight(w)


def _linear_inputs(case, seed):
    gen = _gen(seed)
    w = _weight(gen, "q4" if case["kind"] == "q4_linear" else "bf16", case["n"], case["k"])
    x = _randn(gen, case["m"], case["k"])
    x = x.bfloat16() if case["x"] == "bf16" else x
    bias = (0.02 * _randn(gen, case["n"])).bfloat16() if case["bias"] else None
    return x, w, bias


def _attention_inputs(case, seed):
    g = GEOMETRY[case["arch"]]
    gen = _gen(seed)
    tdt = torch.bfloat16 if case["dtype"] == "bf16" else torch.float16
    k = _randn(gen, case["keys"], g.num_kv_heads, 128).bfloat16()
    v = _randn(gen, case["keys"], g.num_kv_heads, 128).bfloat16()
    return _randn(gen, case["rows"], g.num_heads, 128).to(tdt), k, v


def _layer_weights(gen, g, weights, prefix=""):
    w = {prefix + "input_layernorm.weight": _norm_weight(gen, g.hidden_size),
         prefix + "post_attention_layernorm.weight": _norm_weight(gen, g.hidden_size)}
    if g.qk_norm:
        w[prefix + "self_attn.q_norm.weight"] = _norm_weight(gen, g.head_dim)
        w[prefix + "self_attn.k_norm.weight"] = _norm_weight(gen, g.head_dim)
    for suffix, (n, k) in syn.linear_shapes(g).items():
        w[prefix + suffix + ".weight"] = _weight(gen, weights, n, k)
        if g.qkv_bias and suffix[-6:] in ("q_proj", "k_proj", "v_proj"):
            w[prefix + suffix + ".bias"] = (0.02 * _randn(gen, n)).bfloat16()
    return w


def _layer_inputs(case, seed):
    g = GEOMETRY[case["arch"]]
    gen = _gen(seed)
    w = _layer_weights(gen, g, case["weights"])
    h = _randn(gen, case["rows"], g.hidden_size)
    k = _randn(gen, max(1, case["prefix"]), g.num_kv_heads, 128).bfloat16()
    v = _randn(gen, max(1, case["prefix"]), g.num_kv_heads, 128).bfloat16()
    cos, sin = rope_tables(case["prefix"] + case["rows"], 128, g.rope_theta)
    tables = [torch.from_numpy(np.concatenate([t, t], 1)[case["prefix"]:]).cuda().unsqueeze(1)
              .contiguous() for t in (cos, sin)]
    return h, w, k, v, tables


def _lm_head_inputs(case, seed):
    g = GEOMETRY[case["arch"]]
    gen = _gen(seed)
    w = _weight(gen, case["weights"], g.vocab_size, g.hidden_size)
    return _randn(gen, case["rows"], g.hidden_size), w


def _model(g, weights, seed):
    gen = _gen(seed)
    w = {"model.embed_tokens.weight": _bf16(gen, g.vocab_size, g.hidden_size)}
    for i in range(g.layer_count):
        w.update(_layer_weights(gen, g, weights, f"model.layers.{i}."))
    w["model.norm.weight"] = _norm_weight(gen, g.hidden_size)
    w["lm_head.weight"] = (w["model.embed_tokens.weight"]
                           if weights == "bf16" and g.tie_word_embeddings
                           else _weight(gen, weights, g.vocab_size, g.hidden_size))
    return syn.SyntheticModel(geometry=g, weight_kind=weights, weights=w)


def _session_case(case, seed):
    """(geometry, weight kind, tokens, frontier or scope) of a whole-model case."""
    if case["kind"] == "step":
        g, n = GEOMETRY["bd3"], case["prefix"] + BLOCK
        toks = syn.prompt_ids(seed, case["prefix"]) + [g.mask_token_id] * BLOCK
        rng = np.random.default_rng(seed)
        rows = np.sort(rng.choice(BLOCK, case["frontier"], replace=False)) + case["prefix"]
        known = syn.prompt_ids(seed + 1, BLOCK)
        for p in range(case["prefix"], n):  # the block's rows that earlier steps committed
            if p not in rows:
                toks[p] = known[p - case["prefix"]]
        return g, "q4", toks, [int(p) for p in rows]
    if case["kind"] == "window":
        g = GEOMETRY["bd3"]
        n = case["tokens"]
        first = (n - 1) // BLOCK * BLOCK  # the last block, masked from its start
        toks = syn.prompt_ids(seed, first) + [g.mask_token_id] * (n - first)
        return g, case["weights"], toks, list(range(max(first, n - case["scope"]), n))
    g = GEOMETRY["dream"]
    n, masked = case["tokens"], case["tokens"] // 2
    toks = syn.prompt_ids(seed, n - masked) + [g.mask_token_id] * masked
    rng = np.random.default_rng(seed)
    rows = np.sort(rng.choice(masked, case["frontier"], replace=False)) + n - masked
    for p in set(range(n - masked, n)) - set(int(r) for r in rows):
        toks[p] = int(rng.integers(0, 150000))
    return g, "q4", toks, [int(p) for p in rows]


_streams = []


def _every_queue():
    """Puts work on enough streams that the process has all of its hardware queues. A runtime
    notes at its creation where its stream's work-groups land, and refuses results once a
    hardware queue that came into being later has moved that; several runtimes in one process
    (one for each state here) are created after the queues, as a server would."""
    if not _streams:
        _streams.extend(torch.cuda.Stream() for _ in range(8))
        for s in _streams:
            with torch.cuda.stream(s):
                torch.zeros(1, device="cuda")
        torch.cuda.synchronize()


class _Open:
    """A runtime and its one open session, closed with the state that holds them."""

    def __init__(self, model, session_config, positions):
        _every_queue()
        self.runtime = Runtime(model, max_positions=positions)
        self.session = self.runtime.session(session_config)

    def __del__(self):
        try:
            self.session.close()
            self.runtime.close()
        except Exception:
            pass


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("q4_linear", "bf16_linear"):
        x, w, bias = _linear_inputs(case, seed)
        return {"kind": kind, "x": x, "w": _on_device(w), "bias": bias}
    if kind == "attention":
        q, k, v = _attention_inputs(case, seed)
        cache = PrefixKVCache(1, k.shape[1], case["keys"], dtype=case["dtype"])
        cache.store(0, k, v, 0)
        return {"kind": kind, "q": q, "cache": cache, "case": case}
    if kind == "layer":
        h, w, k, v, tables = _layer_inputs(case, seed)
        cache = PrefixKVCache(1, k.shape[1], case["prefix"] + case["rows"], dtype="f16")
        if case["prefix"]:
            cache.store(0, k, v, 0)
        dev = {n: (t if ".weight" not in n or "norm" in n else _on_device(t))
               for n, t in w.items()}
        return {"kind": kind, "h": h, "w": dev, "cache": cache, "tables": tables, "case": case,
                "g": GEOMETRY[case["arch"]]}
    if kind == "lm_head":
        x, w = _lm_head_inputs(case, seed)
        rows, (n, k) = x.shape[0], (GEOMETRY[case["arch"]].vocab_size, x.shape[1])
        ws = _lib.load().drt_op_lm_head_workspace_bytes(rows, n, k)
        return {"kind": kind, "x": x, "w": _on_device(w), "shape": (rows, n, k), "seed": seed,
                "temperature": case["temperature"],
                "positions": torch.arange(100, 100 + rows, dtype=torch.int32, device="cuda"),
                "scores": torch.empty(rows, dtype=torch.float64, device="cuda"),
                "tokens": torch.empty(rows, dtype=torch.int32, device="cuda"),
                "ws": torch.empty(ws, dtype=torch.uint8, device="cuda")}
    g, weights, toks, rows = _session_case(case, seed)
    config = (fixed_quota_session_config(64, 64, len(toks)) if kind == "canvas"
              else bd3_session_config(BLOCK, 8, len(toks)))
    held = _Open(_model(g, weights, seed), config, len(toks) + BLOCK)
    state = {"kind": kind, "held": held, "toks": toks, "rows": rows, "case": case,
             "mask": g.mask_token_id}
    if kind != "window":
        held.session.start_device(
            toks, prompt_len=len(toks) - len(toks) // 2 if kind == "canvas" else 0,
            block_size=64 if kind == "canvas" else BLOCK, mask_token_id=g.mask_token_id,
            exact_kv=False, steps=8)
    if kind == "step":  # the prefix is committed by the request's first step
        _propose(state)
    return state


# ---------------------------------------------------------------- one pass

def _propose(st):
    kw = ({"window_end": len(st["toks"]), "frozen_prefix": st["case"]["prefix"]}
          if st["kind"] == "step" else {"window_end": len(st["toks"]), "frozen_prefix": 0})
    scores, tokens, _ = st["held"].session.propose_device(st["rows"], **kw)
    return {"scores": np.asarray(scores), "tokens": np.asarray(tokens, dtype=np.int32)}


def _run_layer(st):
    w, g, case, cache = st["w"], st["g"], st["case"], st["cache"]
    cos, sin = st["tables"]
    m, eps, p0 = case["rows"], g.rms_norm_eps, case["prefix"]

    def proj(x, name):
        return KERNELS.linear(x, w[name + ".weight"], w.get(name + ".bias"))

    n = KERNELS.rms_norm(st["h"], w["input_layernorm.weight"], eps)
    q = proj(n, "self_attn.q_proj").view(m, g.num_heads, 128)
    k = proj(n, "self_attn.k_proj").view(m, g.num_kv_heads, 128)
    v = proj(n, "self_attn.v_proj").view(m, g.num_kv_heads, 128)
    if g.qk_norm:
        q = KERNELS.rms_norm(q, w["self_attn.q_norm.weight"], eps)
        k = KERNELS.rms_norm(k, w["self_attn.k_norm.weight"], eps)
    q, k = KERNELS.rope(q, cos, sin), KERNELS.rope(k, cos, sin)
    cache.store(0, k, v, p0)
    a = cache.attention(0, q.half(), n_keys=p0 + m, row_pos0=p0, kind="d2f_hybrid",
                        mask_geometry=(0, BLOCK))
    h = st["h"] + proj(a, "self_attn.o_proj")
    n = KERNELS.rms_norm(h, w["post_attention_layernorm.weight"], eps)
    act = KERNELS.swiglu(proj(n, "mlp.gate_proj"), proj(n, "mlp.up_proj"))
    return {"hidden": h + proj(act, "mlp.down_proj"), "k": k, "v": v}


def run(state):
    kind = state["kind"]
    if kind in ("q4_linear", "bf16_linear"):
        return KERNELS.linear(state["x"], state["w"], state["bias"])
    if kind == "attention":
        case = state["case"]
        d2f = case["mask"] == "d2f"
        return state["cache"].attention(
            0, state["q"], n_keys=case["keys"], row_pos0=case["keys"] - case["rows"],
            kind="d2f_hybrid" if d2f else "full", mask_geometry=(0, BLOCK) if d2f else None)
    if kind == "layer":
        return _run_layer(state)
    if kind == "lm_head":
        w, (rows, n, k) = state["w"], state["shape"]
        qw, sb, wb = ((w.qw, w.sb, None) if isinstance(w, DeviceQ4Weight) else (None, None, w.wb))

        def ptr(t):
            return None if t is None else C.c_void_p(t.data_ptr())

        _lib.check(_lib.load().drt_op_lm_head_score(
            ptr(qw), ptr(sb), ptr(wb), rows, n, k, ptr(state["x"]), state["temperature"],
            state["seed"], 3, ptr(state["positions"]), ptr(state["scores"]),
            ptr(state["tokens"]), None, ptr(state["ws"]), state["ws"].numel(),
            C.c_void_p(torch.cuda.current_stream().cuda_stream)))
        return {"scores": state["scores"], "tokens": state["tokens"]}
    if kind == "window":
        s = state["held"].session
        s.start_device(state["toks"], prompt_len=0, block_size=BLOCK,
                       mask_token_id=state["mask"], exact_kv=False, steps=8)
        return s.execute_window(state["toks"], state["rows"], mask_geometry=(0, BLOCK)).array()
    return _propose(state)


# ---------------------------------------------------------------- what a pass cannot do without

def _weight_bytes(weights, n, k):
    return n * k * (0.5625 if weights == "q4" else 2.0)


def _visible(rows, keys, mask):
    """Visible (row, key) pairs of the last ``rows`` of ``keys`` positions."""
    if mask == "full":
        return float(rows * keys)
    p = np.arange(keys - rows, keys)
    return float(np.minimum(keys, (p // BLOCK + 1) * BLOCK).sum())


def _layer_work(g, weights, rows, prefix, mask):
    params = sum(n * k for n, k in syn.linear_shapes(g).values())
    keys = prefix + rows
    kv = g.num_kv_heads * 128 * 2 * 2.0
    return {"bytes": _weight_bytes(weights, params, 1) + kv * keys + kv * rows,
            "flops": 2.0 * params * rows + 4.0 * 128 * g.num_heads * _visible(rows, keys, mask)}


def work(case):
    kind = case["kind"]
    if kind in ("q4_linear", "bf16_linear"):
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": _weight_bytes("q4" if kind == "q4_linear" else "bf16", n, k) +
                m * k * (2 if case["x"] == "bf16" else 4) + 4 * m * n,
                "flops": 2 * m * n * k}
    if kind == "attention":
        g = GEOMETRY[case["arch"]]
        rows, keys = case["rows"], case["keys"]
        return {"bytes": rows * g.num_heads * 128 * 6 + keys * g.num_kv_heads * 128 * 4,
                "flops": 4 * 128 * g.num_heads * _visible(rows, keys, case["mask"])}
    if kind == "layer":
        g = GEOMETRY[case["arch"]]
        w = _layer_work(g, case["weights"], case["rows"], case["prefix"], "d2f")
        # the residual in and out, and K and V handed back in 32 bits
        io = case["rows"] * (g.hidden_size * 8 + g.num_kv_heads * 128 * 8)
        return {"bytes": w["bytes"] + io, "flops": w["flops"]}
    if kind == "lm_head":
        g = GEOMETRY[case["arch"]]
        n, k = g.vocab_size, g.hidden_size
        return {"bytes": _weight_bytes(case["weights"], n, k) + case["rows"] * (4 * k + 12),
                "flops": 2 * case["rows"] * n * k}
    if kind == "canvas":
        g, weights, rows, prefix, lm, mask = (GEOMETRY["dream"], "q4", case["tokens"], 0,
                                              case["frontier"], "full")
    elif kind == "step":
        g, weights, rows, prefix, lm, mask = (GEOMETRY["bd3"], "q4", BLOCK, case["prefix"],
                                              case["frontier"], "d2f")
    else:
        g, weights, rows, prefix, lm, mask = (GEOMETRY["bd3"], case["weights"], case["tokens"], 0,
                                              min(case["scope"], (case["tokens"] - 1) % BLOCK + 1),
                                              "d2f")
    w = _layer_work(g, weights, rows, prefix, mask)
    head = _weight_bytes(weights, g.vocab_size, g.hidden_size)
    out = lm * (g.vocab_size * 4 if kind == "window" else 12)
    return {"bytes": g.layer_count * w["bytes"] + head + rows * g.hidden_size * 2 + out,
            "flops": g.layer_count * w["flops"] + 2.0 * lm * g.vocab_size * g.hidden_size}


def tolerance(case):
    """About four times what the path is seen to be off the 64-bit result where only its
    operand types set that, or what sums taken in another order change."""
    kind = case["kind"]
    if kind == "q4_linear":  # 32-bit sums; 1e-7 to 6e-7 seen
        return {"rel": 1e-5}
    if kind == "bf16_linear":  # bf16 results: now and then one unit in the last place
        return {"rel": 1e-3, "max": 0.02}
    if kind == "attention":  # probabilities enter the products in the cache's type
        return {"rel": 6e-3 if case["dtype"] == "bf16" else 8e-4, "max": 0.05}
    if kind == "layer":  # q4: the cache's fp16; bf16: every linear's result is rounded
        return {"rel": 6e-3 if case["weights"] == "bf16" else 5e-4, "max": 0.05}
    if kind == "lm_head":  # bf16 logits
        return {"rel": 5e-3 if case["weights"] == "bf16" else 1e-5, "differ": 0.01}
    if kind == "window":  # 28 layers of the above; 7e-3 and 5e-4 seen
        return {"rel": 2e-2 if case["weights"] == "bf16" else 2e-3, "max": 0.2}
    # scores over 28 layers; 3e-4 (step) and 2e-3 (canvas) seen
    return {"rel": 1.5e-3 if kind == "step" else 7e-3, "differ": 0.01}


# ---------------------------------------------------------------- the same in 64 bits

def _dense(w):
    if isinstance(w, syn.Q4Tensor):
        shifts = torch.arange(8, device=w.w_q.device, dtype=torch.int32) * 4
        q = ((w.w_q.unsqueeze(-1) >> shifts) & 15).reshape(w.w_q.shape[0], -1, 64).double()
        return (q * w.scales.double().unsqueeze(-1) +
                w.biases.double().unsqueeze(-1)).reshape(w.w_q.shape[0], -1)
    return w.double()


def _linear64(x, w, bias=None):
    """By output columns, so that a wide weight is never held whole in 64 bits."""
    out = []
    step = 16384
    n = w.shape[0]
    for c in range(0, n, step):
        part = (syn.Q4Tensor(w.w_q[c:c + step], w.scales[c:c + step], w.biases[c:c + step])
                if isinstance(w, syn.Q4Tensor) else w[c:c + step])
        # a bf16 weight takes its input in bf16
        xi = x if isinstance(w, syn.Q4Tensor) else x.to(torch.bfloat16).double()
        out.append(xi.double() @ _dense(part).t())
    y = torch.cat(out, 1)
    return y if bias is None else y + bias.double()


def _rms64(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _rope64(x, cos, sin):
    half = x.shape[-1] // 2
    rot = torch.cat([-x[..., half:], x[..., :half]], -1)
    return x * cos + rot * sin


def _attention64(q, k, v, pos0, mask):
    """``q [rows, Hq, 128]`` at positions from ``pos0`` over ``k``, ``v [keys, Hkv, 128]``."""
    rows, hq, _ = q.shape
    keys, hkv, _ = k.shape
    out = torch.empty_like(q)
    kpos = torch.arange(keys, device=q.device)
    for h in range(hq):
        kh, vh = k[:, h // (hq // hkv)], v[:, h // (hq // hkv)]
        for r in range(0, rows, 2048):
            s = (q[r:r + 2048, h] @ kh.t()) / math.sqrt(128.0)
            if mask == "d2f":
                qpos = torch.arange(pos0 + r, pos0 + min(rows, r + 2048), device=q.device)
                s = s.masked_fill(kpos >= ((qpos // BLOCK + 1) * BLOCK).unsqueeze(1), -math.inf)
            out[r:r + 2048, h] = torch.softmax(s, -1) @ vh
    return out.reshape(rows, hq * 128)


def _layer64(g, w, h, cos, sin, k_prev, v_prev, mask, prefix=""):
    m, eps = h.shape[0], g.rms_norm_eps

    def proj(x, name):
        return _linear64(x, w[prefix + name + ".weight"], w.get(prefix + name + ".bias"))

    n = _rms64(h, w[prefix + "input_layernorm.weight"], eps)
    q = proj(n, "self_attn.q_proj").view(m, g.num_heads, 128)
    k = proj(n, "self_attn.k_proj").view(m, g.num_kv_heads, 128)
    v = proj(n, "self_attn.v_proj").view(m, g.num_kv_heads, 128)
    if g.qk_norm:
        q = _rms64(q, w[prefix + "self_attn.q_norm.weight"], eps)
        k = _rms64(k, w[prefix + "self_attn.k_norm.weight"], eps)
    q, k = _rope64(q, cos, sin), _rope64(k, cos, sin)
    ka, va = (k, v) if k_prev is None else (torch.cat([k_prev, k]), torch.cat([v_prev, v]))
    a = _attention64(q, ka, va, ka.shape[0] - m, mask)
    h = h + proj(a, "self_attn.o_proj")
    n = _rms64(h, w[prefix + "post_attention_layernorm.weight"], eps)
    gate = proj(n, "mlp.gate_proj")
    return (h + proj(gate * torch.sigmoid(gate) * proj(n, "mlp.up_proj"), "mlp.down_proj"), k, v)


def _logits64(case, seed):
    g, weights, toks, rows = _session_case(case, seed)
    w = _model(g, weights, seed).weights
    cos, sin = (torch.from_numpy(np.concatenate([t, t], 1)).cuda().double().unsqueeze(1)
                for t in rope_tables(len(toks), 128, g.rope_theta))
    h = w["model.embed_tokens.weight"][torch.tensor(toks, device="cuda")].double()
    for i in range(g.layer_count):
        h = _layer64(g, w, h, cos, sin, None, None, "full" if case["kind"] == "canvas" else "d2f",
                     f"model.layers.{i}.")[0]
    shift = 1 if g.logits_convention == "dream_ar_shift" else 0
    h = h[torch.tensor([max(0, p - shift) for p in rows], device="cuda")]
    return _linear64(_rms64(h, w["model.norm.weight"], g.rms_norm_eps), w["lm_head.weight"])


def _scored(logits):
    top, arg = logits.max(-1)
    return {"scores": 1.0 / torch.exp(logits - top.unsqueeze(1)).sum(-1),
            "tokens": arg.to(torch.int32)}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("q4_linear", "bf16_linear"):
        x, w, bias = _linear_inputs(case, seed)
        return _linear64(x, w, bias)
    if kind == "attention":
        q, k, v = _attention_inputs(case, seed)
        return _attention64(q.double(), k.double(), v.double(), case["keys"] - case["rows"],
                            case["mask"])
    if kind == "layer":
        h, w, k, v, (cos, sin) = _layer_inputs(case, seed)
        some = case["prefix"] > 0
        out, k, v = _layer64(GEOMETRY[case["arch"]], w, h.double(), cos.double(), sin.double(),
                             k.double() if some else None, v.double() if some else None, "d2f")
        return {"hidden": out, "k": k, "v": v}
    if kind == "lm_head":
        if case["temperature"] > 0:  # keyed by this framework's own counter hash
            return None
        x, w = _lm_head_inputs(case, seed)
        return _scored(_linear64(x, w))
    if kind == "window":
        return _logits64(case, seed)
    return _scored(_logits64(case, seed))
