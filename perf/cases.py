"""The work that programs give this library, as cases that can be timed and compared.

Shapes are the ones the library serves (hidden 2048, intermediate 11008, 16
query and 2 KV heads of 128, NF4 blocks of 64, vocabulary 151,936).  A case is
a dict of plain values; ``kind`` says which entry point it goes through:

* ``decode``  -- one greedy token of the whole 36-layer model: the captured
  step replayed at a cached length, what a generation loop repeats per token.
* ``prefill`` -- a prompt, or a later part of one (``start`` > 0), through a
  quarter of the model (9 of 36 layers, a quarter of the vocabulary, so that
  layers and head keep their shares), what a program does before it decodes.
* ``layers``  -- decoder layers put together from the single entry points
  (QKV+RoPE+cache, graph-mode attention, GEMV, MLP) by a program that captures
  them with the handle's own graph and replays it.
* ``qkv``, ``gqa``, ``lm_head`` -- single decode operations called
  eagerly, as a framework's patched modules call them; fp16 where the entry
  point has an fp16 form.
* ``gemm``, ``gemm_swiglu`` -- the multi-token projections for programs with a
  prefill of their own: any token count, each epilogue.
* ``dequantize``, ``quantize`` -- weights on their way in (loading a model) and
  out (a framework linear that multiplies dense weights).

Weights are normal random matrices quantised here block by block; activations
and cache rows are normal with the spread they have in such a model.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from kudacuda_amd._native import Native
from kudacuda_amd.qwen2_decoder import Qwen2Nf4Decoder
from kudacuda_amd.synthetic import QWEN25_3B

DEV = "cuda:0"
HIDDEN, INTER, Q_OUT, KV_OUT, HEADS, KV_HEADS, DIM = 2048, 11008, 2048, 256, 16, 2, 128
EPS = 1.0e-6
SCALE = 1.0 / math.sqrt(DIM)
VOCAB, LAYERS = QWEN25_3B.vocab, QWEN25_3B.layers
PART_LAYERS, PART_VOCAB = LAYERS // 4, VOCAB // 4
SHAPES = {"q": (Q_OUT, HIDDEN), "k": (KV_OUT, HIDDEN), "v": (KV_OUT, HIDDEN), "o": (HIDDEN, Q_OUT),
          "gate": (INTER, HIDDEN), "up": (INTER, HIDDEN), "down": (HIDDEN, INTER)}
BIASES = {"q_bias": Q_OUT, "k_bias": KV_OUT, "v_bias": KV_OUT}
LAYER_ELEMENTS = sum(n * k for n, k in SHAPES.values())
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
KINDS = {"fp32": 0, "bf16": 1, "fp16": 2}

# The 16 values of the NF4 format (as published with QLoRA / bitsandbytes).
NF4 = (-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453, -0.28444138169288635,
       -0.18477343022823334, -0.09105003625154495, 0.0, 0.07958029955625534, 0.16093020141124725,
       0.24611230194568634, 0.33791524171829224, 0.44070982933044434, 0.5626170039176941, 0.7229568362236023, 1.0)


# ------------------------------------------------------------------ cases
def listed() -> list[dict]:
    return [
        # a chat turn early in a conversation: the per-token step, launch and latency bound
        {"name": "decode at 128 tokens", "kind": "decode", "cached": 128, "capacity": 2048},
        # the same with a long document in the cache
        {"name": "decode at 5000 tokens", "kind": "decode", "cached": 5000, "capacity": 8192},
        # a short question
        {"name": "prefill 64", "kind": "prefill", "start": 0, "count": 64},
        # the next part of a prompt that is fed in parts
        {"name": "prefill 512 after 1024", "kind": "prefill", "start": 1024, "count": 512},
        # a document, of no round length
        {"name": "prefill 1999", "kind": "prefill", "start": 0, "count": 1999},
        # a program's own decode graph over the single entry points
        {"name": "4 layers at 585 tokens", "kind": "layers", "layers": 4, "cached": 585, "capacity": 2048},
        # one projection of a patched framework module, the smallest call
        {"name": "qkv fp16", "kind": "qkv", "dtype": "fp16"},
        # attention alone over a long cache
        {"name": "gqa bf16 30000", "kind": "gqa", "dtype": "bf16", "mode": "direct", "cached": 30000,
         "capacity": 30000},
        # projections of a program with its own prefill: a short prompt into the residual stream ...
        {"name": "gemm down 100 residual", "kind": "gemm", "tokens": 100, "n": HIDDEN, "k": INTER,
         "epilogue": "residual"},
        # ... a middling one with a bias ...
        {"name": "gemm q 700 bias", "kind": "gemm", "tokens": 700, "n": Q_OUT, "k": HIDDEN, "epilogue": "bias"},
        # ... and the widest projection over a long one
        {"name": "gemm swiglu 1000", "kind": "gemm_swiglu", "tokens": 1000, "n": INTER, "k": HIDDEN},
        # a framework linear that multiplies dense weights, the largest matrix
        {"name": "dequantize gate bf16", "kind": "dequantize", "n": INTER, "k": HIDDEN, "dtype": "bf16"},
    ]


def _spread(rng, low: int, high: int) -> int:
    """A whole number from low to high, even over its logarithm."""

    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high + 1))))))


def draw(rng) -> dict:
    kind = rng.choice(["decode", "prefill", "prefill", "prefill", "layers", "gqa", "gqa", "gemm", "gemm",
                       "gemm_swiglu", "dequantize", "quantize", "lm_head", "decode"])
    if kind == "decode":
        cached = _spread(rng, 1, 8000)
        return {"kind": kind, "cached": cached, "capacity": 2048 if cached < 2040 else 8192}
    if kind == "prefill":
        count = _spread(rng, 1, 1900)
        room = max(0, (1999 * 1000) // count - count // 2)  # cached rows read: no more than the longest prompt's
        start = 0 if rng.random() < 0.5 else rng.randint(0, min(room, 3000))
        return {"kind": kind, "start": start, "count": count}
    if kind == "layers":
        cached = _spread(rng, 1, 2000)
        return {"kind": kind, "layers": rng.randint(1, 4), "cached": cached, "capacity": 2048}
    if kind == "gqa":
        mode = rng.choice(["direct", "graph"])
        cached = _spread(rng, 1, 60000 if mode == "direct" else 8000)
        capacity = cached if mode == "direct" else cached + rng.randint(0, 2000)
        return {"kind": kind, "dtype": rng.choice(["bf16", "fp16"]), "mode": mode, "cached": cached,
                "capacity": capacity}
    if kind == "gemm":
        n, k = rng.choice([(Q_OUT, HIDDEN), (KV_OUT, HIDDEN), (HIDDEN, INTER), (INTER, HIDDEN)])
        return {"kind": kind, "tokens": _spread(rng, 1, 2000), "n": n, "k": k,
                "epilogue": rng.choice(["plain", "bias", "residual"])}
    if kind == "gemm_swiglu":
        return {"kind": kind, "tokens": _spread(rng, 1, 1500), "n": INTER, "k": HIDDEN}
    if kind == "dequantize":
        return {"kind": kind, "n": 64 * rng.randint(1, INTER // 64), "k": rng.choice([HIDDEN, INTER // 4]),
                "dtype": rng.choice(["bf16", "fp16", "fp32"])}
    if kind == "quantize":
        return {"kind": kind, "n": 64 * rng.randint(1, INTER // 64), "k": HIDDEN, "dtype": rng.choice(["bf16", "fp32"])}
    return {"kind": "lm_head", "vocab": _spread(rng, 1000, VOCAB)}


# ----------------------------------------------------------------- inputs
_handle: list[Native] = []
_streams: list[torch.cuda.Stream] = []


def _native() -> Native:
    """The program's one handle for eager calls."""

    if not _handle:
        _handle.append(Native(0))
    return _handle[0]


def _stream() -> torch.cuda.Stream:
    """The program's one stream for models and graphs: its steps follow one another."""

    if not _streams:
        _streams.append(torch.cuda.Stream(device=DEV))
    return _streams[0]


def _gen(seed: int, part: int = 0) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(int(seed) * 1000003 + part)


def _normal(gen, shape, std=1.0, dtype=torch.bfloat16, mean=0.0) -> torch.Tensor:
    return (torch.randn(shape, generator=gen, device=DEV) * std + mean).to(dtype)


def _nf4(gen, n: int, k: int, std: float = 0.02) -> tuple[torch.Tensor, torch.Tensor]:
    """Packed codes and block maxima of a normal [n, k] matrix."""

    w = torch.randn(n * k // 64, 64, generator=gen, device=DEV) * std
    absmax = w.abs().amax(dim=1)
    levels = torch.tensor(NF4, device=DEV)
    codes = torch.bucketize(w / absmax[:, None], (levels[1:] + levels[:-1]) / 2, out_int32=True).to(torch.uint8)
    codes = codes.reshape(-1, 2)
    return (codes[:, 0] << 4 | codes[:, 1]).contiguous(), absmax.contiguous()


def _dense(packed: torch.Tensor, absmax: torch.Tensor, n: int, k: int) -> torch.Tensor:
    """The matrix that packed codes stand for, in 64 bits."""

    levels = torch.tensor(NF4, device=DEV, dtype=torch.float32).double()
    codes = torch.stack([packed >> 4, packed & 15], dim=1).reshape(-1, 64).long()
    return (levels[codes] * absmax.double()[:, None]).reshape(n, k)


def _layer(seed: int, index: int) -> dict[str, torch.Tensor]:
    gen = _gen(seed, 10 + index)
    layer = {}
    for name, (n, k) in SHAPES.items():
        layer[f"{name}_packed"], layer[f"{name}_absmax"] = _nf4(gen, n, k)
    for name, n in BIASES.items():
        layer[name] = _normal(gen, n, 0.02)
    for name in ("input_norm", "post_norm"):
        layer[name] = _normal(gen, HIDDEN, 0.02, mean=1.0)
    return layer


def _caches(seed: int, index: int, capacity: int, dtype=torch.bfloat16) -> tuple[torch.Tensor, torch.Tensor]:
    gen = _gen(seed, 5000 + index)
    shape = (KV_HEADS, capacity, DIM)
    return _normal(gen, shape, 0.9, dtype), _normal(gen, shape, 0.9, dtype)


def _tokens(seed: int, count: int, vocab: int) -> np.ndarray:
    return np.random.default_rng([seed, 7]).integers(0, vocab, size=count).astype(np.int32)


def _embedding(seed: int, vocab: int) -> tuple[torch.Tensor, torch.Tensor]:
    gen = _gen(seed, 1)
    return _normal(gen, (vocab, HIDDEN), 0.02), _normal(gen, HIDDEN, 0.02, mean=1.0)


def _model(seed: int, layers: int, vocab: int, capacity: int, cached: int) -> Qwen2Nf4Decoder:
    embed, final_norm = _embedding(seed, vocab)
    dec = Qwen2Nf4Decoder(_native(), torch, QWEN25_3B, [_layer(seed, i) for i in range(layers)], embed, final_norm,
                          kv_capacity=capacity, token_capacity=capacity, device=DEV,
                          stream=_stream())
    torch.cuda.synchronize()
    for i, layer in enumerate(dec.layers if cached else []):
        for name, rows in zip(("key_cache", "value_cache"), _caches(seed, i, capacity)):
            layer[name][:, :cached].copy_(rows[:, :cached])
    torch.cuda.synchronize()
    return dec


def _rope(capacity: int) -> tuple[torch.Tensor, torch.Tensor]:
    inv = QWEN25_3B.rope_theta ** (-torch.arange(0, DIM, 2, dtype=torch.float64, device=DEV) / DIM)
    angle = torch.arange(capacity, dtype=torch.float64, device=DEV)[:, None] * inv[None]
    return angle.cos().float(), angle.sin().float()


def prepare(case: dict, seed: int) -> dict:
    kind, gen = case["kind"], _gen(seed)
    s: dict = {"case": case, "kind": kind}
    if kind == "decode":
        cached, capacity = case["cached"], case["capacity"]
        dec = _model(seed, LAYERS, VOCAB, capacity, cached)
        dec.reset(_tokens(seed, cached + 1, VOCAB), start_step=cached)
        dec.capture()
        s.update(dec=dec, begin=dec.control.clone(), step=cached)
    elif kind == "prefill":
        start, count = case["start"], case["count"]
        capacity = -(-(start + count + 1) // 64) * 64
        dec = _model(seed, PART_LAYERS, PART_VOCAB, capacity, start)
        prompt = _tokens(seed, start + count, PART_VOCAB)
        s.update(dec=dec, prompt=prompt)
        if start:
            nbytes = int(dec.native.lib.kudacuda_qwen2_prefill_workspace_bytes(count))
            s.update(workspace=torch.empty(nbytes, dtype=torch.uint8, device=DEV), nbytes=nbytes)
            dec.reset(prompt)
    elif kind == "layers":
        s.update(_prepare_layers(case, seed))
    elif kind == "qkv":
        dt = DTYPES[case["dtype"]]
        w = [_nf4(gen, n, HIDDEN) for n in (Q_OUT, KV_OUT, KV_OUT)]
        s.update(x=_normal(gen, HIDDEN, 1.0, dt), gamma=_normal(gen, HIDDEN, 0.1, dt, 1.0), w=w,
                 bias=[_normal(gen, n, 0.02, dt) for n in (Q_OUT, KV_OUT, KV_OUT)],
                 out=[torch.empty(n, dtype=dt, device=DEV) for n in (Q_OUT, KV_OUT, KV_OUT)])
    elif kind == "gqa":
        dt = DTYPES[case["dtype"]]
        k, v = _caches(seed, 0, case["capacity"], dt)
        s.update(q=_normal(gen, (HEADS, DIM), 0.9, dt), k=k, v=v, out=torch.empty((HEADS, DIM), dtype=dt, device=DEV),
                 length=torch.tensor([case["cached"]], dtype=torch.int32, device=DEV))
    elif kind == "lm_head":
        embed, norm = _embedding(seed, case["vocab"])
        s.update(x=_normal(gen, HIDDEN), gamma=norm, w=embed,
                 logits=torch.empty(case["vocab"], dtype=torch.bfloat16, device=DEV),
                 token=torch.zeros(1, dtype=torch.int32, device=DEV))
    elif kind in ("gemm", "gemm_swiglu"):
        m, n, k = case["tokens"], case["n"], case["k"]
        s.update(x=_normal(gen, (m, k)), w=[_nf4(gen, n, k) for _ in range(2 if kind == "gemm_swiglu" else 1)],
                 out=torch.empty((m, n), dtype=torch.bfloat16, device=DEV), bias=_normal(gen, n, 0.02),
                 residual=_normal(gen, (m, n)))
    elif kind == "dequantize":
        s.update(w=_nf4(gen, case["n"], case["k"]),
                 out=torch.empty((case["n"], case["k"]), dtype=DTYPES[case["dtype"]], device=DEV))
    else:
        n = case["n"] * case["k"]
        s.update(w=_normal(gen, n, 0.02, DTYPES[case["dtype"]]), packed=torch.empty(n // 2, dtype=torch.uint8, device=DEV),
                 absmax=torch.empty(n // 64, dtype=torch.float32, device=DEV))
    return s


def _prepare_layers(case: dict, seed: int) -> dict:
    """Weights, caches and one captured graph of the chained entry points."""

    native, stream = Native(0), _stream()  # a handle holds one graph: one for each program
    cached, capacity = case["cached"], case["capacity"]
    layers = [_layer(seed, i) for i in range(case["layers"])]
    caches = [_caches(seed, i, capacity) for i in range(case["layers"])]
    cos, sin = _rope(capacity)
    x0 = _normal(_gen(seed), HIDDEN)
    b = {n: torch.empty(k, dtype=torch.bfloat16, device=DEV)
         for n, k in (("q", Q_OUT), ("attn", Q_OUT), ("mid", INTER), ("h", HIDDEN), ("y", HIDDEN))}
    position = torch.tensor([cached], dtype=torch.int32, device=DEV)
    length = position + 1
    p, st = torch.Tensor.data_ptr, stream.cuda_stream
    torch.cuda.synchronize()

    def record():
        x = x0
        for w, (kc, vc) in zip(layers, caches):
            native.call("kudacuda_qwen2_qkv_rope_cache_nf4_bf16", p(x), p(w["input_norm"]), p(w["q_packed"]),
                        p(w["q_absmax"]), p(w["q_bias"]), p(w["k_packed"]), p(w["k_absmax"]), p(w["k_bias"]),
                        p(w["v_packed"]), p(w["v_absmax"]), p(w["v_bias"]), p(cos), p(sin), p(position), p(b["q"]),
                        p(kc), p(vc), capacity, HIDDEN, Q_OUT, KV_OUT, 64, EPS, st)
            native.call("kudacuda_qwen2_gqa_decode_graph_bf16", p(b["q"]), p(kc), p(vc), p(b["attn"]), 1, 1, capacity,
                        HEADS, KV_HEADS, DIM, SCALE, p(length), st)
            native.call("kudacuda_nf4_gemv_bf16", p(b["attn"]), p(w["o_packed"]), p(w["o_absmax"]), 0, p(x), p(b["h"]),
                        1, HIDDEN, HIDDEN, 64, st)
            native.call("kudacuda_qwen2_mlp_nf4_bf16", p(b["h"]), p(w["post_norm"]), p(w["gate_packed"]),
                        p(w["gate_absmax"]), p(w["up_packed"]), p(w["up_absmax"]), p(w["down_packed"]),
                        p(w["down_absmax"]), p(b["mid"]), p(b["h"]), p(b["y"]), 1, HIDDEN, INTER, 64, EPS, st)
            x = b["y"]

    native.call("kudacuda_begin_capture", st)
    record()
    native.call("kudacuda_end_capture", st)
    return {"native": native, "stream": stream, "layers": layers, "caches": caches, "rope": (cos, sin), "x0": x0,
            "buffers": b, "position": position, "length": length}


# -------------------------------------------------------------------- run
def run(s: dict):
    kind, case = s["kind"], s["case"]
    if kind == "decode":
        dec = s["dec"]
        with torch.cuda.stream(dec.stream):
            dec.control.copy_(s["begin"])
        dec.native.check(dec.native.lib.kudacuda_qwen2_model_set_position(dec.model, s["step"]), "set_position")
        dec.replay(1)
        return {"logits": dec.logits, "hidden": dec.hidden, "tokens": dec.tokens,
                "key_cache": dec.layers[-1]["key_cache"], "value_cache": dec.layers[-1]["value_cache"]}
    if kind == "prefill":
        dec = s["dec"]
        if case["start"] == 0:
            dec.prefill(s["prompt"])
        else:
            dec.native.check(dec.native.lib.kudacuda_qwen2_model_prefill(
                dec.model, s["workspace"].data_ptr(), s["nbytes"], case["start"], case["count"],
                dec.stream.cuda_stream), "prefill")
        return {"logits": dec.logits, "tokens": dec.tokens, "key_caches": [w["key_cache"] for w in dec.layers],
                "value_caches": [w["value_cache"] for w in dec.layers]}
    if kind == "layers":
        s["native"].call("kudacuda_replay_graph", s["stream"].cuda_stream)
        return {"out": s["buffers"]["y"], "caches": [list(c) for c in s["caches"]]}
    native, stream, p = _native(), torch.cuda.current_stream().cuda_stream, torch.Tensor.data_ptr
    if kind == "qkv":
        (qw, qa), (kw, ka), (vw, va) = s["w"]
        name = "kudacuda_qwen2_fused_rmsnorm_qkv_nf4" + ("_bf16" if case["dtype"] == "bf16" else "")
        native.call(name, p(s["x"]), p(s["gamma"]), p(qw), p(qa), p(s["bias"][0]), p(kw), p(ka), p(s["bias"][1]),
                    p(vw), p(va), p(s["bias"][2]), *[p(o) for o in s["out"]], 1, HIDDEN, Q_OUT, KV_OUT, 64, EPS,
                    stream)
        return s["out"]
    if kind == "gqa":
        name = "kudacuda_qwen2_gqa_decode" + ("_graph" if case["mode"] == "graph" else "")
        name += "_bf16" if case["dtype"] == "bf16" else ""
        tail = (p(s["length"]), stream) if case["mode"] == "graph" else (stream,)
        native.call(name, p(s["q"]), p(s["k"]), p(s["v"]), p(s["out"]), 1, 1, case["capacity"], HEADS, KV_HEADS, DIM,
                    SCALE, *tail)
        return s["out"]
    if kind == "lm_head":
        native.call("kudacuda_lm_head_argmax_bf16", p(s["x"]), p(s["gamma"]), p(s["w"]), p(s["logits"]), p(s["token"]),
                    case["vocab"], HIDDEN, EPS, stream)
        return {"logits": s["logits"], "token": s["token"]}
    if kind == "gemm":
        (w, a), e = s["w"][0], case["epilogue"]
        native.call("kudacuda_nf4_gemm_bf16", p(s["x"]), p(w), p(a), p(s["bias"]) if e == "bias" else 0,
                    p(s["residual"]) if e == "residual" else 0, p(s["out"]), case["tokens"], case["k"], case["n"], 64,
                    stream)
        return s["out"]
    if kind == "gemm_swiglu":
        (gw, ga), (uw, ua) = s["w"]
        native.call("kudacuda_nf4_gemm_swiglu_bf16", p(s["x"]), p(gw), p(ga), p(uw), p(ua), p(s["out"]),
                    case["tokens"], case["k"], case["n"], 64, stream)
        return s["out"]
    n = case["n"] * case["k"]
    if kind == "dequantize":
        w, a = s["w"]
        native.call("kudacuda_nf4_dequantize", p(w), p(a), n, 64, KINDS[case["dtype"]], p(s["out"]), stream)
        return s["out"]
    native.call("kudacuda_nf4_quantize", p(s["w"]), KINDS[case["dtype"]], n, 64, p(s["packed"]), p(s["absmax"]),
                stream)
    return {"packed": s["packed"], "absmax": s["absmax"]}


# ------------------------------------------------------------------- work
def _nf4_bytes(n: int, k: int) -> int:
    return n * k // 2 + n * k // 64 * 4


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("decode", "layers"):
        layers = LAYERS if kind == "decode" else case["layers"]
        kv = 1024 * (case["cached"] + 1)
        vocab = VOCAB if kind == "decode" else 0
        return {"bytes": layers * (_nf4_bytes(1, LAYER_ELEMENTS) + kv) + vocab * (2 * HIDDEN + 2),
                "flops": layers * (2 * LAYER_ELEMENTS + 4 * HEADS * DIM * (case["cached"] + 1)) + 2 * vocab * HIDDEN}
    if kind == "prefill":
        m, start = case["count"], case["start"]
        pairs = m * start + m * (m + 1) // 2
        return {"bytes": PART_LAYERS * (_nf4_bytes(1, LAYER_ELEMENTS) + 1024 * (start + m)) + m * 2 * HIDDEN
                + PART_VOCAB * (2 * HIDDEN + 2),
                "flops": PART_LAYERS * (2 * m * LAYER_ELEMENTS + 4 * HEADS * DIM * pairs) + 2 * PART_VOCAB * HIDDEN}
    if kind == "qkv":
        n = Q_OUT + 2 * KV_OUT
        return {"bytes": _nf4_bytes(n, HIDDEN) + 2 * (2 * HIDDEN + 2 * n), "flops": 2 * n * HIDDEN}
    if kind == "gqa":
        return {"bytes": 1024 * case["cached"] + 4 * HEADS * DIM, "flops": 4 * HEADS * DIM * case["cached"]}
    if kind == "lm_head":
        return {"bytes": case["vocab"] * (2 * HIDDEN + 2) + 4 * HIDDEN, "flops": 2 * case["vocab"] * HIDDEN}
    n, k = case["n"], case["k"]
    if kind in ("gemm", "gemm_swiglu"):
        m, weights = case["tokens"], 2 if kind == "gemm_swiglu" else 1
        extra = 2 * m * n if case.get("epilogue") == "residual" else 2 * n if case.get("epilogue") == "bias" else 0
        return {"bytes": weights * _nf4_bytes(n, k) + 2 * m * (k + n) + extra, "flops": 2 * m * n * k * weights}
    return {"bytes": _nf4_bytes(n, k) + n * k * DTYPES[case["dtype"]].itemsize, "flops": n * k}


# -------------------------------------------------------------- tolerance
def tolerance(case: dict):
    """About four times what each path differs by from 64-bit sums: the rounding
    of its 16-bit outputs, of the 16-bit weights that the multi-token products
    take, and in a chain of layers what those add up to on the way."""

    kind = case["kind"]
    if kind in ("dequantize", "quantize"):
        return "exact"  # one rounding of one product; comparisons
    if kind == "decode":
        return {"rel": 0.03, "max": 0.5, "differ": 0.005}  # 36 layers: a changed rounding grows through all of them
    if kind == "prefill":
        return {"rel": 0.03, "max": 0.5, "differ": 0.01}  # 9 layers
    if kind == "layers":
        return {"rel": 0.02, "max": 0.2}
    if kind in ("qkv", "gqa") and case["dtype"] == "fp16":
        return {"rel": 1e-3, "max": 1e-2}
    if kind == "lm_head":
        return {"rel": 8e-3, "max": 4e-2, "differ": 0.0}
    return {"rel": 8e-3, "max": 6e-2}


# ------------------------------------------------------------------ exact
def _norm64(x: torch.Tensor, gamma: torch.Tensor) -> torch.Tensor:
    return x / (x.square().mean(dim=-1, keepdim=True) + EPS).sqrt() * gamma.double()


def _attend64(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, start: int) -> torch.Tensor:
    """Causal attention of rows q [m, 16, 128] at positions start .. over k, v [2, start + m, 128]."""

    m, total = q.shape[0], k.shape[1]
    hidden = torch.arange(total, device=DEV)[None] > start + torch.arange(m, device=DEV)[:, None]
    out = torch.empty_like(q)
    for h in range(HEADS):
        g = h // (HEADS // KV_HEADS)
        scores = (q[:, h] @ k[g].T) * SCALE
        out[:, h] = scores.masked_fill(hidden, -math.inf).softmax(dim=-1) @ v[g]
    return out.reshape(m, HEADS * DIM)


def _layers64(x: torch.Tensor, seed: int, layers: int, caches: list, start: int, capacity: int):
    """x [m, 2048] at positions start .. through the layers; the caches with their new rows, as the path lays them out."""

    m = x.shape[0]
    cos, sin = (t[start:start + m, None].double() for t in _rope(capacity))

    def rotate(t):
        lo, hi = t[..., :64], t[..., 64:]
        return torch.cat([lo * cos - hi * sin, hi * cos + lo * sin], dim=-1)

    done = []
    for i in range(layers):
        w = _layer(seed, i)

        def times(t, name):
            return t @ _dense(w[f"{name}_packed"], w[f"{name}_absmax"], *SHAPES[name]).T

        xn = _norm64(x, w["input_norm"])
        q, k, v = (times(xn, n) + w[f"{n}_bias"].double() for n in ("q", "k", "v"))
        q, k = rotate(q.reshape(m, HEADS, DIM)), rotate(k.reshape(m, KV_HEADS, DIM))
        kc, vc = (c.double() for c in caches[i])
        kc[:, start:start + m] = k.transpose(0, 1)
        vc[:, start:start + m] = v.reshape(m, KV_HEADS, DIM).transpose(0, 1)
        x = x + times(_attend64(q, kc[:, :start + m], vc[:, :start + m], start), "o")
        xn = _norm64(x, w["post_norm"])
        x = x + times(torch.nn.functional.silu(times(xn, "gate")) * times(xn, "up"), "down")
        done.append((kc, vc))
    return x, done


def exact(case: dict, seed: int):
    kind, gen = case["kind"], _gen(seed)
    if kind in ("decode", "prefill"):
        if kind == "decode":
            layers, vocab, start, m, capacity = LAYERS, VOCAB, case["cached"], 1, case["capacity"]
            ids = _tokens(seed, start + 1, vocab)[start:]
        else:
            layers, vocab, start, m = PART_LAYERS, PART_VOCAB, case["start"], case["count"]
            capacity = -(-(start + m + 1) // 64) * 64
            ids = _tokens(seed, start + m, vocab)[start:]
        embed, norm = _embedding(seed, vocab)
        caches = []
        for i in range(layers):
            pair = _caches(seed, i, capacity)
            for c in pair:
                c[:, start:] = 0
            caches.append(pair)
        x = embed[torch.from_numpy(ids.astype(np.int64)).to(DEV)].double()
        x, caches = _layers64(x, seed, layers, caches, start, capacity)
        logits = _norm64(x[-1:], norm)[0] @ embed.double().T
        if kind == "decode":
            return {"logits": logits, "hidden": x[-1], "tokens": None, "key_cache": caches[-1][0],
                    "value_cache": caches[-1][1]}
        return {"logits": logits, "tokens": None, "key_caches": [c[0] for c in caches],
                "value_caches": [c[1] for c in caches]}
    if kind == "layers":
        caches = [_caches(seed, i, case["capacity"]) for i in range(case["layers"])]
        x, caches = _layers64(_normal(gen, HIDDEN).double()[None], seed, case["layers"], caches, case["cached"],
                              case["capacity"])
        return {"out": x[0], "caches": [list(c) for c in caches]}
    if kind == "quantize":
        return None  # whole numbers and maxima
    s = prepare(case, seed)
    if kind == "qkv":
        xn = _norm64(s["x"].double(), s["gamma"])
        return [_dense(w, a, n, HIDDEN) @ xn + b.double()
                for (w, a), b, n in zip(s["w"], s["bias"], (Q_OUT, KV_OUT, KV_OUT))]
    if kind == "gqa":
        k, v = (t[:, :case["cached"]].double() for t in (s["k"], s["v"]))
        return _attend64(s["q"].double()[None], k, v, case["cached"] - 1).reshape(HEADS, DIM)
    if kind == "lm_head":
        return {"logits": s["w"].double() @ _norm64(s["x"].double(), s["gamma"]), "token": None}
    if kind == "dequantize":
        return _dense(*s["w"], case["n"], case["k"])
    products = [s["x"].double() @ _dense(w, a, case["n"], case["k"]).T for w, a in s["w"]]
    if kind == "gemm_swiglu":
        return torch.nn.functional.silu(products[0]) * products[1]
    if case["epilogue"] == "residual":
        return products[0] + s["residual"].double()
    return products[0] + s["bias"].double() if case["epilogue"] == "bias" else products[0]
