"""GPU: the prefill's causal attention on the matrix cores (csrc/kc_prefill_attn.hip).

A one-layer model is prefilled; the workspace then holds the layer's rotated
queries and attention output (rows of 2048 bf16 after `hidden` and the
normalised rows), and the caches its keys and values.  The output is compared
with the fp64 softmax of those, to one bf16 step
(tests/test_gpu_prefill.py::_close).  Cache rows past the prompt hold NaN.
"""

from __future__ import annotations

import numpy as np
import pytest

from oracle import oracle as O
from tests._gpu_util import host
from tests.test_gpu_prefill import _close

pytestmark = pytest.mark.gpu
SEED = 20260902
CAPACITY = 2304


@pytest.fixture(scope="module")
def layer(torch_gpu, native):
    from kudacuda_amd.qwen2_decoder import Qwen2Nf4Decoder

    gpu = Qwen2Nf4Decoder.synthetic(native, torch_gpu, seed=SEED, num_layers=1, vocab=512, kv_capacity=CAPACITY,
                                    token_capacity=CAPACITY)
    yield gpu
    gpu.close()


def _prefill(torch, native, gpu, start, count, marked=None, cached=None):
    """Random cache rows [0, start), NaN from there on, then what ``cached`` puts
    there; prefill of count tokens; returns (attention output, q, K, V) as bf16 bits / fp64 values."""

    rng = np.random.default_rng([SEED, start, count])
    for name in ("key_cache", "value_cache"):
        rows = torch.full((2, CAPACITY, 128), float("nan"), dtype=torch.bfloat16)
        rows[:, :start] = torch.from_numpy(rng.standard_normal((2, start, 128)).astype(np.float32)).bfloat16()
        gpu.layers[0][name].copy_(rows)
    if cached is not None:
        cached()
    prompt = rng.integers(1, 512, size=start + count, dtype=np.int64).astype(np.int32)
    if marked is not None:
        prompt[start + marked] = 0
    gpu.reset(prompt)
    nbytes = int(native.lib.kudacuda_qwen2_prefill_workspace_bytes(count))
    ws = torch.zeros(nbytes, dtype=torch.uint8, device="cuda:0")
    torch.cuda.synchronize()
    native.check(native.lib.kudacuda_qwen2_model_prefill(gpu.model, ws.data_ptr(), nbytes, start, count,
                                                         gpu.stream.cuda_stream), "prefill")
    gpu.stream.synchronize()
    rows = ws[: count * 4 * 2048 * 2].view(torch.int16).reshape(4, count, 2048)
    kv = [O.bf16_to_f32(host(gpu.layers[0][n]).reshape(2, CAPACITY, 128)[:, : start + count]).astype(np.float64)
          for n in ("key_cache", "value_cache")]
    q = O.bf16_to_f32(host(rows[2]).reshape(count, 16, 128)).astype(np.float64)
    return host(rows[3]), q, kv[0], kv[1]


def _attention(q, k, v, start):
    count = q.shape[0]
    out = np.empty((count, 16, 128))
    hidden = np.arange(start + count)[None, :] > start + np.arange(count)[:, None]
    for h in range(16):
        s = q[:, h] @ k[h // 8].T / np.sqrt(128.0)
        s = np.where(hidden, -np.inf, s)
        p = np.exp(s - s.max(axis=1, keepdims=True))
        out[:, h] = (p / p.sum(axis=1, keepdims=True)) @ v[h // 8]
    return out.reshape(count, 2048)


@pytest.mark.parametrize("start,count", [
    (0, 129),     # two windows, a token tile of one row
    (128, 1),     # one row, one key of the second window
    (127, 2),     # rows on both sides of a window's end
    (255, 9),     # two token tiles over three windows, split keys
    (1000, 7),    # 8 splits: merged by one thread per (head, dims)
    (2000, 40),   # 16 splits: merged in groups; partly filled tile
    (64, 641),    # many tiles, few splits of uneven length
    (0, 2250),    # unsplit
])
def test_prefill_attention_matches_fp64(torch_gpu, native, layer, start, count):
    print(f"prefill attention of {count} tokens after {start}", flush=True)
    got, q, k, v = _prefill(torch_gpu, native, layer, start, count)
    _close(got, _attention(q, k, v, start))


@pytest.mark.parametrize("start,count,marked", [(0, 150, 140), (1500, 20, 3)])
def test_a_later_token_of_nan_leaves_earlier_rows_alone(torch_gpu, native, layer, start, count, marked):
    """A token whose embedding is NaN has NaN keys and values: rows before it
    have none of it (unsplit and split keys), rows from it on are NaN."""

    print(f"prefill attention of {count} tokens after {start}, NaN at {marked}", flush=True)
    clean = layer.embed[0].clone()
    layer.embed[0].fill_(float("nan"))
    try:
        got, q, k, v = _prefill(torch_gpu, native, layer, start, count, marked)
    finally:
        layer.embed[0].copy_(clean)
    end = start + marked
    _close(got[:marked], _attention(q[:marked], k[:, :end], v[:, :end], start))
    assert np.isnan(O.bf16_to_f32(got[marked:])).all()


def _parts(w):
    """fp32 values as two bf16 parts, each rounded to nearest: (their sum - w) / w."""

    hi = O.bf16_to_f32(O.f32_to_bf16(w))
    lo = O.bf16_to_f32(O.f32_to_bf16(w - hi))
    return (hi.astype(np.float64) + lo - w) / w


@pytest.mark.parametrize("start,count", [
    (200, 1),     # two windows, split keys and their merge
    (150, 2100),  # unsplit
])
def test_softmax_weights_have_all_their_bits(torch_gpu, native, layer, start, count):
    """Cached rows such that the first row's result nearly cancels: what is left
    shows the error of the weights, not the rounding of the output.

    One head's scores are exact (each K row has one element): key 0 scores 0, keys
    1 and 2 take the weights whose first 16 bits err most, one up, one down, with
    values of opposite sign; keys 3 to 5, of ever smaller weight, cancel the rest,
    every other cached row weighs nothing.  In fp32 a weight is off by at most half
    an ulp of its argument (|y| < 4: 2^-23 ln 2), as much by the scale's rounding
    and an ulp of exp2 (2^-23), the sum by half an ulp for each of at most six
    additions: 2^-20 of the sum of |weight * value| in all.  Weights of 16 bits
    err by 2^-18."""

    rng = np.random.default_rng([SEED, 3, start])
    _, q, k, v = _prefill(torch_gpu, native, layer, start, count)
    scale = 1.0 / np.sqrt(128.0)
    own = np.array([q[0, h] @ k[h // 8, start] * scale for h in range(16)])
    head = int(own.argmin())
    assert own[head] < 0
    g, dim = head // 8, int(np.abs(q[0, head]).argmax())
    qd = q[0, head, dim]
    wanted = O.bf16_to_f32(O.f32_to_bf16((rng.uniform(-1.4, -0.1, 4000) / (qd * scale)).astype(np.float32)))
    err = _parts(np.exp(wanted.astype(np.float64) * qd * scale).astype(np.float32))
    rows = np.zeros((start, 128), np.float32)
    rows[:, dim] = -200.0 / (qd * scale)
    rows[:6] = 0.0
    rows[1, dim], rows[2, dim] = wanted[err.argmax()], wanted[err.argmin()]
    rows[3:6, dim] = np.array([-6.0, -12.0, -18.0]) / (qd * scale)
    keys = O.bf16_to_f32(O.f32_to_bf16(rows)).astype(np.float64)
    w = np.exp(np.append(keys[:, dim] * qd * scale, own[head]))
    values = np.zeros((start + 1, 128))
    values[6:start] = rng.standard_normal((start - 6, 128))
    values[1] = rng.uniform(1.0, 2.0, 128)
    values = O.bf16_to_f32(O.f32_to_bf16(values.astype(np.float32))).astype(np.float64)
    values[start] = v[g, start]
    for i in (2, 3, 4, 5):
        left = -(w @ values) / w[i]
        values[i] = O.bf16_to_f32(O.f32_to_bf16(left.astype(np.float32)))
    want = w @ values / w.sum()
    bound = 2.0**-20 * (w @ np.abs(values)) / w.sum() + 2.0**-8 * np.abs(want)

    def fill():
        for name, new in (("key_cache", keys), ("value_cache", values)):
            new = torch_gpu.from_numpy(new[:start].astype(np.float32)).bfloat16()
            layer.layers[0][name][g, :start].copy_(new)

    got, q2, k2, v2 = _prefill(torch_gpu, native, layer, start, count, cached=fill)
    assert np.array_equal(q2[0], q[0]) and np.array_equal(k2[g, :start + 1], np.vstack([keys, k[g, start]]))
    assert np.array_equal(v2[g, :start + 1], values)
    out = O.bf16_to_f32(got.reshape(count, 16, 128)[0, head]).astype(np.float64)
    off = np.abs(out - want)
    print(f"head {head}: largest error {float((off / bound).max()):.2f} of the bound", flush=True)
    assert (off <= bound).all()
