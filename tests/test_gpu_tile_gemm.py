"""GPU: the NF4 GEMM for more than 64 tokens (csrc/kc_gemm.hip).

Sizes pick every block shape of its dispatch and the edges of each: a last
token tile with one token, a last row tile half empty, one K window, an odd
number of windows, split and unsplit K.  Beside each stands what the dispatch
makes of it: (shape, splits of K), which tests/test_gemm_plan.py checks.  The reference sums the same
bf16-rounded weights in fp64; the bound is one bf16 step of the output
(tests/test_gpu_prefill.py::_close).
"""

from __future__ import annotations

import numpy as np
import pytest

from oracle import oracle as O
from tests._gpu_util import dev, empty, host, p
from tests.test_gpu_prefill import _acts, _bf16_ulps_apart, _close, _weights

pytestmark = pytest.mark.gpu
SEED = 20260901


PLANS = {
    (65, 64, 128): ("low", 1),       # one window a K-group, half a row tile, one token in the last tile
    (129, 192, 2048): ("few1", 8),   # (the few-token kernel)
    (300, 320, 384): ("low", 3),     # one window a split
    (300, 1088, 1152): ("low", 5),   # nine windows over five splits, half a row tile
    (300, 3328, 1152): ("low", 1),   # nine windows
    (100, 11008, 2048): ("low", 1),  # 16 windows
    (300, 192, 4224): ("square", 33),
    (257, 2112, 4224): ("square", 5),   # half a row tile
    (300, 1152, 4224): ("square", 9),   # 33 windows over nine splits
    (1100, 2048, 4224): ("square", 1),  # 33 windows, the residual stream's down projection
    (705, 6208, 128): ("wide", 1),   # two windows, a quarter of the last row tile
    (1025, 4160, 384): ("wide", 1),  # one token in the last tile
}
SWIGLU_PLANS = {
    (65, 64, 256): ("few1", 1),      # (the few-token kernel)
    (65, 64, 1152): ("pair", 9),     # one window a split
    (127, 192, 128): ("pair", 1),    # one window a K-group
    (200, 2048, 1152): ("pair", 3),  # nine windows over three splits
    (300, 3840, 640): ("pair", 1),   # five windows
    (1100, 1984, 128): ("wide", 1),  # half the last row tile
    (1025, 1920, 384): ("wide", 1),  # six windows, one token in the last tile
}
EXACT_PLANS = {
    (64, 8192, 256): ("few2", 1),
    (500, 3968, 128): ("pair", 1),
    (300, 11008, 128): ("wide", 1),
}
# one layer's q, k and v
PREFILL_PLANS = {
    200: ("few2", 1),
    301: ("few2", 1),
    385: ("square", 3),  # one token in the last tile
    641: ("square", 2),
    900: ("pair", 1),
    1700: ("wide", 1),
}


@pytest.mark.parametrize("m,n,k", PLANS)
@pytest.mark.parametrize("epi", ["plain", "bias", "residual"])
def test_nf4_gemm_of_many_tokens_matches_fp64(torch_gpu, native, stream, m, n, k, epi):
    torch = torch_gpu
    rng = np.random.default_rng([SEED, m, n, k])
    print(f"nf4_gemm m={m} n={n} k={k} epi={epi}", flush=True)
    packed, absmax, wbf = _weights(rng, n, k)
    xb, x = _acts(rng, m, k)
    acc = (x @ wbf.T).astype(np.float32)
    bias = O.f32_to_bf16((rng.standard_normal(n) * 0.02).astype(np.float32))
    res = O.f32_to_bf16(rng.standard_normal((m, n)).astype(np.float32))
    want = {"plain": acc, "bias": acc + O.bf16_to_f32(bias),
            "residual": O.bf16_to_f32(res) + O.bf16_to_f32(O.f32_to_bf16(acc))}[epi]
    d_x, d_w, d_a, d_b = (dev(torch, t) for t in (xb, packed, absmax, bias))
    out = dev(torch, res) if epi == "residual" else empty(torch, m * n, "u16")  # residual in place
    native.call("kudacuda_nf4_gemm_bf16", p(d_x), p(d_w), p(d_a), p(d_b) if epi == "bias" else 0,
                p(out) if epi == "residual" else 0, p(out), m, k, n, 64, stream.cuda_stream)
    stream.synchronize()
    _close(host(out).reshape(m, n), want, inner=acc if epi == "residual" else None)


@pytest.mark.parametrize("m,n,k", SWIGLU_PLANS)
def test_nf4_gemm_swiglu_of_many_tokens_matches_fp64(torch_gpu, native, stream, m, n, k):
    torch = torch_gpu
    rng = np.random.default_rng([SEED, 7, m, n, k])
    print(f"nf4_gemm_swiglu m={m} n={n} k={k}", flush=True)
    gp, ga, gw = _weights(rng, n, k, std=0.06)
    up, ua, uw = _weights(rng, n, k, std=0.06)
    xb, x = _acts(rng, m, k)
    want = O.silu((x @ gw.T).astype(np.float32)) * (x @ uw.T).astype(np.float32)
    out = empty(torch, m * n, "u16")
    bufs = [dev(torch, t) for t in (xb, gp, ga, up, ua)]
    native.call("kudacuda_nf4_gemm_swiglu_bf16", *[p(b) for b in bufs], p(out), m, k, n, 64, stream.cuda_stream)
    stream.synchronize()
    _close(host(out).reshape(m, n), want)


@pytest.mark.parametrize("m,n,k", EXACT_PLANS)
def test_swiglu_of_exact_sums_is_the_oracles(torch_gpu, native, stream, m, n, k):
    """Each token has two elements, powers of two 9 bits apart: the sums are exact,
    so every output is bf16(silu(gate) * up) of the oracle's fp32 silu to the bit,
    in every kernel (a silu 1 ulp off moves about 1 output in 80,000).  The gates
    of the last token are large enough for either branch of the silu."""

    torch = torch_gpu
    rng = np.random.default_rng([SEED, 8, m, n, k])
    print(f"nf4_gemm_swiglu of two-element tokens m={m} n={n} k={k}", flush=True)
    gp, ga, gw = _weights(rng, n, k, std=0.06)
    up, ua, uw = _weights(rng, n, k, std=0.06)
    x = np.zeros((m, k), np.float32)
    scale = 2.0 ** rng.integers(0, 6, m)
    scale[-1] = 2.0 ** 11
    at = rng.integers(0, k // 2, m)
    x[np.arange(m), at] = scale
    x[np.arange(m), at + k // 2] = scale * 2.0 ** -9
    gate, upv = (x.astype(np.float64) @ w.T for w in (gw, uw))
    for sums in (gate, upv):
        assert np.array_equal(sums, sums.astype(np.float32))
    assert np.abs(gate[-1]).max() > 128
    out = empty(torch, m * n, "u16")
    bufs = [dev(torch, t) for t in (O.f32_to_bf16(x), gp, ga, up, ua)]
    native.call("kudacuda_nf4_gemm_swiglu_bf16", *[p(b) for b in bufs], p(out), m, k, n, 64, stream.cuda_stream)
    stream.synchronize()
    got = O.bf16_to_f32(host(out).reshape(m, n))
    want = O.bf16_to_f32(O.f32_to_bf16(O.silu(gate.astype(np.float32)) * upv.astype(np.float32)))
    print(f"{int(np.count_nonzero(got != want))} of {got.size} differ", flush=True)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("count", PREFILL_PLANS)
def test_prefill_rows_equal_those_of_64_token_parts(torch_gpu, native, count):
    """One layer: a long prompt at once (q, k, v in the blocks of PREFILL_PLANS)
    writes the cache rows that its 64-token parts write, to the bound of
    test_gpu_prefill (0.2 % of the elements more than one bf16 step apart)."""

    from kudacuda_amd import synthetic
    from kudacuda_amd.qwen2_decoder import Qwen2Nf4Decoder

    torch = torch_gpu
    gpu = Qwen2Nf4Decoder.synthetic(native, torch, seed=SEED, num_layers=1, vocab=512, kv_capacity=1728,
                                    token_capacity=1728)
    try:
        lib = native.lib
        prompt = synthetic.prompt_ids(SEED, count, 512)
        print(f"prefill of {count} tokens in 64-token parts and at once", flush=True)
        nbytes = int(lib.kudacuda_qwen2_prefill_workspace_bytes(64))
        ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda:0")
        gpu.reset(prompt)
        for start in range(0, count, 64):
            part = min(64, count - start)
            native.check(lib.kudacuda_qwen2_model_prefill(gpu.model, ws.data_ptr(), nbytes, start, part,
                                                          gpu.stream.cuda_stream), "prefill")
        gpu.stream.synchronize()
        names = ("key_cache", "value_cache")
        parts = [O.bf16_to_f32(host(gpu.layers[0][n]).reshape(2, -1, 128)[:, :count]) for n in names]
        logits = O.bf16_to_f32(host(gpu.logits))
        for n in names:
            gpu.layers[0][n].zero_()
        torch.cuda.synchronize()
        gpu.prefill(prompt)
        gpu.stream.synchronize()
        for n, want in zip(names, parts):
            got = O.bf16_to_f32(host(gpu.layers[0][n]).reshape(2, -1, 128)[:, :count])
            far = int(np.count_nonzero(_bf16_ulps_apart(got, want) > 1))
            print(f"{n}: {far} of {got.size} more than one bf16 step apart", flush=True)
            assert far <= 0.002 * got.size
        assert float(np.abs(O.bf16_to_f32(host(gpu.logits)) - logits).max()) <= 0.03
    finally:
        gpu.close()
