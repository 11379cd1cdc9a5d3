"""GPU: the NF4 GEMM for few tokens (csrc/kc_gemm_few.hip).

Sizes pick every block shape of its dispatch and the edges of each: one token, a
token tile full or with one token, a last block with dead fragments, one step of
K, fewer steps than prefetched, uneven splits.  Beside each stands what the
dispatch makes of it: (shape, splits of K), which tests/test_gemm_plan.py
checks.  The reference sums the same
bf16-rounded weights in fp64; the bound is one bf16 step of the output
(tests/test_gpu_prefill.py::_close).
"""

from __future__ import annotations

import numpy as np
import pytest

from oracle import oracle as O
from tests._gpu_util import dev, empty, host, p
from tests.test_gpu_prefill import _acts, _close, _weights

pytestmark = pytest.mark.gpu
SEED = 20260902


PLANS = {
    (1, 64, 256): ("few1", 1),       # one step, one token
    (32, 256, 2048): ("few1", 8),    # a full token tile
    (40, 192, 2816): ("few1", 8),    # eleven steps over eight splits
    (33, 2112, 1280): ("few1", 1),   # one token in the second tile, five steps
    (20, 9280, 256): ("few2", 1),
    (64, 16448, 512): ("few3", 1),   # one fragment dead in the last block
    (31, 16448, 768): ("few3", 1),   # the same, one token tile
    (64, 2048, 11008): ("few2", 8),  # a long k: 43 steps over eight splits
    (17, 64, 4352): ("few1", 8),     # a long k over few blocks
    (17, 2048, 4352): ("few2", 8),   # a long k, 17 steps, one token tile
    (193, 2048, 2304): ("few1", 1),  # four token tiles, one token in the last
    (200, 192, 4608): ("few1", 9),   # a long k over few blocks, four token tiles
    (100, 1088, 4352): ("few2", 7),  # a long k, two token tiles
    (512, 2048, 768): ("few2", 1),   # eight token tiles, three steps
}
SWIGLU_PLANS = {
    (1, 64, 256): ("few1", 1),        # one step, one token
    (1, 64, 1792): ("few1", 7),       # split: gate and up partials and their reduce
    (40, 128, 2816): ("few1", 8),     # eleven steps over eight splits
    (33, 1024, 4352): ("few2", 8),    # a long k: 17 steps over eight splits
    (40, 1024, 512): ("few1", 1),
    (64, 4160, 256): ("few2", 1),
    (32, 8256, 768): ("few3", 1),     # one token tile
    (63, 8256, 512): ("few3", 1),     # two token tiles
    (65, 8256, 256): ("few3x128", 1),   # one token past 64
    (128, 8192, 512): ("few3x128", 1),  # a full tile, two fragments alive in the last block
    (256, 512, 256): ("few1", 1),     # four token tiles
}


@pytest.mark.parametrize("m,n,k", PLANS)
@pytest.mark.parametrize("epi", ["plain", "bias", "residual"])
def test_nf4_gemm_of_few_tokens_matches_fp64(torch_gpu, native, stream, m, n, k, epi):
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
def test_nf4_gemm_swiglu_of_few_tokens_matches_fp64(torch_gpu, native, stream, m, n, k):
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
