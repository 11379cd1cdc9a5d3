"""GPU: the NF4 GEMM for few tokens (csrc/kc_gemm_few.hip).

Sizes pick every block shape of its dispatch and the edges of each: one token, a
token tile full or with one token, a last block with dead fragments, one step of
K, fewer steps than prefetched, uneven splits.  The reference sums the same
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


@pytest.mark.parametrize("m,n,k", [
    (1, 64, 256),        # one fragment a block, one step, one token
    (32, 256, 2048),     # split over blocks of one fragment, a full token tile
    (33, 2112, 1280),    # unsplit, one token in the second tile, five steps
    (20, 9280, 256),     # two fragments a block
    (64, 16448, 512),    # three fragments a block, one dead in the last block
    (31, 16448, 768),    # the same, one token tile
    (64, 2048, 11008),   # a long k: 43 steps over eight splits
    (17, 64, 4352),      # a long k over 17 steps, one token tile
    (193, 2048, 2304),   # four token tiles, one token in the last
    (200, 192, 4608),    # a long k, four token tiles
])
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


@pytest.mark.parametrize("m,n,k", [
    (1, 64, 256),       # one fragment a block, split
    (40, 1024, 512),    # unsplit
    (64, 4160, 256),    # two fragments a block
    (32, 8256, 768),    # three, one token tile
    (63, 8256, 512),    # three, two token tiles
    (65, 8256, 256),    # 128-token tiles, one token past 64
    (128, 8192, 512),   # a full one, two fragments alive in the last block
    (256, 512, 256),    # four token tiles
])
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
