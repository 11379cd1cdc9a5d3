"""GPU: the NF4 GEMM in launches of 64 tokens (csrc/kc_prefill.hip), which takes
the calls whose buffers are not aligned to 16 bytes, at up to 64 tokens a k that
is no multiple of 256, and at up to 16 tokens wide weights of little k; and the prefill over an unaligned workspace, which
runs all of its GEMMs there and its attention row by row at any length.
"""

from __future__ import annotations

import numpy as np
import pytest

from oracle import oracle as O
from tests._gpu_util import dev, host, p
from tests.test_gpu_prefill import _acts, _bf16_ulps_apart, _close, _weights

pytestmark = pytest.mark.gpu
SEED = 20260903


def _off(torch, bits, elements):
    """A device copy of 16-bit values that starts ``elements`` past an aligned address."""

    flat = torch.empty(bits.size + elements, dtype=torch.int16, device="cuda:0")
    out = flat[elements:]
    out.copy_(dev(torch, np.ascontiguousarray(bits).reshape(-1)))
    return out


# elements off alignment: 4 (8 bytes), which no other kernel takes; the last two need none
@pytest.mark.parametrize("m,n,k,elements", [(100, 192, 2048, 4), (129, 64, 384, 4), (40, 320, 256, 4), (33, 192, 128, 0),
                                            (16, 16448, 512, 0)])
@pytest.mark.parametrize("epi", ["plain", "bias", "residual", "swiglu"])
def test_gemm_in_parts_matches_fp64(torch_gpu, native, stream, m, n, k, elements, epi):
    torch = torch_gpu
    rng = np.random.default_rng([SEED, m, n, k])
    print(f"nf4_gemm in parts m={m} n={n} k={k} epi={epi}", flush=True)
    std = 0.06 if epi == "swiglu" else 0.02
    packed, absmax, wbf = _weights(rng, n, k, std)
    xb, x = _acts(rng, m, k)
    acc = (x @ wbf.T).astype(np.float32)
    d_x, d_w, d_a = _off(torch, xb, elements), dev(torch, packed), dev(torch, absmax)
    out = _off(torch, np.zeros(m * n, np.uint16), elements)
    if epi == "swiglu":
        up, ua, uw = _weights(rng, n, k, std)
        want, inner = O.silu(acc) * (x @ uw.T).astype(np.float32), None
        d_u, d_ua = dev(torch, up), dev(torch, ua)
        torch.cuda.synchronize()  # the uploads, before another stream reads them
        native.call("kudacuda_nf4_gemm_swiglu_bf16", p(d_x), p(d_w), p(d_a), p(d_u), p(d_ua), p(out), m, k, n, 64,
                    stream.cuda_stream)
    else:
        bias = O.f32_to_bf16((rng.standard_normal(n) * 0.02).astype(np.float32))
        res = O.f32_to_bf16(rng.standard_normal((m, n)).astype(np.float32))
        d_b = _off(torch, bias, 1)
        want = {"plain": acc, "bias": acc + O.bf16_to_f32(bias),
                "residual": O.bf16_to_f32(res) + O.bf16_to_f32(O.f32_to_bf16(acc))}[epi]
        inner = acc if epi == "residual" else None
        if epi == "residual":  # in place
            out.copy_(dev(torch, res.reshape(-1)))
        torch.cuda.synchronize()
        native.call("kudacuda_nf4_gemm_bf16", p(d_x), p(d_w), p(d_a), p(d_b) if epi == "bias" else 0,
                    p(out) if epi == "residual" else 0, p(out), m, k, n, 64, stream.cuda_stream)
    stream.synchronize()
    _close(host(out).reshape(m, n), want, inner=inner)


@pytest.mark.parametrize("start,count", [(0, 150), (130, 70)])
def test_prefill_over_an_unaligned_workspace(torch_gpu, native, start, count):
    """One layer, a workspace 8 bytes off alignment: cache rows and logits of the
    aligned run, to the bound of test_gpu_prefill (0.2 % of the elements more than
    one bf16 step apart; last-row logits within 0.03)."""

    from kudacuda_amd import synthetic
    from kudacuda_amd.qwen2_decoder import Qwen2Nf4Decoder

    torch = torch_gpu
    total = start + count
    gpu = Qwen2Nf4Decoder.synthetic(native, torch, seed=SEED, num_layers=1, vocab=512, kv_capacity=256,
                                    token_capacity=256)
    try:
        lib = native.lib
        nbytes = int(lib.kudacuda_qwen2_prefill_workspace_bytes(total))
        ws = torch.empty(nbytes + 16, dtype=torch.uint8, device="cuda:0")
        base = -(-ws.data_ptr() // 16) * 16
        results = []
        for offset in (0, 8):
            print(f"prefill of {count} tokens after {start}, workspace {offset} bytes off", flush=True)
            gpu.reset(synthetic.prompt_ids(SEED, total, 512))
            torch.cuda.synchronize()
            if start:
                native.check(lib.kudacuda_qwen2_model_prefill(gpu.model, base, nbytes, 0, start, gpu.stream.cuda_stream),
                             "prefill")
            native.check(lib.kudacuda_qwen2_model_prefill(gpu.model, base + offset, nbytes, start, count,
                                                          gpu.stream.cuda_stream), "prefill")
            gpu.stream.synchronize()
            results.append([O.bf16_to_f32(host(gpu.layers[0][n]).reshape(2, -1, 128)[:, :total])
                            for n in ("key_cache", "value_cache")] + [O.bf16_to_f32(host(gpu.logits))])
        for got, want in zip(results[1][:2], results[0][:2]):
            far = int(np.count_nonzero(_bf16_ulps_apart(got, want) > 1))
            print(f"{far} of {got.size} more than one bf16 step apart", flush=True)
            assert far <= 0.002 * got.size
        assert float(np.abs(results[1][2] - results[0][2]).max()) <= 0.03
    finally:
        gpu.close()
