"""GPU: NF4 quantise / dequantise by 8-element units against the oracle and,
where the unit kernels do not apply (small or odd counts, unaligned buffers),
against the element kernels.  Whole outputs, bit for bit."""

from __future__ import annotations

import numpy as np
import pytest

from oracle import oracle as O
from tests._gpu_util import dev, empty, host, p

pytestmark = pytest.mark.gpu
SEED = 20260903


# units from 393,216 elements on
@pytest.mark.parametrize("count", [64, 64 * 33, 64 * 257, 393216 - 64, 393216, 393216 + 64 * 33])
@pytest.mark.parametrize("dtype", [0, 1])
def test_quantize_units_match_the_oracle_and_the_element_kernel(torch_gpu, native, stream, count, dtype):
    torch = torch_gpu
    rng = np.random.default_rng([SEED, count, dtype])
    x = (rng.standard_normal(count) * 0.02).astype(np.float32)
    x[:64] = 0.0 if count > 64 else x[:64]
    src = O.f32_to_bf16(x) if dtype else x
    print(f"quantize {count} elements, dtype {dtype}", flush=True)

    def run(values, offset):
        # offset elements of padding: 0 is 16-byte aligned, 1 takes the element kernel
        buf = dev(torch, np.concatenate([np.zeros(offset, values.dtype), values]))[offset:]
        packed, absmax = empty(torch, count // 2, "u8"), empty(torch, count // 64, "f32")
        torch.cuda.synchronize()
        native.call("kudacuda_nf4_quantize", p(buf), dtype, count, 64, p(packed), p(absmax), stream.cuda_stream)
        stream.synchronize()
        return host(packed), host(absmax).view(np.uint32)

    got = run(src, 0)
    want = O.nf4_quantize(O.bf16_to_f32(src) if dtype else src)
    assert np.array_equal(got[0], want[0].reshape(-1)) and np.array_equal(got[1], want[1].reshape(-1).view(np.uint32))
    odd = src.copy()
    odd[[3, 40, 63]] = [0x7FC0, 0xFF80, 0x7F80] if dtype else [np.nan, -np.inf, np.inf]
    for values in (src, odd):
        for a, b in zip(run(values, 0), run(values, 1)):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("count,blocksize", [
    # units of each kind (from 524,288 elements on, to bf16 from 1,048,576): whole blocks of threads, one
    # unit past them, a ragged last block, other block sizes
    (1 << 20, 64), ((1 << 20) + 8, 64), ((1 << 20) + 64 * 515, 64), ((1 << 20) + 8, 128), ((1 << 20) + 2056, 1024),
    ((1 << 20) + 8, 8),
    (1 << 19, 64), ((1 << 19) - 8, 64),  # to fp32 and fp16 the first of units, the last of elements
    # odd counts, a block size that is no power of two: element by element
    ((1 << 20) + 1, 64), ((1 << 20) + 48, 48),
    # few elements: element by element
    (64, 64), (8, 8), (8192, 64), (8200, 64), (64 * 515, 64), (4096 + 8, 128), (2056, 1024), (8193, 64), (6, 64),
    (4096, 48),
])
@pytest.mark.parametrize("kind", [0, 1, 2])
def test_dequantize_units_and_elements_are_exact(torch_gpu, native, stream, count, blocksize, kind):
    torch = torch_gpu
    rng = np.random.default_rng([SEED, count, blocksize])
    print(f"dequantize {count} elements, blocks of {blocksize}, kind {kind}", flush=True)
    packed = rng.integers(0, 256, size=(count + 1) // 2, dtype=np.uint8)
    absmax = (rng.random(-(-count // blocksize)) * 0.1).astype(np.float32)
    codes = np.stack([packed >> 4, packed & 15], axis=1).reshape(-1)[:count]
    levels = O.nf4_dequantize(np.arange(256, dtype=np.uint8), np.ones(8, np.float32), 512)[:32].reshape(16, 2)[:, 1]
    values = levels[codes] * absmax[np.arange(count) // blocksize]
    want = [values.view(np.uint32), O.f32_to_bf16(values), values.astype(np.float16).view(np.uint16)][kind]
    d_p, d_a = dev(torch, packed), dev(torch, absmax)
    for offset in (0, 1):  # 1: the output is not 16-byte aligned
        out = empty(torch, count + offset, "f32" if kind == 0 else "u16")[offset:]
        torch.cuda.synchronize()
        native.call("kudacuda_nf4_dequantize", p(d_p), p(d_a), count, blocksize, kind, p(out), stream.cuda_stream)
        stream.synchronize()
        got = host(out)
        assert np.array_equal(got.view(np.uint32) if kind == 0 else got, want)
