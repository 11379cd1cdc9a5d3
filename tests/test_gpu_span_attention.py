"""GPU: the decode step's attention over splits of several rounds
(csrc/kc_gqa.hip, gqa_span_kernel_bf16), bit for bit against the oracle.

The steps cross into it from one-round splits, end a split inside a round and
inside a quad, fill a span of eight rounds and go on into a second one, and run it
by a stale position over a cache that needs one split, or one round a split.
"""

from __future__ import annotations

import pytest

from tests import test_gpu_decoder as decoder

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("start,capacity,mode", [
    (1021, 2048, "graph"),                          # 32 one-round splits -> 17 of two rounds
    (2045, 4096, "graph"),                          # two -> three rounds
    (8160, 8192, "graph"),                          # eight rounds: a whole span
    (8190, 9216, "graph"),                          # eight -> nine rounds: a second span
    (3, 1100, "graph, position stale high"),        # one split
    (700, 1100, "graph, position stale high"),      # one-round splits
])
def test_span_attention_matches_oracle(torch_gpu, native, start, capacity, mode):
    decoder.test_decode_from_a_seeded_long_cache_matches_oracle(torch_gpu, native, start, capacity, mode)
