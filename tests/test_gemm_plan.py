"""The GEMM dispatch (csrc/kc_gemm_plan.h) on the host.

The sizes of the GPU tests reach the block shapes and splits that they are there
for, and over a wide grid every plan is one its launcher has: blocks within the
chip where the rule says one round, partial tiles within the scratch, no empty
split, pairs and rotations only in shapes that hold both fragments.
"""

from __future__ import annotations

import pytest

from tests import _gemm_plan as P
from tests import test_gpu_few_gemm as few
from tests import test_gpu_tile_gemm as tile

pytestmark = pytest.mark.skipif(not P.LIBRARY.exists(), reason="native checks not built (python tests/native/build.py)")
SCRATCH_FLOATS = 4 << 20
FEW = ("few1", "few2", "few3", "few3x128")
POSSIBLE = {
    "plain": ("few1", "few2", "few3", "low", "square", "wide"),
    "residual": ("few1", "few2", "few3", "low", "square", "wide"),
    "residual_norm": ("few1", "few2", "low", "square", "wide"),
    "swiglu": (*FEW, "pair", "wide"),
    "qkv_rope": ("few1", "few2", "square", "pair", "wide"),
}


def test_gpu_cases_reach_their_shapes():
    for epilogue, cases in (("plain", tile.PLANS), ("residual", tile.PLANS), ("swiglu", tile.SWIGLU_PLANS),
                            ("swiglu", tile.EXACT_PLANS), ("plain", few.PLANS), ("residual", few.PLANS),
                            ("swiglu", few.SWIGLU_PLANS)):
        for size, (shape, splits) in cases.items():
            assert P.plan(epilogue, *size)[::2] == (shape, splits), (epilogue, size)
    for count, (shape, splits) in tile.PREFILL_PLANS.items():
        assert P.plan("qkv_rope", count, 2560, 2048)[::2] == (shape, splits), count


def test_gpu_cases_reach_every_shape():
    """... split and unsplit, with several windows a split, where a plan can be."""

    def reached(cases):
        return {(shape, splits > 1) for (_, _, k), (shape, splits) in cases.items()
                if k // P.WINDOW[shape] > splits}

    assert reached(tile.PLANS) >= {("low", False), ("low", True), ("square", False), ("square", True), ("wide", False)}
    assert reached(tile.SWIGLU_PLANS) >= {("pair", False), ("pair", True), ("wide", False)}
    assert reached(few.PLANS) >= {("few1", False), ("few1", True), ("few2", False), ("few2", True), ("few3", False)}
    assert reached(few.SWIGLU_PLANS) >= {("few1", False), ("few1", True), ("few2", True), ("few3", False), ("few3x128", False)}


@pytest.mark.parametrize("epilogue", POSSIBLE)
def test_plans_are_ones_their_launchers_have(epilogue):
    rows = {"qkv_rope": (2560,), "residual_norm": (2048,)}.get(epilogue, (64, 192, 1024, 2048, 8256, 11008, 16384, 22016))
    depths = {"qkv_rope": (2048,), "residual_norm": (2048, 11008)}.get(epilogue, (128, 256, 384, 1152, 2048, 4352, 11008))
    counts = [*range(1, 140), *range(140, 1100, 31), 1999, 2049, 4096, 8192]
    for n in rows:
        for k in depths:
            for m in counts:
                shape, tokens, splits = P.plan(epilogue, m, n, k)
                where = (m, n, k, shape, tokens, splits)
                if shape == "parts":  # no whole steps, or all CUs full of two fragments and little k
                    full = n // (16 if epilogue == "swiglu" else 32) >= 512
                    assert m <= 64 and k % 256 != 0 or m <= 16 and k <= 1024 and full, where
                    continue
                assert shape in POSSIBLE[epilogue], where
                assert splits == 1 or (2 if epilogue == "swiglu" else 1) * splits * m * n <= SCRATCH_FLOATS, where
                steps = k // P.WINDOW[shape]
                assert k % P.WINDOW[shape] == 0 and 1 <= splits <= steps, where
                if shape in FEW:
                    outputs = P.ROWS[shape] // (2 if epilogue == "swiglu" else 1)
                    blocks = -(-n // outputs) * -(-m // tokens) * splits
                    assert m <= 64 or blocks <= 256, where
                else:
                    per = -(-steps // splits)  # windows of a split
                    assert (splits - 1) * per < steps, where
                    assert epilogue != "qkv_rope" or shape != "square" or splits > 1, where


def test_unaligned_buffers_go_in_parts():
    for epilogue in ("plain", "residual", "swiglu"):
        assert P.plan(epilogue, 100, 192, 2048, offset=8)[0] == "parts"
        assert P.plan(epilogue, 100, 192, 2048)[0] != "parts"
