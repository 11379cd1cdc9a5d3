"""The GEMM dispatch (csrc/kc_gemm_plan.h) on the host.

Over a wide grid every plan is one its launcher has: blocks within the chip
where the rule says one round, partial tiles within the scratch, no empty split,
pairs and rotations only in shapes that hold both fragments.
"""

from __future__ import annotations

import pytest

from tests import _gemm_plan as P

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


@pytest.mark.parametrize("epilogue", POSSIBLE)
def test_plans_are_ones_their_launchers_have(epilogue):
    rows = {"qkv_rope": (2560,), "residual_norm": (2048,)}.get(epilogue, (64, 192, 1024, 2048, 8256, 11008, 22016))
    depths = {"qkv_rope": (2048,), "residual_norm": (2048, 11008)}.get(epilogue, (128, 256, 384, 1152, 2048, 4352, 11008))
    counts = [*range(1, 140), *range(140, 1100, 31), 1999, 2049, 4096, 8192]
    for n in rows:
        for k in depths:
            for m in counts:
                shape, tokens, splits = P.plan(epilogue, m, n, k)
                where = (m, n, k, shape, tokens, splits)
                if shape == "parts":
                    assert m <= 64 and k % 256 != 0, where
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
