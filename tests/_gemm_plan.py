"""Which kernel and block shape an NF4 GEMM takes (csrc/kc_gemm_plan.h)."""

from __future__ import annotations

import ctypes
from pathlib import Path

LIBRARY = Path(__file__).resolve().parent / "native" / "libgemm_plan.so"
EPILOGUES = {"plain": 0, "bias": 0, "residual": 1, "swiglu": 2, "qkv_rope": 3, "residual_norm": 4}
SHAPES = ("parts", "few1", "few2", "few3", "few3x128", "low", "square", "pair", "wide")
ROWS = {"few1": 32, "few2": 64, "few3": 96, "few3x128": 96, "low": 128, "square": 128, "pair": 128, "wide": 256}
WINDOW = {"few1": 256, "few2": 256, "few3": 256, "few3x128": 128, "low": 128, "square": 128, "pair": 128, "wide": 64}


def plan(epilogue: str, m: int, n: int, k: int, offset: int = 0) -> tuple[str, int, int]:
    """(shape, tokens of a block, splits of K); the output ``offset`` bytes off alignment."""

    out = (ctypes.c_int64 * 3)()
    sizes = [ctypes.c_int64(v) for v in (m, n, k, offset)]
    ctypes.CDLL(str(LIBRARY)).gemm_plan(EPILOGUES[epilogue], *sizes, out)
    return SHAPES[out[0]], out[1], out[2]
