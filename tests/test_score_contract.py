"""The score contract's quotient by one Markstein step (``contract`` of ``csrc/lmk_topk_slice.hpp``) against division, for every
16-bit value of both types and both head dims' square roots.  Steps are evaluated exactly and rounded once.
"""
from fractions import Fraction

import numpy as np
import pytest

f32 = np.float32


def _round(x: Fraction) -> np.float32:
    near = f32(float(x))                                       # within one place; the neighbours settle double rounding
    best = min((c for c in (np.nextafter(near, f32(-np.inf)), near, np.nextafter(near, f32(np.inf))) if np.isfinite(c)),
               key=lambda c: (abs(Fraction(float(c)) - x), int(c.view(np.uint32)) & 1))
    return best


def _to_type(x: np.float32, dtype: str) -> int:
    if dtype == "fp16":
        return int(np.float16(x).view(np.uint16))
    u = int(x.view(np.uint32))
    return (u + 0x7FFF + ((u >> 16) & 1)) >> 16


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("dim", [64, 128])
def test_one_step_rounds_to_the_quotient_for_every_value(dtype, dim):
    bits = np.arange(65536, dtype=np.uint32)
    values = (bits << 16).view(f32) if dtype == "bf16" else bits.astype(np.uint16).view(np.float16).astype(f32)
    s = f32(np.sqrt(float(dim)))
    y = f32(1.0) / s
    for x in values[np.isfinite(values)]:
        q = x * y
        r = _round(Fraction(float(x)) - Fraction(float(q)) * Fraction(float(s)))
        got = _round(Fraction(float(r)) * Fraction(float(y)) + Fraction(float(q))) if abs(r) > 0 else q
        assert _to_type(got, dtype) == _to_type(x / s, dtype), (dtype, dim, x)
