"""The UNORM8 decode of vct_texel.hpp (one multiply and one FMA) equals the
IEEE division by 255 for every byte: its two constants are read from the
source and the FMA evaluated exactly in integers scaled by powers of two."""
import re
from fractions import Fraction
from pathlib import Path

import numpy as np

SRC = Path(__file__).resolve().parent.parent / "vk_voxel_cone_tracing_amd" / "csrc" / "vct_texel.hpp"


def test_u8_decode_is_the_division():
    hi, lo = re.search(r"__builtin_fmaf\(f, (\S+)f, f \* (\S+)f\)", SRC.read_text()).groups()
    hi, lo = np.float32(float.fromhex(hi)), np.float32(float.fromhex(lo))
    assert hi == np.float32(1) / np.float32(255)
    for b in range(256):
        f = np.float32(b)
        exact = Fraction(float(f)) * Fraction(float(hi)) + Fraction(float(f * lo))
        # rounded to float32 by way of float64: exact's double rounding cannot
        # cross a float32 tie, which has 25 significant bits
        got = np.float32(float(exact))
        assert Fraction(float(exact)) == exact or abs(Fraction(float(exact)) - exact) < abs(exact) / 2 ** 50
        assert got == f / np.float32(255), b
