"""The matrix-instruction GEMVs' host-checkable rules (``csrc/gemv_mfma.hip``), called in the built library.

``rows_offset`` is the kernel's own lane offset into a wave's 64 weight columns, compiled for the host too.  It
is compared with exact integers over the widths that the ops admit, a matrix of more than 2 GiB among them;
the 32-bit product of an unclamped column fails the same comparison.
"""

from __future__ import annotations

import ctypes

import pytest


def _internal(symbol: str, restype, *argtypes):
    from uocr_moe import _lib

    f = getattr(_lib.load(), symbol)
    f.restype, f.argtypes = restype, argtypes
    return f


def _unclamped(col: int, cols: int, rowb: int, piece: int) -> int:
    """The last column's offset as a 32-bit product, then the smaller of the two offsets."""
    last = ctypes.c_int32((cols - 1) * rowb + 16 * piece).value
    return min(col * rowb + 16 * piece, last)


SHAPES = [(1, 128), (7, 256), (63, 131072), (64, 131072), (65, 131072), (896, 1280), (129280, 2560),
          (131072, 16384), (262144, 16384), (32769, 65536), (1 << 30, 131072)]


@pytest.mark.parametrize(("cols", "rowb"), SHAPES)
def test_weight_offsets_stay_in_the_matrix(cols, rowb) -> None:
    offset = _internal("_ZN4uocr11rows_offsetEiiii", ctypes.c_int, *[ctypes.c_int] * 4)
    for col in range(64):
        for piece in range(8):
            assert offset(col, cols, rowb, piece) == min(col, cols - 1) * rowb + 16 * piece


def test_the_unclamped_product_fails() -> None:
    """From 2 GiB a matrix its last column's offset is negative and would be taken."""
    wrong = [s for s in SHAPES if any(_unclamped(c, *s, 0) != min(c, s[0] - 1) * s[1] for c in range(64))]
    assert (262144, 16384) in wrong and (32769, 65536) in wrong and (129280, 2560) not in wrong
