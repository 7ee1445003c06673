"""Host-checkable rules of the matrix-instruction kernels, called in the built library.

``rows_offset`` (``csrc/gemv_mfma.hip``) is the kernel's own lane offset into a wave's 64 weight columns, compiled for the host too.  It
is compared with exact integers over the widths that the ops admit, a matrix of more than 2 GiB among them;
the 32-bit product of an unclamped column fails the same comparison.

``rows_routed_ok`` and ``rows_dense_ok`` say which calls these kernels take.  A call without any k is not one of
them: their loops read at least one step, and a plan of no chunks divides by their number.

``gemm_staged_ok`` (``csrc/gemm.hip``) admits what the prefill's LDS-staged kernels can address and hold.
"""

from __future__ import annotations

import ctypes
import os
import subprocess
import sys

import pytest

from conftest import PKG_DIR


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


class _Rows(ctypes.Structure):
    _fields_ = [("n_groups", ctypes.c_void_p), ("group_expert", ctypes.c_void_p), ("group_start", ctypes.c_void_p),
                ("group_rows", ctypes.c_void_p), ("identity", ctypes.c_int), ("ids", ctypes.c_void_p),
                ("nids", ctypes.c_int)]


class _Proj(ctypes.Structure):
    _fields_ = [("w", ctypes.c_void_p), ("s", ctypes.c_void_p)]


class _GemvArgs(ctypes.Structure):
    """``GemvArgs`` of ``csrc/uocr_kernels.h``."""

    _fields_ = [("out", ctypes.c_void_p), ("ldo", ctypes.c_int64), ("x", ctypes.c_void_p), ("ldx", ctypes.c_int64),
                ("x_div", ctypes.c_int), ("p", _Proj * 2), ("kind", ctypes.c_int), ("E", ctypes.c_int),
                ("N", ctypes.c_int), ("K", ctypes.c_int), ("gsize", ctypes.c_int), ("nchunks", ctypes.c_int),
                ("vec", ctypes.c_int), ("batch", ctypes.c_int), ("rows", _Rows)]


INT8_ROWS, BF16_ROWS, BF16_KBLOCKED = 0, 1, 2


def _takes(kind: int, K: int, rows: int = 4, N: int = 64, x: int = 0, gsize: int = 128) -> bool:
    a = _GemvArgs(x=x, ldx=K, x_div=1, kind=kind, E=1, N=N, K=K, gsize=gsize, nchunks=-(-K // 128), vec=1)
    if kind == BF16_KBLOCKED:
        a.rows.identity = rows
        check = _internal("_ZN4uocr13rows_dense_okERKNS_8GemvArgsE", ctypes.c_bool, ctypes.POINTER(_GemvArgs))
    else:
        a.rows.n_groups = 256
        check = _internal("_ZN4uocr14rows_routed_okERKNS_8GemvArgsE", ctypes.c_bool, ctypes.POINTER(_GemvArgs))
    return check(ctypes.byref(a))


@pytest.mark.parametrize("kind", [INT8_ROWS, BF16_ROWS, BF16_KBLOCKED])
def test_a_call_without_k_is_not_taken(kind) -> None:
    assert _takes(kind, 128) and _takes(kind, 1280)
    assert not _takes(kind, 0)


def test_dense_rows_beyond_a_grid_are_not_taken() -> None:
    """A workgroup of 256 threads to 32 rows: 2^29 rows would make a grid of 2^32 threads."""
    assert _takes(BF16_KBLOCKED, 64, rows=1 << 28)
    assert not _takes(BF16_KBLOCKED, 64, rows=1 << 29)


def test_dense_call_without_k_returns() -> None:
    """Rows, columns and no k: an error without a GPU (none is visible to the child), never a signal."""
    code = ("import ctypes\nfrom uocr_moe import _lib\n"
            "err = ctypes.create_string_buffer(256)\n"
            "rc = _lib.load().uocr_dense_bf16_qmv(None, 3, 64, None, 3, 0, None, 0, 64, 16, 1, None, err, 256)\n"
            "assert rc != 0 and err.value")
    env = {**os.environ, "PYTHONPATH": str(PKG_DIR), "HIP_VISIBLE_DEVICES": "-1", "ROCR_VISIBLE_DEVICES": "-1"}
    assert subprocess.run([sys.executable, "-c", code], env=env, timeout=300).returncode == 0


class _GemmProblem(ctypes.Structure):
    """``GemmProblem`` of ``csrc/uocr_kernels.h``."""

    _fields_ = [("a", ctypes.c_void_p), ("lda", ctypes.c_int64), ("a_by_token", ctypes.c_int), ("x_div", ctypes.c_int),
                ("p", _Proj * 2), ("kind", ctypes.c_int), ("N", ctypes.c_int), ("K", ctypes.c_int),
                ("groups", ctypes.c_int), ("rows", _Rows), ("max_groups", ctypes.c_int), ("M", ctypes.c_int),
                ("swiglu", ctypes.c_int), ("outb", ctypes.c_void_p), ("outf", ctypes.c_void_p), ("ldo", ctypes.c_int64),
                ("out_by_position", ctypes.c_int), ("kparts", ctypes.c_int), ("part_stride", ctypes.c_int64)]


@pytest.mark.parametrize(("kind", "k", "groups", "max_groups", "vec", "takes"), [
    (INT8_ROWS, 1280, 10, 64, True, True), (INT8_ROWS, 1280, 10, 64, False, False),
    (INT8_ROWS, 1024, 16, 1, True, True), (INT8_ROWS, 1088, 17, 1, True, False),
    (BF16_ROWS, 6848, 1, 64, True, True), (BF16_ROWS, 1280, 1, 65, True, False),
    # 256 weight rows of a tile within 32 bits
    (INT8_ROWS, (1 << 24) - 128, 8, 1, True, True), (INT8_ROWS, 1 << 24, 8, 1, True, False),
    (BF16_ROWS, (1 << 23) - 128, 1, 1, True, True), (BF16_ROWS, 1 << 23, 1, 1, True, False),
])
def test_staged_gemm_takes(kind, k, groups, max_groups, vec, takes) -> None:
    problem = _GemmProblem(kind=kind, N=128, K=k, groups=groups, max_groups=max_groups)
    check = _internal("_ZN4uocr14gemm_staged_okERKNS_11GemmProblemEb", ctypes.c_bool, ctypes.POINTER(_GemmProblem),
                      ctypes.c_bool)
    assert check(ctypes.byref(problem), vec) == takes


def test_prefill_beyond_its_row_offsets_is_refused() -> None:
    """h of 400 000 tokens (top 6, ffn 896) has more than 2^31 elements: refused before anything is allocated."""
    from uocr_moe import _lib

    layer = _lib.Layer(64, 1280, 896, 1792, 6, 128, 1, 0, *[16] * 10)
    with pytest.raises(_lib.UocrError, match="seq out of range"):
        _lib.call("uocr_moe_forward", 16, 16, 400_000, 1280, ctypes.byref(layer), None, None, None, 0, None)
