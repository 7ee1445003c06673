"""The decode GEMVs on the fp32 matrix instruction, bit for bit against the oracle's chunk chains.

Sizes at the edges of its tiles: row groups of 1 to 35 (4-row tiles, passes of 16 rows), column counts that
are no multiple of a wave's 64 or 16, K that ends half a chunk short, one chunk, one wave, and dense shapes
that land on each way a launch is cut (16 or 64 columns a wave, chunks split over waves or not, 1 to 8 row
tiles a wave).
"""

from __future__ import annotations

import numpy as np
import pytest

from _gpu import bits_equal, moe_for, n, t

pytestmark = pytest.mark.gpu

# rows of the groups: every tile count, its edges, and more than one pass
GROUP_ROWS = [1, 2, 3, 4, 5, 7, 8, 9, 12, 13, 16, 17, 35]


def _ids(rng) -> np.ndarray:
    ids = np.concatenate([np.full(c, e, np.int32) for e, c in enumerate(GROUP_ROWS)])
    rng.shuffle(ids)
    return ids


@pytest.mark.parametrize(("n_", "k"), [(64, 128), (96, 256), (7, 384), (320, 1280)])
def test_int8_groups(oracle, n_, k) -> None:
    from uocr_moe import ops

    rng = np.random.default_rng(n_ + k)
    ids = _ids(rng)
    e = len(GROUP_ROWS)
    x = rng.standard_normal((len(ids), k)).astype(np.float32)
    w = rng.integers(-127, 128, (e, n_, k)).astype(np.int8)
    s = rng.uniform(1e-4, 1e-2, (e, n_, k // 128)).astype(np.float32)
    assert bits_equal(n(ops.moe_int8_qmv(t(x), t(ids), t(w), t(s))), oracle.moe_int8_qmv(x, ids, w, s))


@pytest.mark.parametrize(("n_", "k"), [(64, 64), (96, 192), (7, 384), (320, 1280)])
def test_bf16_groups(oracle, n_, k) -> None:
    from uocr_moe import ops

    rng = np.random.default_rng(n_ + k)
    ids = _ids(rng)
    x = rng.standard_normal((len(ids), k)).astype(np.float32)
    w = oracle.bf16_bits(rng.standard_normal((len(GROUP_ROWS), n_, k)).astype(np.float32))
    assert bits_equal(n(ops.moe_bf16_qmv(t(x), t(ids), t(w))), oracle.moe_bf16_qmv_chunked(x, ids, w))


@pytest.mark.parametrize(("n_", "k"), [(40, 64), (16, 192), (1300, 704), (130, 1280), (20000, 128), (40000, 192)])
@pytest.mark.parametrize("m", [1, 2, 4, 5, 11, 16, 21, 33])
def test_dense(oracle, m, n_, k) -> None:
    from uocr_moe import ops

    rng = np.random.default_rng(m * 7 + n_ + k)
    x = rng.standard_normal((m, k)).astype(np.float32)
    w = oracle.bf16_bits(rng.standard_normal((k // 16, n_, 16)).astype(np.float32))
    assert bits_equal(n(ops.dense_bf16_qmv(t(x), t(w))), oracle.dense_bf16_qmv_chunked(x, w))


@pytest.mark.parametrize("int8", [True, False], ids=["int8", "bf16"])
@pytest.mark.parametrize("rows", [9, 20, 64])
@pytest.mark.parametrize("skew", [False, True], ids=["plain", "skewed"])
def test_decode_rows(oracle, rows, int8, skew) -> None:
    """Past 8 rows the layer runs on these kernels; skewed: every row takes the same experts (up to 64 rows
    a group).  The widths are no multiples of the four column blocks of a workgroup."""
    layer = oracle.make_layer(31, E=10, H=384, F=128, topk=6, int8=int8, std=0.05, router_std=0.1)
    rng = np.random.default_rng(rows)
    x = rng.standard_normal((rows, 384)).astype(np.float32)
    if skew:
        x[:] = x[0] + np.float32(1e-3) * x
    moe = moe_for(layer)
    out, ids, _ = moe.decode_rows(t(x), routing=True)
    want, ids_o, _ = oracle.moe_decode_exact(x, layer)
    assert np.array_equal(n(ids), ids_o) and bits_equal(n(out), want)


def test_special_values(oracle) -> None:
    """Denormal activations keep their bits through the matrix instruction, and an infinite or NaN row stays
    its own: the rows beside it in its 4-row tile do not see it."""
    from uocr_moe import ops

    rng = np.random.default_rng(3)
    x = rng.standard_normal((6, 256)).astype(np.float32)
    x[1] *= np.float32(1e-41)
    x[2, 5], x[3, 200] = np.inf, np.nan
    w = oracle.bf16_bits(rng.standard_normal((16, 80, 16)).astype(np.float32))
    got, want = n(ops.dense_bf16_qmv(t(x), t(w))), oracle.dense_bf16_qmv_chunked(x, w)
    assert np.isnan(got[3]).all() and np.isinf(got[2]).all()
    assert bits_equal(got[[0, 1, 2, 4, 5]], want[[0, 1, 2, 4, 5]])


@pytest.mark.parametrize("topk", [2, 12])
@pytest.mark.parametrize("b", [15, 16, 33, 64])
def test_layer_groups_from_the_ids(oracle, b, topk) -> None:
    """From 16 rows on the routed GEMVs find their rows among the ids (more than 512 of them at 64 x 12)."""
    layer = oracle.make_layer(b + topk, E=64, H=128, F=64 if b % 2 else 128, topk=topk, int8=False, std=0.05,
                              router_std=0.3)
    x = np.random.default_rng(b).standard_normal((b, 128)).astype(np.float32)
    want, _, _ = oracle.moe_decode_exact(x, layer)
    assert bits_equal(n(moe_for(layer).decode_rows(t(x))), want)


@pytest.mark.parametrize("rows", [1, 3, 20])
def test_no_k(rows) -> None:
    """Sums over no k are zero, at every size of call."""
    import torch

    from uocr_moe import ops

    x = torch.empty((rows, 0), device="cuda:0")
    for n_ in (40, 20000):
        w = torch.empty((0, n_, 16), dtype=torch.bfloat16, device="cuda:0")
        out = torch.full((rows, n_), float("nan"), device="cuda:0")
        assert not n(ops.dense_bf16_qmv(x, w, out=out)).any()
    ids = torch.arange(rows, dtype=torch.int32, device="cuda:0") % 3
    out = torch.full((rows, 70), float("nan"), device="cuda:0")
    assert not n(ops.moe_bf16_qmv(x, ids, torch.empty((3, 70, 0), dtype=torch.bfloat16, device="cuda:0"), out=out)).any()


@pytest.mark.parametrize(("kind", "e", "n_", "rows", "kernel"), [
    ("int8", 8, 1088, 7, "gemv_op"), ("int8", 8, 1088, 8, "rows_op"), ("int8", 8, 1088, 100, "rows_op"),
    ("int8", 16, 256, 31, "gemv_op"), ("int8", 16, 256, 32, "rows_op"), ("int8", 3, 320, 200, "gemv_op"),
    ("bf16", 8, 384, 4, "gemv_op"), ("bf16", 8, 384, 5, "rows_op"),
    ("bf16", 1, 384, 8, "gemv_op"), ("bf16", 1, 384, 9, "rows_op"),
])
def test_routed_ops_at_the_edges_of_the_rule(oracle, kind, e, n_, rows, kernel) -> None:
    """Few column waves stay on the VALU kernel, a stack of few experts and many rows does not; same bits."""
    from uocr_moe import _lib, ops

    rng = np.random.default_rng(rows)
    ids = rng.integers(0, e, rows).astype(np.int32)
    x = rng.standard_normal((rows, 256)).astype(np.float32)
    _lib.timing_begin(8)
    if kind == "int8":
        w = rng.integers(-127, 128, (e, n_, 256)).astype(np.int8)
        s = rng.uniform(1e-4, 1e-2, (e, n_, 2)).astype(np.float32)
        got, want = n(ops.moe_int8_qmv(t(x), t(ids), t(w), t(s))), oracle.moe_int8_qmv(x, ids, w, s)
    else:
        w = oracle.bf16_bits(rng.standard_normal((e, n_, 256)).astype(np.float32))
        got, want = n(ops.moe_bf16_qmv(t(x), t(ids), t(w))), oracle.moe_bf16_qmv_chunked(x, ids, w)
    assert kernel in [name for name, _ in _lib.timing_end(8)]
    assert bits_equal(got, want)


@pytest.mark.parametrize("value", [1e-41, np.inf, np.nan], ids=["denormal", "inf", "nan"])
def test_special_weights_and_scales(oracle, value) -> None:
    """A denormal, infinite or NaN weight (bf16) or scale (int8) stays in its own column, with the chain's bits."""
    from uocr_moe import ops

    rng = np.random.default_rng(11)
    x = rng.standard_normal((12, 256)).astype(np.float32)
    col = 37

    def same(got, want) -> None:
        other = np.arange(got.shape[1]) != col
        assert bits_equal(got[:, other], want[:, other])
        nan = np.isnan(want[:, col])
        assert np.array_equal(np.isnan(got[:, col]), nan)
        assert bits_equal(got[~nan][:, [col]], want[~nan][:, [col]])

    dense = rng.standard_normal((16, 80, 16)).astype(np.float32)
    dense[3, col, 5] = value
    dense = oracle.bf16_bits(dense)
    same(n(ops.dense_bf16_qmv(t(x), t(dense))), oracle.dense_bf16_qmv_chunked(x, dense))
    ids = np.zeros(12, np.int32)
    rows = rng.standard_normal((1, 80, 256)).astype(np.float32)
    rows[0, col, 200] = value
    rows = oracle.bf16_bits(rows)
    same(n(ops.moe_bf16_qmv(t(x), t(ids), t(rows))), oracle.moe_bf16_qmv_chunked(x, ids, rows))
    # int8: wide enough for the matrix kernel
    ids = np.arange(12, dtype=np.int32)
    w = rng.integers(-127, 128, (12, 704, 256)).astype(np.int8)
    s = rng.uniform(1e-4, 1e-2, (12, 704, 2)).astype(np.float32)
    s[:, col, 1] = value
    same(n(ops.moe_int8_qmv(t(x), t(ids), t(w), t(s))), oracle.moe_int8_qmv(x, ids, w, s))
