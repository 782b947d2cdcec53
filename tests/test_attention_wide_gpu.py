"""Fused attention with head sizes up to 128 and additive masks
(attention_wide.hpp) on the GPU against fp64: ragged query and key counts,
every mask broadcast and type, rows that meet no key, a late key, large
finite masks, split key ranges."""
from __future__ import annotations

import ctypes
import os

import numpy as np
import pytest

from attention_check import HALF_ULP, check, exact, softmax64
from helpers import cu, down, rnd, up

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LOW = float(np.finfo(np.float32).min)


def masks(kind, b, h, sq, sk, rng, dtype):
    if kind == "causal":
        return np.where(np.arange(sk)[None, :] > np.arange(sq)[:, None] + max(0, sk - sq), -np.inf, 0.0)
    if kind == "pad":  # [B, 1, 1, Sk]: the second half, and all but one key of the last sample
        m = np.zeros((b, 1, 1, sk))
        m[0, ..., sk // 2:] = -np.inf
        m[-1, ..., :] = -np.inf
        m[-1, ..., sk - 1] = 0.0
        return m
    if kind == "left-low":  # only the last keys count; the earlier ones hold the lowest value or -1e9
        m = np.zeros((b, 1, 1, sk))
        m[0, ..., : sk - 3] = LOW
        m[-1, ..., : sk - 3] = -1e9
        return m
    if kind == "rows":  # whole rows at -inf (NaN), the lowest value, -1e9, and a mixture
        m = np.zeros((h, sq, sk))
        m[:, 0] = -np.inf
        m[:, sq // 2] = LOW
        m[:, sq // 3] = -1e9
        m[:, sq - 1] = -np.inf
        m[:, sq - 1, sk // 2:] = LOW
        return m
    return rnd(rng, (b, h, sq, sk), 3.0, dtype)  # "bias"


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("d", [72, 96, 104, 128])
@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 127, 65), (3, 129, 64), (1, 300, 1000)],
                         ids=lambda s: "x".join(map(str, s)))
def test_wide_heads(dtype, d, shape):
    bh, sq, sk = shape
    rng = np.random.default_rng(d + sq + sk)
    q, k, v = (rnd(rng, (bh, s, d), 1.0, dtype) for s in (sq, sk, sk))
    y = down(cu().dev_scaled_dot_product_attention(up(q, dtype), up(k, dtype), up(v, dtype)))
    check(y, exact(q, k, v, d ** -0.5, None, dtype), dtype)


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("d,scale", [(40, None), (64, None), (64, 1.0), (80, None), (128, None)])
@pytest.mark.parametrize("kind,mdtype", [("causal", "float32"), ("pad", "float32"), ("left-low", "float32"),
                                         ("rows", "float32"), ("bias", "float32"), ("bias", None)])
def test_masks(dtype, d, scale, kind, mdtype):
    """Sk = 203 (a partial last block, mask rows at no 16-byte boundary) and
    two batch entries of three heads; scale 1 takes the FMA path."""
    b, h, sq, sk = 2, 3, 133, 203
    rng = np.random.default_rng(d + len(kind))
    q, k, v = (rnd(rng, (b, h, s, d), 0.5 if scale else 1.0, dtype) for s in (sq, sk, sk))
    m = masks(kind, b, h, sq, sk, rng, dtype).astype(np.float32)
    gm = up(m, mdtype or dtype)
    y = down(cu().dev_scaled_dot_product_attention(up(q, dtype), up(k, dtype), up(v, dtype), scale, gm))
    check(y, exact(q, k, v, scale or d ** -0.5, m, dtype), dtype)


@pytest.mark.parametrize("kind", ["none", "causal", "left-low", "rows"])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
def test_split_key_ranges(kind, d, dtype):
    """Every item in three key ranges (test hook): parts in which a row meets
    no key weigh nothing, rows without any key are finished by the merge."""
    b, h, sq, sk = 2, 2, 130, 700
    rng = np.random.default_rng(d)
    q, k, v = (rnd(rng, (b, h, s, d), 1.0, dtype) for s in (sq, sk, sk))
    m = None if kind == "none" else masks(kind, b, h, sq, sk, rng, dtype).astype(np.float32)
    g = cu()
    g._set_test_hooks(attn_parts=3)
    try:
        y = down(g.dev_scaled_dot_product_attention(up(q, dtype), up(k, dtype), up(v, dtype), None,
                                                    None if m is None else up(m, "float32")))
    finally:
        g._set_test_hooks()
    check(y, exact(q, k, v, d ** -0.5, m, dtype), dtype)


def test_nan_and_inf_scores_reach_their_rows():
    """A NaN in one query row and an infinite key: the rows that a plain
    softmax makes NaN are NaN, and no other."""
    rng = np.random.default_rng(3)
    q, k, v = (rnd(rng, (1, s, 128), 1.0, "bfloat16") for s in (100, 90, 90))
    q[0, 7, 3] = np.nan
    k[0, 50, 5] = np.inf
    m = np.zeros((100, 90), np.float32)
    m[20:, 50] = -np.inf
    y = down(cu().dev_scaled_dot_product_attention(up(q, "bfloat16"), up(k, "bfloat16"), up(v, "bfloat16"), None,
                                                   up(m, "float32")))
    with np.errstate(invalid="ignore"):
        s = 128 ** -0.5 * np.matmul(q.astype(np.float64), np.swapaxes(k, -2, -1).astype(np.float64)) + m
        y64 = np.matmul(softmax64(s), v.astype(np.float64))
    assert np.array_equal(np.isnan(y), np.isnan(y64))


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("masked", [False, True])
def test_split_parts_of_nan_scores(d, masked):
    """A key range whose every score is NaN (one part of three, test hook),
    a NaN query row and an infinite key: NaN wherever the plain softmax is,
    and nowhere else."""
    sq, sk = 130, 700
    rng = np.random.default_rng(d + masked)
    q, k, v = (rnd(rng, (3, s, d), 1.0, "bfloat16") for s in (sq, sk, sk))
    k[0, 192:448] = np.nan  # 11 blocks of 64 keys: part 1 is blocks 3 to 6
    q[1, 7, 3] = np.nan
    k[2, 50, 5] = np.inf
    m = None
    if masked:
        m = np.zeros((3, sq, sk), np.float32)
        m[0, :, :192] = -np.inf  # and the first part has no key
        m[2, 20:, 50] = -np.inf
    g = cu()
    g._set_test_hooks(attn_parts=3)
    try:
        y = down(g.dev_scaled_dot_product_attention(up(q, "bfloat16"), up(k, "bfloat16"), up(v, "bfloat16"), None,
                                                    None if m is None else up(m, "float32")))
    finally:
        g._set_test_hooks()
    with np.errstate(invalid="ignore"):
        s = d ** -0.5 * np.matmul(q.astype(np.float64), np.swapaxes(k, -2, -1).astype(np.float64))
        y64 = np.matmul(softmax64(s if m is None else s + m), v.astype(np.float64))
    assert np.array_equal(np.isnan(y), np.isnan(y64))


def test_packed_heads_of_80_and_columns_past_d():
    """Heads of 80 read in place from a packed projection (the 96-wide tile
    must not take its neighbour's columns), written side by side."""
    b, n, h, d = 2, 150, 3, 80
    rng = np.random.default_rng(8)
    qkv = rnd(rng, (b, n, 3 * h * d), 1.0, "float16")
    y = down(cu().dev_attention_packed(up(qkv, "float16"), h))
    q, k, v = (x.reshape(b, n, h, d).transpose(0, 2, 1, 3) for x in np.split(qkv, 3, -1))
    ref = exact(q, k, v, d ** -0.5, None, "float16")
    check(y, [x.transpose(0, 2, 1, 3).reshape(b, n, h * d) for x in ref], "float16")


@pytest.mark.parametrize("shape", [(0, 4, 16, 16), (2, 0, 16, 16), (2, 3, 0, 16), (2, 3, 16, 0)],
                         ids=["batch", "heads", "queries", "keys"])
@pytest.mark.parametrize("d,masked", [(64, True), (128, False), (128, True)])
def test_empty_operands(shape, d, masked):
    """Empty batches, and rows without a key, give what the three launches
    give: an empty result, zeros."""
    b, h, sq, sk = shape
    g = cu()
    q, k, v = (g.zeros((b, h, s, d), g.BFLOAT16) for s in (sq, sk, sk))
    for m in [(sq, sk), (b, 1, sq, sk)] if masked else [None]:
        gm = None if m is None else g.zeros(m, np.float32)
        y = g.dev_scaled_dot_product_attention(q, k, v, None, gm)
        assert y.shape == (b, h, sq, d) and not down(y).any()


def test_abi_rules():
    """sf_attention keeps refusing head sizes above 64; the masked entry
    refuses what neither takes."""
    lib = ctypes.CDLL(os.path.join(ROOT, "scaffolding_amd", "libsfgemm.so"))
    I64, P, F = ctypes.c_int64, ctypes.c_void_p, ctypes.c_float
    x = up(np.zeros((64, 136), np.float32), "bfloat16")

    def masked(d, mdt, row, dt=2):
        p = P(x.data_ptr)
        s = [I64(136), I64(0), I64(0)]
        o = [I64(136), I64(64 * 136), I64(64 * 136)]
        return lib.sf_attention_masked(p, *s, p, *s, p, *s, p, *o, I64(1), I64(1), I64(8), I64(8), I64(d), F(0.1), dt,
                                       p, mdt, I64(0), I64(0), I64(row), None)

    assert masked(136, 2, 0) == -3 and masked(12, 2, 0) == -3 and masked(64, 2, 0, dt=0) == -3
    assert masked(64, 1, 0) == -3 and masked(64, 7, 0) == -2 and masked(64, 2, -1) == -2
    p = P(x.data_ptr)
    assert lib.sf_attention(p, I64(80), I64(0), p, I64(80), I64(0), p, I64(80), I64(0), p, I64(80), I64(0), I64(1),
                            I64(8), I64(8), I64(80), F(0.1), 2, None) == -3


def test_non_finite_values_at_keys_without_weight():
    """Rows whose mask holds only lowest values (or -inf and one of them):
    P V multiplies every key's V by its weight, so a NaN or infinite V at a
    key of weight 0 makes its column NaN as in any other row."""
    rng = np.random.default_rng(12)
    q, k, v = (rnd(rng, (2, s, 72), 1.0, "float16") for s in (20, 90, 90))
    v[0, 10, 3] = np.nan
    v[1, 70, 65] = -np.inf
    m = np.full((20, 90), LOW, np.float32)
    m[5:, 10] = -np.inf
    m[9:, 64:] = -np.inf
    m[12] = 0.0
    y = down(cu().dev_scaled_dot_product_attention(up(q, "float16"), up(k, "float16"), up(v, "float16"), None,
                                                   up(m, "float32")))
    s = (72 ** -0.5 * np.matmul(q, np.swapaxes(k, -2, -1))).astype(np.float32) + m
    with np.errstate(invalid="ignore"):
        y64 = np.matmul(softmax64(s.astype(np.float64)), v.astype(np.float64))
    ok = np.isfinite(y64)
    assert np.array_equal(np.isnan(y), np.isnan(y64)) and np.array_equal(y[np.isinf(y64)], y64[np.isinf(y64)])
    # the weights of keys that count are 1 and exact, but in row 12
    assert np.abs(y[ok] - y64[ok]).max() <= 6 * HALF_ULP["float16"] * np.abs(v[np.isfinite(v)]).max()


def _nonfinite_case(seed, d, dtype):
    rng = np.random.default_rng(seed)
    return tuple(rnd(rng, (2, s, d), 1.0, dtype) for s in (40, 203, 203))


def _check_rows(q, k, v, scale, m, dtype, parts):
    g = cu()
    g._set_test_hooks(attn_parts=parts)
    try:
        y = down(g.dev_scaled_dot_product_attention(up(q, dtype), up(k, dtype), up(v, dtype), scale, up(m, "float32")))
    finally:
        g._set_test_hooks()
    with np.errstate(invalid="ignore", over="ignore"):
        ref = exact(q, k, v, scale or q.shape[-1] ** -0.5, m, dtype)
    check(y, ref, dtype)


@pytest.mark.parametrize("parts", [0, 3])
@pytest.mark.parametrize("dtype,d,scale", [("bfloat16", 64, None), ("float16", 128, None), ("bfloat16", 96, 2.0)])
def test_scores_of_minus_infinity_under_a_mask(dtype, d, scale, parts):
    """An infinite key gives rows of one sign a score of -inf there.  Where
    no other key counts the row is NaN, not the average that rows without a
    key in reach of the mask get; beside lowest-value keys those count."""
    q, k, v = _nonfinite_case(d, d, dtype)
    q[:, :, 0] = np.abs(q[:, :, 0]) + 0.5  # so score(key) = -inf
    k[:, :70, 0] = -np.inf
    m = np.full((40, 203), -np.inf, np.float32)
    m[:10, :70] = 0.0    # only -inf scores: NaN
    m[10:20, :30] = 0.0  # beside lowest-value keys with finite scores: those
    m[10:20, 100:] = LOW
    m[20:30, :] = 0.0    # beside ordinary keys
    m[30:, 20:] = LOW    # lowest-value keys, some of -inf scores
    _check_rows(q, k, v, scale, m, dtype, parts)


@pytest.mark.parametrize("parts", [0, 3])
@pytest.mark.parametrize("dtype,d,scale", [("bfloat16", 64, None), ("float16", 128, None), ("bfloat16", 96, 2.0)])
def test_large_positive_masks(dtype, d, scale, parts):
    """Masks up to the largest fp32 value: the sum with the score is rounded
    to fp32, and rows of one such value are uniform over its keys (scores
    below 32, half an ulp of 1e9)."""
    q, k, v = _nonfinite_case(d + 1, d, dtype)
    if scale:
        q *= 0.25
    m = np.zeros((40, 203), np.float32)
    m[:5] = 1e9
    m[5:10, 100:] = (1e9 + 62528 * np.arange(5))[:, None]  # small masks before
    m[10:15, 150:] = -LOW
    m[15:20] = 3e38
    m[20:25, 7] = 2.5e38
    m[25:30, ::3] = 2.5e38
    m[25:30, 1] = np.nan
    m[30:35, 64:66] = 2.4e38
    m[35:, 100] = np.inf  # inf - inf
    _check_rows(q, k, v, scale, m, dtype, parts)
