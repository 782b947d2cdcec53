"""What the fused attention may differ by from softmax(scale q k^T + mask) v
in fp64, shared by its GPU tests and the CPU test that shows what the check
refuses."""
from __future__ import annotations

import numpy as np

HALF_ULP = {"float16": 2.0 ** -11, "bfloat16": 2.0 ** -8}


def softmax64(s):
    m = np.max(s, -1, keepdims=True)
    with np.errstate(invalid="ignore"):
        e = np.exp(s - m)
    return e / e.sum(-1, keepdims=True)


def exact(q, k, v, scale, mask=None, dtype="bfloat16"):
    """(y, bound): fp64, with score + mask rounded to fp32 once as the
    device's sum is (which decides rows of large finite masks), and the
    largest difference that `dtype`'s roundings can make, element by element.

    With u the type's half ulp, Q scaled and rounded once moves exponent j by
    at most u a_j, a_j = scale sum_d |q_d k_jd|, and P is rounded once, so
    each weight p_j changes by a factor within 1 +- u (1 + a_j); the row sum
    is over the same rounded P.  Hence |y' - y| <= u sum_j p_j (1 + a_j)
    (|v_j| + |y|), and u |y| for the output's own rounding; 5 % more for the
    terms in u^2 and the fp32 arithmetic.  fp16 weights below 2^-14 of the
    largest are subnormal: 2^-25 of it each."""
    u = HALF_ULP[dtype]
    q, k, v = (x.astype(np.float64) for x in (q, k, v))
    s = scale * np.matmul(q, np.swapaxes(k, -2, -1))
    if mask is not None:
        s = (s.astype(np.float32) + mask.astype(np.float32)).astype(np.float64)
    p = softmax64(s)
    y = np.matmul(p, v)
    a = scale * np.matmul(np.abs(q), np.swapaxes(np.abs(k), -2, -1))
    w = p * (1.0 + np.where(p > 0, a, 0.0))
    bound = 1.05 * u * (np.matmul(w, np.abs(v)) + np.abs(y) * (w.sum(-1, keepdims=True) + 1.0))
    if dtype == "float16":
        bound = bound + k.shape[-2] * 2.0 ** -25 * np.max(np.abs(v))
    return y, bound


def check(y, ref, dtype):
    """NaN where the reference is NaN, every other element within its bound,
    and all of them together within 2.5 u in the 2-norm: the roundings are
    independent, u / sqrt(3) each relative to the terms of y, which adds up
    to about u for unit-variance heads, while a lost key, a wrong row sum or
    a wrong weight of a key range moves whole rows."""
    y64, bound = ref
    assert np.array_equal(np.isnan(y), np.isnan(y64))
    ok = ~np.isnan(y64)
    err = np.abs(y.astype(np.float64) - y64)[ok]
    over = err - bound[ok]
    assert over.size == 0 or over.max() <= 0, (err[over.argmax()], bound[ok][over.argmax()])
    norm = np.sqrt(np.sum(y64[ok] ** 2))
    assert np.sqrt(np.sum(err ** 2)) <= 2.5 * HALF_ULP[dtype] * norm, np.sqrt(np.sum(err ** 2)) / norm
