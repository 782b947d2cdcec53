"""The fused attention's check accepts the kernel's roundings, restated in
NumPy, and refuses planted mistakes: a lost key block, a row sum off by a
tenth, a key range of a split item with a wrong weight, a key past the end."""
from __future__ import annotations

import numpy as np
import pytest

from attention_check import HALF_ULP, check, exact
from helpers import quantize, rnd


def kernel(q, k, v, dtype, wrong=None):
    """One head as the kernel rounds it: Q scaled by scale log2 e and P, the
    output, in `dtype`; exponents and sums in fp32."""
    x = quantize(q * np.float32(q.shape[-1] ** -0.5 * 1.4426950408889634), dtype) @ k.T
    if wrong == "keys past the end":
        pad = -len(k) % 64
        x, v = np.pad(x, ((0, 0), (0, pad))), np.pad(v, ((0, pad), (0, 0)))
    p = quantize(np.exp2(x - x[:, :64].max(1, keepdims=True)), dtype)
    if wrong == "block":
        p[:, 64:128] = 0
    if wrong == "range":
        p[:, len(k) // 3: 2 * len(k) // 3] *= 1.25
    n = p.sum(1, keepdims=True)
    return quantize(p @ v / (n * 1.1 if wrong == "sum" else n), dtype)


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("d,sq,sk", [(64, 130, 700), (72, 300, 1000), (128, 300, 1000), (128, 127, 65), (96, 20, 203)])
def test_check_accepts_the_roundings_and_refuses_mistakes(dtype, d, sq, sk):
    rng = np.random.default_rng(d + sq + sk)
    q, k, v = (rnd(rng, (s, d), 1.0, dtype) for s in (sq, sk, sk))
    ref = exact(q, k, v, d ** -0.5, None, dtype)
    check(kernel(q, k, v, dtype), ref, dtype)
    # a few spare keys beside many are within the rounding
    for wrong in ["block", "sum", "range"] + (["keys past the end"] if sk < 256 else []):
        with pytest.raises(AssertionError):
            check(kernel(q, k, v, dtype, wrong), ref, dtype)


def test_check_refuses_a_missing_or_a_spare_nan():
    q, k, v = (rnd(np.random.default_rng(1), (9, 8), 1.0, "float16") for _ in range(3))
    y64, bound = exact(q, k, v, 0.3, None, "float16")
    y = quantize(y64.astype(np.float32), "float16")
    check(y, (y64, bound), "float16")
    assert HALF_ULP["float16"] == np.finfo(np.float16).eps / 2
    y64[3, 2] = np.nan
    with pytest.raises(AssertionError):
        check(y, (y64, bound), "float16")
