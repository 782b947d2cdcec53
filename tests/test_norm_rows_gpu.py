"""Row norms at the edges of their register-resident kernels: the last column
count of each width, one past it, odd counts (rows off any vector
alignment), vectors off 16-byte alignment, against fp64."""
from __future__ import annotations

import ctypes
import os

import numpy as np
import pytest

from helpers import cu, down, out_half_ulp_rel, rnd, up

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SFD = {"float32": 0, "float16": 1, "bfloat16": 2}
COLS = [1, 7, 8, 9, 511, 512, 513, 2047, 4095, 4096, 4097, 4104, 5120, 6145, 8191, 8200, 16383, 16384, 16385]


def _bound(y64, h64, cols, dtype):
    """fp32 arithmetic on normalised values h of order sqrt(cols) at most:
    sums of `cols` terms in a tree of depth < 64 (64 * 2^-24 relative), a
    few roundings of terms as large as |h| and |y|, one output rounding."""
    return (out_half_ulp_rel(dtype) + 1e-6) * np.abs(y64) + 2.0 ** -17 * (np.abs(h64) + 1.0) + 1e-7


@pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("cols", COLS)
@pytest.mark.parametrize("kind", ["rms", "layer", "ada"])
def test_row_widths(dtype, cols, kind):
    rows, groups = 6, 2
    rng = np.random.default_rng(cols + len(kind))
    x = rnd(rng, (rows, cols), 2.0, dtype)
    g, b = rnd(rng, (cols,), 1.0, dtype), rnd(rng, (cols,), 0.5, dtype)
    mod = rnd(rng, (groups, 2 * cols), 0.3, dtype)
    # every operand one element into its buffer, NaN around it
    shift = 1 if cols % 2 else 0

    def put(a):
        return up(np.r_[np.full(shift, np.nan, np.float32), a.ravel(), np.full(3, np.nan, np.float32)], dtype)

    es = 4 if dtype == "float32" else 2
    gx, gg, gb, gm = put(x), put(g), put(b), put(mod)
    gy = put(np.full((rows, cols), np.nan, np.float32))
    P, I64 = ctypes.c_void_p, ctypes.c_int64
    at = lambda t, o=0: P(t.data_ptr + es * (shift + o))  # noqa: E731
    lib = ctypes.CDLL(os.path.join(ROOT, "scaffolding_amd", "libsfgemm.so"))
    stats = up(np.zeros((2, rows), np.float32), "float32")
    eps = ctypes.c_float(1e-5)
    if kind == "rms":
        rc = lib.sf_rms_norm(at(gx), at(gy), I64(rows), I64(cols), at(gg), eps, SFD[dtype], None)
    else:
        m = (at(gm), at(gm, cols), I64(2 * cols), I64(rows // groups)) if kind == "ada" else (None, None, I64(0), I64(1))
        rc = lib.sf_layer_norm(at(gx), at(gy), I64(rows), I64(cols), at(gg), at(gb), eps, *m, P(stats.data_ptr),
                               P(stats.data_ptr + 4 * rows), SFD[dtype], None)
    assert rc == 0
    cu().device_synchronize()
    out = down(gy)
    assert np.isnan(out[:shift]).all() and np.isnan(out[shift + rows * cols:]).all()
    y = out[shift:shift + rows * cols].reshape(rows, cols)
    x64 = x.astype(np.float64)
    mu = 0.0 if kind == "rms" else x64.mean(1, keepdims=True)
    rstd = 1.0 / np.sqrt(((x64 - mu) ** 2).mean(1, keepdims=True) + float(np.float32(1e-5)))
    h = (x64 - mu) * rstd
    y64 = h * g
    if kind != "rms":
        y64 = y64 + b
        st = down(stats)
        assert np.allclose(st[0], np.ravel(mu), atol=1e-5) and np.allclose(st[1], np.ravel(rstd), rtol=1e-5)
    s = np.abs(g) + 1.0
    if kind == "ada":
        sc, sh = (np.repeat(t.astype(np.float64), rows // groups, 0) for t in (mod[:, :cols], mod[:, cols:]))
        y64 = y64 * (1.0 + sc) + sh
        s = s * (1.0 + np.abs(sc))
    err = np.abs(y - y64)
    assert np.all(err <= _bound(y64, np.abs(h) * s + np.abs(b), cols, dtype)), err.max()
