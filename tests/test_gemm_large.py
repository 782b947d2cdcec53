"""16-bit GEMMs with an operand of more than 2 GiB: the plan on both sides of
that size, and on the GPU sampled outputs at its two ends (the last rows lie
past 2^31 bytes) against fp64."""
from __future__ import annotations

import ctypes
import os

import numpy as np
import pytest

from helpers import check_bound, cu, gemm_walk_bound, rnd, up

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
I64, P, F = ctypes.c_int64, ctypes.c_void_p, ctypes.c_float
RAGGED = "gemm tile generic 128x128"


def _plan(ta, tb, m, n, k):
    g = cu()
    return g.gemm_plan(tb, m, n, k, 1, 1 << 20, m if ta else k, 0, 1 << 20, k if tb else n, 0, n, 0, g.BFLOAT16,
                       transA=ta)


@pytest.mark.parametrize("ta,tb,m,n,k,large,below", [
    (0, 1, 4096, 262144, 4096, "gemm tile 256x256", "gemm nt 256x256"),
    (0, 1, 262144, 4096, 4096, "gemm tile 256x256", "gemm nt 256x256"),
    (0, 0, 262144, 4096, 4096, "gemm tile 256x256", "gemm nn 256x256"),
    (0, 1, 262144, 64, 4096, "gemm tile 256x64", "gemm tile 256x64"),
    (0, 1, 128, 262144, 4096, RAGGED, "gemm nt 256x256"),
    (1, 0, 4096, 512, 262144, RAGGED, "gemm tile 128x128"),
])
def test_plans_around_2_gib(ta, tb, m, n, k, large, below):
    """An operand of 2^31 bytes, and one eight elements smaller a side."""
    assert _plan(ta, tb, m, n, k).startswith(large)
    if k == 262144:
        k -= 128
    elif m == 262144:
        m -= 8
    else:
        n -= 8
    assert _plan(ta, tb, m, n, k).startswith(below)


CASES = [
    # (transA, transB, M, N, K, pad, plan): the large operand has pad unused
    # columns a row
    (0, 1, 300, 262400, 4096, 8, "gemm tile 256x256"),
    (0, 1, 262400, 264, 4096, 0, "gemm tile 256x256"),
    (0, 0, 262400, 264, 4096, 0, "gemm tile 256x256"),
    (0, 1, 262400, 40, 4096, 0, "gemm tile 256x64"),
    (0, 1, 72, 262400, 4096, 0, "gemm tile generic"),
    (0, 1, 130, 262400, 4097, 0, "gemm tile generic"),
    (1, 0, 4096, 264, 262400, 0, "gemm tile generic 128x128 16-bit split"),
    (0, 0, 136, 4096, 262401, 0, "gemm tile generic"),
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=lambda c: "%s%s-%dx%dx%d" % ("NT"[c[0]], "NT"[c[1]], *c[2:5]))
def test_sampled_outputs(case):
    ta, tb, m, n, k, pad, expect = case
    g = cu()
    lib = ctypes.CDLL(os.path.join(ROOT, "scaffolding_amd", "libsfgemm.so"))
    lib.sf_last_error.restype = ctypes.c_char_p
    rng = np.random.default_rng(m + n + k)
    period = 16777213  # elements; a prime, so no two rows are alike
    base = rnd(rng, (period,), 1.0, "bfloat16")
    gbase = up(base, "bfloat16")

    def operand(rows, cols):
        """rows x cols, element e = base[e mod period] where that takes over
        2 GiB, else random; its host rows, and columns of given k, by index."""
        if 2 * rows * cols >= 1 << 31:
            ld = cols + pad
            t = g.empty((rows, ld), g.BFLOAT16)
            for e in range(0, rows * ld, period):
                cnt = min(period, rows * ld - e)
                assert lib.sf_memcpy_d2d(P(t.data_ptr + 2 * e), P(gbase.data_ptr), ctypes.c_size_t(2 * cnt), None) == 0
            return t, ld, lambda r, c: base[(r[:, None].astype(np.int64) * ld + c[None, :]) % period]
        x = rnd(rng, (rows, cols), 1.0 / np.sqrt(k), "bfloat16")
        return up(x, "bfloat16"), cols, lambda r, c: x[np.ix_(r, c)]

    ga, lda, ah = operand(k, m) if ta else operand(m, k)
    gb, ldb, bh = operand(n, k) if tb else operand(k, n)
    gc = g.empty((m, n), g.BFLOAT16)
    plan = g.gemm_plan(tb, m, n, k, 1, ga.data_ptr, lda, 0, gb.data_ptr, ldb, 0, n, 0, g.BFLOAT16, transA=ta)
    assert plan.startswith(expect), plan
    print(case, plan, flush=True)
    rc = lib.sf_gemm(ta, tb, I64(m), I64(n), I64(k), I64(1), P(ga.data_ptr), I64(lda), I64(0), P(gb.data_ptr),
                     I64(ldb), I64(0), P(gc.data_ptr), I64(n), I64(0), 2, 2, F(1.0), None, 0, None)
    assert rc == 0, lib.sf_last_error()
    y = down_rows(g, lib, gc, m, n)

    def ends(x):
        return np.unique(np.clip(np.r_[0, 1, x // 2, x - 257, x - 2, x - 1], 0, x - 1))

    rows, cols, ks = ends(m), ends(n), np.arange(k)
    a = (ah(ks, rows).T if ta else ah(rows, ks)).astype(np.float64)
    b = (bh(cols, ks).T if tb else bh(ks, cols)).astype(np.float64)
    got = np.stack([y(int(r))[cols] for r in rows])
    y64 = a @ b
    check_bound(got, y64, gemm_walk_bound(a, b, y64, "bfloat16"), "%s" % (case,))


def down_rows(g, lib, gc, m, n):
    """Reads single rows of a device matrix (the whole may take gigabytes)."""
    def row(r):
        bits = np.empty(n, np.uint16)
        assert lib.sf_memcpy_d2h(bits.ctypes.data_as(P), P(gc.data_ptr + 2 * r * n), ctypes.c_size_t(2 * n), None) == 0
        return (bits.astype(np.uint32) << 16).view(np.float32)
    return row
