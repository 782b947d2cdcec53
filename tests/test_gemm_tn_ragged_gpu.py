"""16-bit products of two operands with k-rows (dW = dY^T X) at a K that is no
multiple of 8: the 256 x 256 direct-to-LDS kernel, whole and split, and the
register-staged tiles.  NaN rows follow both operands: nothing past K may
reach the result."""
from __future__ import annotations

import ctypes
import os

import numpy as np
import pytest

from helpers import check_bound, cu, gemm_walk_bound, rnd, sample_rows, up

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
I64, P, F = ctypes.c_int64, ctypes.c_void_p, ctypes.c_float
SFD = {"float16": 1, "bfloat16": 2}
CASES = [
    # (dtype, M, N, K, plan)
    ("bfloat16", 1920, 1920, 2047, "gemm tn 256x256 lds-dma 16-bit split-tail"),
    ("float16", 1920, 1920, 4001, "gemm tn 256x256 lds-dma 16-bit split-tail"),
    ("bfloat16", 7680, 1920, 17771, "gemm tn 256x256 lds-dma"),
    ("float16", 4104, 4088, 131, "gemm tn 256x256 lds-dma"),
    ("bfloat16", 4096, 4096, 101, "gemm tile 256x256"),
    ("float16", 4096, 2048, 77, "gemm tile 256x128"),
    ("bfloat16", 65544, 40, 77, "gemm tile 256x64"),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "%s-%dx%dx%d" % c[:4])
def test_tn_with_a_ragged_k(case):
    dtype, m, n, k, expect = case
    g = cu()
    lib = ctypes.CDLL(os.path.join(ROOT, "scaffolding_amd", "libsfgemm.so"))
    rng = np.random.default_rng(m + n + k)
    a, b = rnd(rng, (k, m), 1.0, dtype), rnd(rng, (k, n), 1.0 / np.sqrt(k), dtype)
    past = np.full((130, max(m, n)), np.nan, np.float32)
    ga, gb = up(np.r_[a, past[:, :m]], dtype), up(np.r_[b, past[:, :n]], dtype)
    gc = up(np.zeros((m, n), np.float32), dtype)
    plan = g.gemm_plan(0, m, n, k, 1, ga.data_ptr, m, 0, gb.data_ptr, n, 0, n, 0, ga.dtype, transA=1)
    assert plan.startswith(expect), plan
    for _ in range(2):
        assert lib.sf_gemm(1, 0, I64(m), I64(n), I64(k), I64(1), P(ga.data_ptr), I64(m), I64(0), P(gb.data_ptr),
                           I64(n), I64(0), P(gc.data_ptr), I64(n), I64(0), SFD[dtype], SFD[dtype], F(1.0), None, 0,
                           None) == 0
    y = g.gputensor_to_numpy(gc)
    assert np.isfinite(y).all()
    rows = np.unique(np.r_[sample_rows(m, 8, k)[::4], m - 1])
    am, bm = a[:, rows].T.astype(np.float64), b.astype(np.float64)
    y64 = am @ bm
    check_bound(y[rows], y64, gemm_walk_bound(am, bm, y64, dtype), "%s" % (case,))
