"""The fp32 direct-to-LDS GEMM (gemm32dma.hpp) on the GPU with an
M-contiguous A, a K that is no multiple of 32, and operands at any 4-byte
alignment: every layout, tile edges and remainders, k splits, against fp64."""
from __future__ import annotations

import ctypes
import os

import numpy as np
import pytest

from helpers import check_bound, cu, gemm_bound, ref, rnd, up

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
I64, P, F = ctypes.c_int64, ctypes.c_void_p, ctypes.c_float
RAG = "gemm tile generic 64x64 lds-dma"

CASES = [
    # (transA, transB, M, N, K, batch, row padding, first element, plan)
    (0, 1, 1, 1, 1, 1, 0, 1, RAG + " k-groups"),
    (0, 1, 65, 63, 31, 1, 3, 1, RAG + " k-groups"),
    (0, 0, 63, 65, 33, 2, 1, 0, RAG + " k-groups"),
    (1, 0, 67, 130, 65, 3, 1, 1, RAG + " k-groups"),
    (1, 1, 129, 62, 127, 1, 0, 1, RAG + " k-groups"),
    (0, 1, 33, 1025, 4097, 1, 0, 0, RAG + " fp32 split"),
    (0, 0, 100, 333, 513, 1, 1, 3, RAG + " fp32 split"),
    (1, 0, 515, 77, 2001, 1, 0, 0, RAG + " fp32 split"),
    (1, 1, 130, 131, 300, 1, 1, 1, RAG + " fp32 split"),
    (0, 1, 777, 1283, 1001, 1, 0, 0, RAG + " k-groups"),
    (0, 0, 515, 1001, 8197, 1, 0, 0, RAG + " fp32 split"),
    (1, 0, 1000, 1028, 333, 1, 4, 0, "gemm tile 64x64 lds-dma k-groups"),
    (1, 0, 64, 68, 130, 1, 0, 4, "gemm tile 64x64 lds-dma"),
    (1, 1, 1000, 1028, 164, 1, 4, 4, "gemm tile 64x64 lds-dma k-groups"),
    (1, 0, 512, 500, 4100, 1, 0, 0, "gemm tile 64x64 lds-dma fp32 split"),
    (0, 1, 777, 1284, 1000, 1, 0, 0, "gemm tile 64x64 lds-dma k-groups"),
    (0, 0, 1000, 1028, 132, 1, 4, 4, "gemm tile 64x64 lds-dma k-groups"),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "%s%s-%dx%dx%d" % ("NT"[c[0]], "NT"[c[1]], *c[2:5]))
def test_layouts_edges_and_alignments(case):
    """bias, SiLU and a residual; NaN around every operand, so nothing
    outside it may reach the result, and nothing outside C is written."""
    ta, tb, m, n, k, batch, pad, off, expect = case
    rng = np.random.default_rng(m * 7 + n * 3 + k + ta + 2 * tb)

    def placed(x):
        rows, cols = x.shape[-2:]
        full = np.full(off + batch * rows * (cols + pad), np.nan, np.float32)
        full[off:].reshape(batch, rows, cols + pad)[..., :cols] = x
        return up(full, "float32")

    a = rnd(rng, (batch, k, m) if ta else (batch, m, k), 1.0, "float32")
    b = rnd(rng, (batch, n, k) if tb else (batch, k, n), 1.0 / np.sqrt(k), "float32")
    bias, res = rnd(rng, (n,), 0.5, "float32"), rnd(rng, (batch, m, n), 1.0, "float32")
    ga, gb, gr, gbias = placed(a), placed(b), placed(res), up(bias, "float32")
    gc = up(np.full(off + batch * m * (n + pad), np.nan, np.float32), "float32")
    lda, ldb, ldc = a.shape[2] + pad, b.shape[2] + pad, n + pad
    sa, sb, sc = a.shape[1] * lda, b.shape[1] * ldb, m * ldc
    at = lambda g: g.data_ptr + 4 * off  # noqa: E731
    plan = cu().gemm_plan(tb, m, n, k, batch, at(ga), lda, sa, at(gb), ldb, sb, ldc, sc, np.float32, epi=2,
                          ptr_bias=gbias.data_ptr, transA=ta)
    assert plan.startswith(expect), plan
    lib = ctypes.CDLL(os.path.join(ROOT, "scaffolding_amd", "libsfgemm.so"))
    lib.sf_last_error.restype = ctypes.c_char_p
    for _ in range(2):  # the split counters are zero again after a launch
        rc = lib.sf_gemm_add(ta, tb, I64(m), I64(n), I64(k), I64(batch), P(at(ga)), I64(lda), I64(sa), P(at(gb)),
                             I64(ldb), I64(sb), P(at(gc)), I64(ldc), I64(sc), 0, 0, F(1.0), P(gbias.data_ptr), 2,
                             P(at(gr)), I64(ldc), I64(sc), None)
        assert rc == 0, lib.sf_last_error()
    got = cu().gputensor_to_numpy(gc)
    y = got[off:].reshape(batch, m, ldc)
    assert np.isnan(y[..., n:]).all() and np.isnan(got[:off]).all(), "written outside C"
    am = (np.swapaxes(a, 1, 2) if ta else a).astype(np.float64)
    bm = (np.swapaxes(b, 1, 2) if tb else b).astype(np.float64)
    pre = np.matmul(am, bm) + bias
    y64 = ref.act_f64(pre, "silu") + res
    bound = gemm_bound(ref.act_f64(pre, "silu"), np.matmul(np.abs(am), np.abs(bm)) + np.abs(bias), k, "float32", "silu")
    check_bound(y[..., :n], y64, bound + 2.0 ** -24 * np.abs(y64), "%s" % (case,))
