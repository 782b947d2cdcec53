"""The mid-size 16-bit GEMM (gemm16mid.hpp) on the GPU: 128 x 128, 64 x 64
and 32 x 64 tiles, k splits, and operands at any 2-byte alignment, in every
layout, at tile edges and remainders, against fp64."""
from __future__ import annotations

import ctypes
import os

import numpy as np
import pytest

from helpers import check_bound, cu, gemm_bound, ref, rnd, storage, up

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
I64, P, F = ctypes.c_int64, ctypes.c_void_p, ctypes.c_float
SFD = {"float16": 1, "bfloat16": 2}


def _lib():
    lib = ctypes.CDLL(os.path.join(ROOT, "scaffolding_amd", "libsfgemm.so"))
    lib.sf_last_error.restype = ctypes.c_char_p
    return lib


def _run(case, pad=0, offset=0, stream=None, reps=1):
    """sf_gemm_add through the C ABI with rows `pad` elements longer than
    needed and every operand starting `offset` elements into its buffer
    (poisoned with NaN around the operand); returns the checked output."""
    dtype, ta, tb, m, n, k, expect = case
    rng = np.random.default_rng(m * 7 + n * 3 + k + ta + 2 * tb)

    def padded(x):
        r, c = x.shape
        full = np.full(offset + r * (c + pad), np.nan, np.float32)
        for i in range(r):
            full[offset + i * (c + pad): offset + i * (c + pad) + c] = x[i]
        return full

    a = rnd(rng, (k, m) if ta else (m, k), 1.0, dtype)
    b = rnd(rng, (n, k) if tb else (k, n), 1.0 / np.sqrt(k), dtype)
    bias = rnd(rng, (n,), 0.5, dtype)
    res = rnd(rng, (m, n), 1.0, dtype)
    ga, gb, gr = (up(padded(x), dtype) for x in (a, b, res))
    gbias = up(bias, dtype)
    gc = up(np.full(offset + m * (n + pad), np.nan, np.float32), dtype)
    lda, ldb, ldc = a.shape[1] + pad, b.shape[1] + pad, n + pad
    at = lambda g: g.data_ptr + 2 * offset  # noqa: E731
    plan = cu().gemm_plan(tb, m, n, k, 1, at(ga), lda, 0, at(gb), ldb, 0, ldc, 0, storage(dtype), epi=2,
                          ptr_bias=gbias.data_ptr, transA=ta)
    assert plan.startswith(expect), plan
    lib = _lib()
    for _ in range(reps):
        rc = lib.sf_gemm_add(ta, tb, I64(m), I64(n), I64(k), I64(1), P(at(ga)), I64(lda), I64(0), P(at(gb)),
                             I64(ldb), I64(0), P(at(gc)), I64(ldc), I64(0), SFD[dtype], SFD[dtype], F(1.0),
                             P(gbias.data_ptr), 2, P(at(gr)), I64(ldc), I64(0), stream)
        assert rc == 0, lib.sf_last_error()
    cu().device_synchronize()
    got = cu().gputensor_to_numpy(gc).astype(np.float32)
    y = got[offset:].reshape(m, n + pad)
    assert np.isnan(y[:, n:]).all() and np.isnan(got[:offset]).all(), "columns past N were written"
    am = (a.T if ta else a).astype(np.float64)
    bm = (b.T if tb else b).astype(np.float64)
    pre = am @ bm + bias
    y64 = ref.act_f64(pre, "silu") + res
    bound = gemm_bound(ref.act_f64(pre, "silu"), np.abs(am) @ np.abs(bm) + np.abs(bias), k, dtype, "silu")
    bound += {"float16": 2.0 ** -11, "bfloat16": 2.0 ** -8}[dtype] * np.abs(y64)  # the sum's one rounding
    check_bound(y[:, :n], y64, bound, "%s" % (case,))
    return y[:, :n].copy()


ALIGNED = [
    # (dtype, transA, transB, M, N, K, plan): one row and column past a tile,
    # a K that is no multiple of 64 (and, with k-rows, of 8), short K
    ("bfloat16", 0, 1, 17, 64, 320, "gemm tile 32x64"),
    ("float16", 0, 1, 33, 72, 4104, "gemm tile 32x64 16-bit split"),
    ("bfloat16", 0, 1, 256, 1000, 1000, "gemm tile 32x64"),
    ("bfloat16", 0, 1, 65, 136, 8, "gemm tile 64x64"),
    ("float16", 0, 1, 300, 500, 2056, "gemm tile 64x64 16-bit split"),
    ("bfloat16", 0, 0, 5, 200, 72, "gemm tile 64x64"),
    ("bfloat16", 0, 0, 600, 1032, 3208, "gemm tile 64x64 16-bit split"),
    ("float16", 1, 0, 200, 136, 77, "gemm tile 64x64"),
    ("bfloat16", 1, 0, 1000, 136, 1350, "gemm tile 64x64 16-bit split"),
    ("bfloat16", 1, 1, 72, 200, 264, "gemm tile 64x64"),
    ("bfloat16", 0, 1, 2700, 2056, 200, "gemm tile 128x128"),
    ("float16", 0, 1, 1297, 1800, 7688, "gemm tile 128x128 16-bit split"),
    ("float16", 0, 0, 2049, 2056, 520, "gemm tile 128x128"),
    ("bfloat16", 1, 0, 2056, 1928, 333, "gemm tile 128x128"),
    ("float16", 1, 1, 2056, 1929, 264, "gemm tile 128x128"),
]
RAGGED = [
    ("float16", 0, 1, 1, 65, 33, "gemm tile generic 64x64"),
    ("bfloat16", 0, 1, 4, 515, 4097, "gemm tile generic 64x64 16-bit split"),
    ("float16", 0, 1, 777, 1283, 1001, "gemm tile generic 64x64"),
    ("bfloat16", 0, 0, 41, 517, 4095, "gemm tile generic 64x64 16-bit split"),
    ("bfloat16", 1, 0, 129, 131, 201, "gemm tile generic 64x64"),
    ("float16", 1, 1, 131, 67, 77, "gemm tile generic 64x64"),
    ("bfloat16", 0, 1, 2500, 1283, 1001, "gemm tile generic"),
    ("bfloat16", 1, 0, 515, 4097, 2001, "gemm tile generic 128x128 16-bit split"),
]


def _id(c):
    return "%s-%s%s-%dx%dx%d" % (c[0], "T" if c[1] else "N", "T" if c[2] else "N", c[3], c[4], c[5])


@pytest.mark.parametrize("case", ALIGNED, ids=_id)
def test_aligned_tiles(case):
    """Rows 8 elements longer than needed, NaN past every edge: nothing
    outside the operands may reach the result."""
    _run(case, pad=8)


@pytest.mark.parametrize("case", RAGGED, ids=_id)
def test_ragged_tiles(case):
    _run(case, pad=3, offset=1)


@pytest.mark.parametrize("case", [ALIGNED[4], ALIGNED[11], RAGGED[7]], ids=_id)
def test_split_sums_are_deterministic_off_their_xcd_too(case):
    """The parts are summed in part order whichever arrives last, and when
    every part takes the agent-scope hand-off (test hook)."""
    y0 = _run(case, reps=3)
    cu()._set_test_hooks(3)
    try:
        y1 = _run(case)
    finally:
        cu()._set_test_hooks()
    assert np.array_equal(y0, y1)


def test_capture_without_a_warm_workspace():
    """A mid-size split call captured into a graph on another stream takes
    the unsplit plan (no allocation, no wait), and every replay matches it."""
    g = cu()
    hip = ctypes.CDLL("libamdhip64.so.7")
    lib = _lib()
    m, n, k = 226, 1920, 4096
    rng = np.random.default_rng(5)
    x, w = rnd(rng, (m, k), 1.0, "bfloat16"), rnd(rng, (n, k), 0.02, "bfloat16")
    gx, gw = up(x, "bfloat16"), up(w, "bfloat16")
    assert "split" in g.gemm_plan(1, m, n, k, 1, gx.data_ptr, k, 0, gw.data_ptr, k, 0, n, 0, gx.dtype)
    gc = up(np.zeros((m, n), np.float32), "bfloat16")
    y64 = ref.linear_f64(x, w)
    bound = gemm_bound(y64, np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T, k, "bfloat16")
    st, graph, ex = P(), P(), P()
    assert lib.sf_stream_create(ctypes.byref(st)) == 0
    g.device_synchronize()
    assert hip.hipStreamBeginCapture(st, 2) == 0  # relaxed
    rc = lib.sf_gemm(0, 1, I64(m), I64(n), I64(k), I64(1), P(gx.data_ptr), I64(k), I64(0), P(gw.data_ptr), I64(k),
                     I64(0), P(gc.data_ptr), I64(n), I64(0), 2, 2, F(1.0), None, 0, st)
    assert hip.hipStreamEndCapture(st, ctypes.byref(graph)) == 0
    assert rc == 0, lib.sf_last_error()
    assert hip.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, ctypes.c_size_t(0)) == 0
    for _ in range(3):
        g.dev_copy(up(np.full((m, n), np.nan, np.float32), "bfloat16"), gc)
        g.device_synchronize()
        assert hip.hipGraphLaunch(ex, st) == 0
        assert lib.sf_stream_synchronize(st) == 0
        check_bound(g.gputensor_to_numpy(gc), y64, bound, "replay")
    hip.hipGraphExecDestroy(ex)
    hip.hipGraphDestroy(graph)
    lib.sf_stream_destroy(st)
