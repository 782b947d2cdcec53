"""Split plans on several streams and threads: streams with a workspace of
their own overlap, more streams than workspaces share them in order, and
their sums stay what they are on one stream."""
from __future__ import annotations

import ctypes
import json
import os
import subprocess
import sys
import threading

import numpy as np
import pytest

from helpers import cu, down, rnd, up

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
I64, P, F = ctypes.c_int64, ctypes.c_void_p, ctypes.c_float
M, N, K = 226, 1920, 4096  # four k parts on 64 x 64 tiles


def _lib():
    return ctypes.CDLL(os.path.join(ROOT, "scaffolding_amd", "libsfgemm.so"))


def _operands(seed):
    rng = np.random.default_rng(seed)
    return up(rnd(rng, (M, K), 1.0, "bfloat16"), "bfloat16"), up(rnd(rng, (N, K), 0.02, "bfloat16"), "bfloat16")


def _gemm(lib, x, w, out, st):
    return lib.sf_gemm(0, 1, I64(M), I64(N), I64(K), I64(1), P(x.data_ptr), I64(K), I64(0), P(w.data_ptr), I64(K),
                       I64(0), P(out.data_ptr), I64(N), I64(0), 2, 2, F(1.0), None, 0, st)


def _streams(lib, n):
    streams = [P() for _ in range(n)]
    for s in streams:
        assert lib.sf_stream_create(ctypes.byref(s)) == 0
    return streams


def test_two_streams_overlap():
    """A split call on one stream does not wait for the split call that
    another stream has behind a long, one-workgroup launch."""
    g, lib = cu(), _lib()
    hip = ctypes.CDLL("libamdhip64.so.7")
    assert g.gemm_plan(1, M, N, K, 1, 1 << 20, K, 0, 1 << 20, K, 0, N, 0, g.BFLOAT16).endswith("4")
    x, w = _operands(1)
    outs = [g.empty((M, N), g.BFLOAT16) for _ in range(2)]
    cols = 40_000_000
    row = g.zeros((1, cols))
    row_out = g.empty((1, cols))
    a, b = _streams(lib, 2)
    g.device_synchronize()
    for st in (a, b, a, b):  # workspaces allocated, code loaded
        assert _gemm(lib, x, w, outs[0], st) == 0
        assert lib.sf_stream_synchronize(st) == 0
    assert lib.sf_rms_norm(P(row.data_ptr), P(row_out.data_ptr), I64(1), I64(8), None, F(1e-5), 0, a) == 0
    assert lib.sf_stream_synchronize(a) == 0
    assert lib.sf_rms_norm(P(row.data_ptr), P(row_out.data_ptr), I64(1), I64(cols), None, F(1e-5), 0, a) == 0
    assert _gemm(lib, x, w, outs[0], a) == 0
    assert _gemm(lib, x, w, outs[1], b) == 0
    assert lib.sf_stream_synchronize(b) == 0
    still_running = hip.hipStreamQuery(a) == 600  # hipErrorNotReady
    assert lib.sf_stream_synchronize(a) == 0
    hip.hipGetLastError()
    assert still_running
    assert np.array_equal(down(outs[0]), down(outs[1]))
    for st in (a, b):
        lib.sf_stream_destroy(st)


def test_more_streams_than_workspaces():
    """Six streams from three threads, then streams destroyed right after
    their last call and new ones in their place: every sum bit for bit."""
    g, lib = cu(), _lib()
    ops = [_operands(10 + i) for i in range(6)]
    want = []
    for x, w in ops:
        out = g.empty((M, N), g.BFLOAT16)
        assert _gemm(lib, x, w, out, None) == 0
        want.append(down(out))
    outs = [g.empty((M, N), g.BFLOAT16) for _ in range(6)]
    g.device_synchronize()
    errors = []
    for _ in range(3):
        streams = _streams(lib, 6)

        def worker(t):
            for i in range(60):
                j = 2 * t + i % 2
                rc = _gemm(lib, *ops[j], outs[j], streams[j])
                if rc != 0:
                    errors.append(rc)

        ts = [threading.Thread(target=worker, args=(t,)) for t in range(3)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        assert not errors
        for s in streams:
            assert lib.sf_stream_destroy(s) == 0
        g.device_synchronize()
        for out, y in zip(outs, want):
            assert np.array_equal(down(out), y)


def test_cache_empty_gives_back_all_but_one():
    g, lib = cu(), _lib()
    x, w = _operands(2)
    out = g.empty((M, N), g.BFLOAT16)
    held = lambda: (lib.sf_workspace_bytes(0, ctypes.byref(n)), n.value)[1]  # noqa: E731
    n = ctypes.c_size_t(0)
    assert _gemm(lib, x, w, out, None) == 0
    y = down(out)
    assert lib.sf_cache_empty(-1) == 0
    one = held()
    streams = _streams(lib, 3)
    g.device_synchronize()
    for st in streams:
        assert _gemm(lib, x, w, out, st) == 0 and lib.sf_stream_synchronize(st) == 0
    assert held() > one
    assert lib.sf_cache_empty(-1) == 0
    assert held() <= one
    for st in streams:  # and they are taken again
        assert _gemm(lib, x, w, out, st) == 0 and lib.sf_stream_synchronize(st) == 0
        assert np.array_equal(down(out), y)
        lib.sf_stream_destroy(st)


def test_eager_split_call_beside_a_capture():
    """An eager call whose first split needs memory succeeds while another
    stream is being captured in the global mode, and leaves that capture
    valid."""
    g, lib = cu(), _lib()
    hip = ctypes.CDLL("libamdhip64.so.7")
    x, w = _operands(4)
    outs = [up(np.zeros((M, N), np.float32), "bfloat16") for _ in range(2)]
    assert lib.sf_cache_empty(-1) == 0  # no second workspace is left
    streams = _streams(lib, 2)
    g.device_synchronize()
    graph = P()
    assert hip.hipStreamBeginCapture(streams[0], 0) == 0
    rc0 = _gemm(lib, x, w, outs[0], streams[0])
    rc1 = _gemm(lib, x, w, outs[1], streams[1])
    assert hip.hipStreamEndCapture(streams[0], ctypes.byref(graph)) == 0 and graph.value
    assert rc0 == 0 and rc1 == 0
    assert lib.sf_stream_synchronize(streams[1]) == 0
    want = up(np.zeros((M, N), np.float32), "bfloat16")
    g.device_synchronize()
    assert _gemm(lib, x, w, want, None) == 0
    g.device_synchronize()
    assert np.array_equal(down(outs[1]), down(want))
    hip.hipGraphDestroy(graph)
    for s in streams:
        lib.sf_stream_destroy(s)


def test_no_memory_left_for_a_workspace():
    """A split plan runs unsplit where its workspace cannot be allocated."""
    r = subprocess.run([sys.executable, os.path.join(ROOT, "tests", "low_memory_process.py")], capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
    out = json.loads(r.stdout.strip().splitlines()[-1])
    assert out["rcs"] == [0, 0, 0] and out["ws"] == 0 and out["held"] > 0 and out["worst"] <= 1.0, out


def test_per_thread_streams():
    """hipStreamPerThread is another stream in every thread: split calls on
    it from several threads keep apart."""
    g, lib = cu(), _lib()
    ops = [_operands(20 + i) for i in range(3)]
    want, outs = [], [g.empty((M, N), g.BFLOAT16) for _ in range(3)]
    for x, w in ops:
        out = g.empty((M, N), g.BFLOAT16)
        assert _gemm(lib, x, w, out, None) == 0
        want.append(down(out))
    g.device_synchronize()
    errors = []

    def worker(i):
        for _ in range(40):
            rc = _gemm(lib, *ops[i], outs[i], P(2))
            if rc != 0:
                errors.append(rc)
        lib.sf_stream_synchronize(P(2))

    ts = [threading.Thread(target=worker, args=(i,)) for i in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    g.device_synchronize()
    assert not errors
    for out, y in zip(outs, want):
        assert np.array_equal(down(out), y)
