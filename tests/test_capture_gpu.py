"""Calls captured into HIP graphs: split-plan GEMMs hold no library memory,
attention and column sums only the capture buffer, and every replay gives
what the eager call gives, whatever eager calls run between."""
from __future__ import annotations

import ctypes
import json
import os
import subprocess
import sys

import numpy as np
import pytest

from helpers import cu, down, rnd, up

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
I64, P, F = ctypes.c_int64, ctypes.c_void_p, ctypes.c_float


def test_cold_captures_of_split_gemms():
    """In a fresh process: the captures allocate nothing, and the replays are
    right after eager calls have allocated and grown the split workspace."""
    r = subprocess.run([sys.executable, os.path.join(ROOT, "tests", "capture_fresh_process.py")],
                       capture_output=True, text=True, timeout=240)
    assert r.returncode == 0, r.stdout + r.stderr
    out = json.loads(r.stdout.strip().splitlines()[-1])
    assert out["ws"][0] == 0 and out["ws"][1] == 0 and out["ws"][2] > 0, out
    assert out["free"][1] == out["free"][0], out
    assert out["worst"] <= 1.0, out


def test_captured_attention_and_column_sums():
    """Split attention and column sums captured, the second graph's partials
    larger than the first's (the capture buffer moves), eager calls of both
    between the replays: each replay equals the eager result bit for bit."""
    g = cu()
    hip = ctypes.CDLL("libamdhip64.so.7")
    lib = ctypes.CDLL(os.path.join(ROOT, "scaffolding_amd", "libsfgemm.so"))
    rng = np.random.default_rng(2)
    x = up(rnd(rng, (5000, 640), 1.0, "bfloat16"), "bfloat16")
    q = up(rnd(rng, (1, 300, 64), 1.0, "bfloat16"), "bfloat16")
    kv = up(rnd(rng, (1, 4096, 64), 1.0, "bfloat16"), "bfloat16")
    sums, att = g.empty((640,), g.BFLOAT16), g.empty((1, 300, 64), g.BFLOAT16)

    def run_sum(st):
        return lib.sf_sum_dim(P(x.data_ptr), P(sums.data_ptr), I64(1), I64(5000), I64(640), 2, 2, st)

    def run_att(st):
        k = [P(kv.data_ptr), I64(64), I64(0)]
        return lib.sf_attention(P(q.data_ptr), I64(64), I64(0), *k, *k, P(att.data_ptr), I64(64), I64(300 * 64), I64(1),
                                I64(300), I64(4096), I64(64), F(0.125), 2, st)

    st = P()
    assert lib.sf_stream_create(ctypes.byref(st)) == 0
    runs, want, graphs = [(run_sum, sums), (run_att, att)], [], []
    for run, out in runs:
        assert run(None) == 0
        want.append(down(out))
    g.device_synchronize()
    for run, _ in runs:
        graph, ex = P(), P()
        assert hip.hipStreamBeginCapture(st, 0) == 0
        rc = run(st)
        assert hip.hipStreamEndCapture(st, ctypes.byref(graph)) == 0 and rc == 0
        assert hip.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, ctypes.c_size_t(0)) == 0
        graphs.append((graph, ex))
    for _ in range(3):
        for run, _o in runs:
            assert run(None) == 0
        g.device_synchronize()
        for (graph, ex), (_r, out), y in zip(graphs, runs, want):
            assert lib.sf_zero(P(out.data_ptr), ctypes.c_size_t(out.nbytes), st) == 0
            assert hip.hipGraphLaunch(ex, st) == 0 and lib.sf_stream_synchronize(st) == 0
            assert np.array_equal(down(out), y)
    for graph, ex in graphs:
        hip.hipGraphExecDestroy(ex)
        hip.hipGraphDestroy(graph)
    lib.sf_stream_destroy(st)
