"""Run by tests/test_capture_gpu.py in a fresh child process, so no split
plan has run on the device before: captures split-plan GEMMs of every kind
cold, then lets eager calls allocate and grow the split workspace before and
between the replays.  Prints one JSON line."""
from __future__ import annotations

import ctypes
import json
import os
import sys

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
for p in (ROOT, HERE):
    if p not in sys.path:
        sys.path.insert(0, p)

from helpers import cu, gemm_bound, rnd, sample_rows, up  # noqa: E402

I64, P, F, SZ = ctypes.c_int64, ctypes.c_void_p, ctypes.c_float, ctypes.c_size_t
SFD = {"float32": 0, "float16": 1, "bfloat16": 2}
CASES = [
    # (dtype, transA, transB, M, N, K): mid-size, every 256 x 256 tile split
    # (NT, NN, TN), a split tail, fp32 with and without whole slices
    ("bfloat16", 0, 1, 226, 1920, 4096),
    ("bfloat16", 0, 1, 2048, 2048, 16384),
    ("float16", 0, 0, 2048, 2048, 16384),
    ("bfloat16", 1, 0, 1920, 1920, 4000),
    ("bfloat16", 0, 1, 4352, 4096, 4096),
    ("float32", 0, 1, 64, 4096, 4096),
    ("float32", 0, 1, 33, 1025, 4097),
    ("float32", 1, 0, 512, 512, 4096),
]


def main() -> None:
    g = cu()
    lib = ctypes.CDLL(os.path.join(ROOT, "scaffolding_amd", "libsfgemm.so"))
    hip = ctypes.CDLL("libamdhip64.so.7")
    lib.sf_last_error.restype = ctypes.c_char_p
    g.set_device(0)

    def args(c, a, b, out, st):
        dt, ta, tb, m, n, k = c
        return (ta, tb, I64(m), I64(n), I64(k), I64(1), P(a.data_ptr), I64(m if ta else k), I64(0), P(b.data_ptr),
                I64(k if tb else n), I64(0), P(out.data_ptr), I64(n), I64(0), SFD[dt], SFD[dt], F(1.0), None, 0) + st

    def ok(rc):
        if rc != 0:
            raise RuntimeError(lib.sf_last_error().decode())

    def held():
        free, total, ws = SZ(0), SZ(0), SZ(0)
        ok(lib.sf_device_synchronize())
        ok(lib.sf_mem_get_info(ctypes.byref(free), ctypes.byref(total)))
        ok(lib.sf_workspace_bytes(0, ctypes.byref(ws)))
        return int(free.value), int(ws.value)

    # operands, outputs and, uncaptured and unsplit, one call (code objects)
    ops = []
    for i, c in enumerate(CASES):
        dt, ta, tb, m, n, k = c
        rng = np.random.default_rng(i)
        a = rnd(rng, (k, m) if ta else (m, k), 1.0, dt)
        b = rnd(rng, (n, k) if tb else (k, n), 1.0 / np.sqrt(k), dt)
        rows = sample_rows(m, 6, i)
        am = (a.T if ta else a)[rows].astype(np.float64)
        bm = (b.T if tb else b).astype(np.float64)
        y64 = am @ bm
        bound = gemm_bound(y64, np.abs(am) @ np.abs(bm), k, dt)
        ops.append((up(a, dt), up(b, dt), up(np.zeros((m, n), np.float32), dt), rows, y64, bound))
        buf = ctypes.create_string_buffer(96)
        ok(lib.sf_gemm_plan(*args(c, *ops[i][:3], (buf, 96))))
        if b"split" not in buf.value:
            raise RuntimeError("%s: plan %s has no split" % (c, buf.value))
    for dt in ("float32", "float16", "bfloat16"):
        w = up(np.zeros((256, 256), np.float32), dt)
        ok(lib.sf_gemm(*args((dt, 0, 1, 256, 256, 256), w, w, up(np.zeros((256, 256), np.float32), dt), (None,))))
    st = P()
    ok(lib.sf_stream_create(ctypes.byref(st)))
    free0, ws0 = held()

    graphs = []
    for c, op in zip(CASES, ops):
        print("capture", c, file=sys.stderr, flush=True)
        graph, ex = P(), P()
        assert hip.hipStreamBeginCapture(st, 0) == 0  # global mode
        rc = lib.sf_gemm(*args(c, *op[:3], (st,)))
        assert hip.hipStreamEndCapture(st, ctypes.byref(graph)) == 0
        ok(rc)
        graphs.append((graph, ex))
    free1, ws1 = held()
    for graph, ex in graphs:
        assert hip.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, SZ(0)) == 0

    worst = 0.0
    for rep in range(3):
        # eager split calls, small then large: the workspace is allocated and
        # grown after the capture; the last one still runs beside the replay
        for i in (0, 5, 1, 4):
            tmp = up(np.zeros(CASES[i][3:5], np.float32), CASES[i][0])
            ok(lib.sf_gemm(*args(CASES[i], ops[i][0], ops[i][1], tmp, (None,))))
        for c, op, (graph, ex) in zip(CASES, ops, graphs):
            print("replay", rep, c, file=sys.stderr, flush=True)
            ok(lib.sf_zero(P(op[2].data_ptr), SZ(op[2].nbytes), st))
            assert hip.hipGraphLaunch(ex, st) == 0
            ok(lib.sf_stream_synchronize(st))
            y = g.gputensor_to_numpy(op[2])[op[3]].astype(np.float64)
            worst = max(worst, float(np.max(np.abs(y - op[4]) / op[5])))
    print(json.dumps({"ws": [ws0, ws1, held()[1]], "free": [free0, free1], "worst": worst}), flush=True)
    for graph, ex in graphs:
        hip.hipGraphExecDestroy(ex)
        hip.hipGraphDestroy(graph)


if __name__ == "__main__":
    main()
