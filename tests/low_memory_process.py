"""Run by tests/test_workspace_streams_gpu.py in a child process: takes the
device's memory but for a rest smaller than a split workspace, then runs
split-plan GEMMs.  Prints one JSON line."""
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

from helpers import cu, gemm_walk_bound, rnd, up  # noqa: E402

I64, P, F, SZ = ctypes.c_int64, ctypes.c_void_p, ctypes.c_float, ctypes.c_size_t
MB = 1 << 20


def main() -> None:
    g = cu()
    lib = ctypes.CDLL(os.path.join(ROOT, "scaffolding_amd", "libsfgemm.so"))
    lib.sf_last_error.restype = ctypes.c_char_p
    g.set_device(0)
    m, n, k = 2048, 2048, 16384  # 64 tiles in 4 parts of 256 KB
    rng = np.random.default_rng(6)
    x, w = rnd(rng, (m, k), 1.0, "bfloat16"), rnd(rng, (n, k), 1.0 / np.sqrt(k), "bfloat16")
    gx, gw, out = up(x, "bfloat16"), up(w, "bfloat16"), g.empty((m, n), g.BFLOAT16)

    def gemm(mm, nn, kk, a, b, c):
        return lib.sf_gemm(0, 1, I64(mm), I64(nn), I64(kk), I64(1), P(a.data_ptr), I64(kk), I64(0), P(b.data_ptr),
                           I64(kk), I64(0), P(c.data_ptr), I64(nn), I64(0), 2, 2, F(1.0), None, 0, None)

    z, zc = g.zeros((256, 256), g.BFLOAT16), g.empty((256, 256), g.BFLOAT16)
    rcs = [gemm(256, 256, 256, z, z, zc)]  # unsplit: code loaded, queue made
    g.device_synchronize()
    held = []
    size = 64 * 1024 * MB
    while size >= 32 * MB:
        ptr = P()
        if lib.sf_malloc(ctypes.byref(ptr), SZ(size)) == 0:
            held.append(ptr)
        else:
            size //= 2
    rcs.append(gemm(m, n, k, gx, gw, out))
    err = lib.sf_last_error().decode()
    rcs.append(lib.sf_device_synchronize())
    ws = SZ(0)
    lib.sf_workspace_bytes(0, ctypes.byref(ws))
    for ptr in held:
        lib.sf_free(ptr)
    rows = np.array([0, 255, 256, m - 1])
    a, b = x[rows].astype(np.float64), w.T.astype(np.float64)
    y64 = a @ b
    worst = float(np.max(np.abs(g.gputensor_to_numpy(out)[rows] - y64) / gemm_walk_bound(a, b, y64, "bfloat16")))
    print(json.dumps({"rcs": rcs, "error": err, "ws": int(ws.value), "held": len(held), "worst": worst}), flush=True)


if __name__ == "__main__":
    main()
