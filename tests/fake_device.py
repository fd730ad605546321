"""The library's host code on a HIP runtime without a GPU (fake_device.cpp):
plans, footprints and the server's scheduling, checked on the CPU."""
from __future__ import annotations

import ctypes as C
import subprocess
import time
from pathlib import Path

import numpy as np

from gpumemefficient_amd import _lib, _server_abi

HERE = Path(__file__).resolve().parent
CSRC = HERE.parent / "gpumemefficient_amd" / "csrc"
SOURCES = ["wf_api.cpp", "wf_server.cpp", "wf_tune.cpp", "wf_stencil_api.cpp", "wf_noalloc.hip"]


def build(out: Path) -> "Fake":
    so = out / "libfake.so"
    cmd = ["g++", "-std=c++17", "-O1", "-w", "-fPIC", "-shared", "-Wl,-Bsymbolic", "-D__HIP_PLATFORM_AMD__",
           "-I/opt/rocm/include", "-include", str(HERE / "fake_device.h"), "-x", "c++",
           *(str(CSRC / s) for s in SOURCES), str(HERE / "fake_device.cpp"), "-o", str(so), "-lpthread", "-ldl"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    return Fake(so)


def i32(x):
    return x.ctypes.data_as(C.POINTER(C.c_int32))


class Fake:
    def __init__(self, so: Path):
        P, i64, size = C.c_void_p, C.c_int64, C.c_size_t
        self.c = lib = C.CDLL(str(so))
        for name, res, args in [
                ("fake_set_memory", None, [size]), ("fake_live", size, []), ("fake_peak", size, []),
                ("fake_hold", None, [C.c_int]), ("fake_free_hold", None, [C.c_int]), ("fake_release", None, []), ("fake_launches", C.c_int, []), ("fake_last_engine", C.c_int, []),
                ("fake_tasks", i64, []), ("hipMalloc", C.c_int, [C.POINTER(P), size]), ("hipFree", C.c_int, [P]),
                ("wf_ctx_create", C.c_int, [C.c_int, C.POINTER(P)]), ("wf_ctx_destroy", None, [P]),
                ("wf_align_batch", C.c_int, [P, P, i64, P, P]),
                ("wf_align_noalloc", C.c_int, [P, C.c_int, P, i64, P, i64, P, P]),
                ("wf_plan_create", C.c_int, [P, P, i64, P, C.POINTER(P)]), ("wf_plan_run", C.c_int, [P, C.c_int]),
                ("wf_plan_describe", C.c_int, [P, P, P, P, P, C.POINTER(i64), P]), ("wf_plan_destroy", None, [P]),
                ("wf_stencil_device", C.c_int, [P, C.c_int, i64, i64, P, i64, P, P])]:
            f = getattr(lib, name)
            f.restype, f.argtypes = res, args
        _server_abi.bind(lib)
        self.ctx = P()
        assert lib.wf_ctx_create(0, C.byref(self.ctx)) == 0

    def jobs(self, pairs):
        """wf_job array of (problem, a, b[, flags]); keeps the symbols alive."""
        arr = (_lib.wf_job * len(pairs))()
        for j, (prob, a, b, *fl) in zip(arr, pairs):
            j.problem, j.flags = _lib.PROBLEMS[prob], fl[0] if fl else 0
            j.a, j.n1, j.b, j.n2 = i32(a), a.size, i32(b), b.size
        arr.keep = pairs
        return arr

    def server(self, **opts):
        h = C.c_void_p()
        o = _server_abi.wf_server_opts(**opts)
        assert self.c.wf_server_create(0, C.byref(o), C.byref(h)) == 0
        return h

    def submit(self, srv, job):
        assert self.c.wf_server_submit(srv, self.jobs([job]), None) == 0

    def stats(self, srv):
        st = _server_abi.wf_server_stats_t()
        assert self.c.wf_server_stats(srv, C.byref(st)) == 0
        return st

    def done(self, srv, n, limit=20.0):
        """Statuses of n completions (fewer after `limit` seconds)."""
        out, got, k, end = (_server_abi.wf_completion * n)(), [], C.c_int(), time.monotonic() + limit
        while len(got) < n and time.monotonic() < end:
            assert self.c.wf_server_poll(srv, out, n - len(got), C.byref(k)) == 0
            got += [out[i].status for i in range(k.value)]
            time.sleep(0.0005)
        return got

    def plan(self, pairs):
        """(status, plan handle, tasks)."""
        h, n = C.c_void_p(), C.c_int64()
        st = self.c.wf_plan_create(self.ctx, self.jobs(pairs), len(pairs), None, C.byref(h))
        if st == 0:
            self.c.wf_plan_describe(h, None, None, None, None, C.byref(n), None)
        return st, h, n.value


def pair(prob, n1, n2, k=4, seed=0, flags=0):
    rng = np.random.default_rng(seed)
    a, b = rng.integers(0, k, n1, dtype=np.int32), rng.integers(0, k, n2, dtype=np.int32)
    a[:min(k, n1)] = np.arange(min(k, n1))  # all of the alphabet
    return prob, a, b, flags
