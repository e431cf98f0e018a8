"""Build of main_amd/csrc/mpcx_stage.hip for the host (tests/stage), through ctypes."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


class Stage:
    def __init__(self, folder):
        gxx = shutil.which("g++")
        if gxx is None:
            pytest.skip("no g++")
        so = os.path.join(str(folder), "libstage_host.so")
        d = os.path.join(HERE, "stage")
        subprocess.run([gxx, "-std=c++17", "-O1", "-g", "-fPIC", "-shared", "-pthread", "-I", d,
                        os.path.join(d, "stage_host.cpp"), "-o", so], check=True)
        self.c = C.CDLL(so)
        for f in ("t_used", "t_mallocs", "t_frees", "t_host_mallocs", "t_events", "t_direct"):
            getattr(self.c, f).restype = C.c_size_t
        for f in ("t_alloc", "t_block_get"):
            getattr(self.c, f).restype = C.c_void_p

    def reset(self, heap=1 << 60):
        self.c.t_reset(C.c_size_t(heap))

    def get(self, n):
        """A block of at least n bytes: (address, its size), or None."""
        got = C.c_size_t()
        p = self.c.t_block_get(C.c_size_t(n), C.byref(got))
        return (p, got.value) if p else None

    def put(self, block):
        self.c.t_block_put(C.c_void_p(block[0]), C.c_size_t(block[1]))

    def pin(self, a):
        self.c.t_pin(C.c_void_p(a.ctypes.data), C.c_size_t(a.nbytes))

    def copy(self, host, dev, out, widen=None, fail_at=-1):
        n = len(host)
        arr = lambda v, t: (t * n)(*v)
        widen = widen or [0] * n
        addr = lambda a: None if a is None else a.ctypes.data
        return self.c.t_copy(C.c_int(n), arr([addr(a) for a in host], C.c_void_p), arr([addr(a) for a in dev], C.c_void_p),
                             arr([a.nbytes for a in dev], C.c_size_t), arr(widen, C.c_int), C.c_int(out),
                             C.c_long(fail_at))


def rng_bytes(n, seed):
    return np.random.default_rng(seed).integers(0, 256, n, dtype=np.uint8)
