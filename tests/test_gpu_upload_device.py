"""mdx_upload_device reads arrays that the caller's own stream may still be
writing: the call waits for that work, for a first state and for one that takes
the arrays of the state before it (no allocation, no free)."""
import ctypes as C

import numpy as np
import pytest

import ls1amd
import scenarios
from ls1amd import Context

pytestmark = pytest.mark.gpu
NONBLOCKING, H2D, D2D = 1, 1, 3


class Hip:
    """The HIP runtime that the library is linked with."""

    def __init__(self):
        ls1amd.load()
        with open("/proc/self/maps") as f:
            path = next(line.split()[-1] for line in f
                        if "libamdhip64" in line and "torch" not in line)
        self.lib = C.CDLL(path)
        self.mem = []
        self.stream = C.c_void_p()
        self("hipStreamCreateWithFlags", C.byref(self.stream), C.c_uint(NONBLOCKING))

    def __call__(self, name, *args):
        rc = getattr(self.lib, name)(*args)
        assert rc == 0, (name, rc)

    def array(self, data=None, nbytes=0):
        p = C.c_void_p()
        self("hipMalloc", C.byref(p), C.c_size_t(nbytes or data.nbytes))
        self.mem.append(p)
        if data is not None:
            self("hipMemcpy", p, data.ctypes.data_as(C.c_void_p), C.c_size_t(data.nbytes), H2D)
        return p

    def copy_on_stream(self, dst, src, nbytes):
        self("hipMemcpyAsync", dst, src, C.c_size_t(nbytes), D2D, self.stream)

    def close(self):
        self("hipStreamSynchronize", self.stream)
        for p in self.mem:
            self("hipFree", p)
        self("hipStreamDestroy", self.stream)


def test_work_of_another_stream_is_waited_for():
    s = scenarios.small_mixture(n=4000, seed=2)
    keys = ("r", "v", "q", "L")
    hip = Hip()
    big = 256 << 20
    a, b = hip.array(nbytes=big), hip.array(nbytes=big)
    cid = hip.array(s.cid)
    with Context(0) as c:
        c.setup(s.ncomp, s.comp_desc, s.mix, s.eps_rf, s.box, s.rc, s.rc_lj, True, 0, 0)
        for shift in (0.0, 0.25, 0.5):
            print("upload", shift, flush=True)
            rows = [np.ascontiguousarray((getattr(s, k) + shift * (k != "r")).T) for k in keys]
            want = [hip.array(x) for x in rows]
            given = [hip.array(np.zeros_like(x)) for x in rows]
            for _ in range(40):  # milliseconds of work before the arrays are written
                hip.copy_on_stream(a, b, big)
            for g, w, x in zip(given, want, rows):
                hip.copy_on_stream(g, w, x.nbytes)
            c._chk(c.L.mdx_upload_device(c.h, s.n, *given, cid), "mdx_upload_device")
            c.n = s.n
            d = c.download(keys)
            for key, x in zip(keys, rows):
                np.testing.assert_array_equal(d[key], x.T)
    hip.close()
