"""mdx_upload_device reads arrays that the caller's own stream may still be
writing: the call waits for that work, for a first state and for one that takes
the arrays of the state before it (no allocation, no free)."""
import ctypes as C

import numpy as np
import pytest

import scenarios
from ls1amd import Context

pytestmark = pytest.mark.gpu


def put(c, s, arrays, cid):
    ptr = [C.c_void_p(a.data_ptr()) for a in arrays + [cid]]
    c._chk(c.L.mdx_upload_device(c.h, s.n, *ptr), "mdx_upload_device")
    c.n = s.n


def test_work_of_another_stream_is_waited_for():
    import torch

    s = scenarios.small_mixture(n=4000, seed=2)
    dev = torch.device("cuda:0")
    rows = [np.ascontiguousarray(a.T) for a in (s.r, s.v, s.q, s.L)]
    cid = torch.from_numpy(s.cid).to(dev)
    busy = torch.zeros((4096, 4096), device=dev)
    side = torch.cuda.Stream()  # (not ordered with the null stream)
    with Context(0) as c:
        c.setup(s.ncomp, s.comp_desc, s.mix, s.eps_rf, s.box, s.rc, s.rc_lj, True, 0, 0)
        for shift in (0.0, 0.25, 0.5):
            print("upload", shift, flush=True)
            want = [torch.from_numpy(a + shift * (k > 0)).to(dev) for k, a in enumerate(rows)]
            given = [torch.zeros_like(a) for a in want]
            torch.cuda.synchronize()
            with torch.cuda.stream(side):
                for _ in range(40):  # some milliseconds of work before the arrays are written
                    busy = busy @ busy
                for g, w in zip(given, want):
                    g.copy_(w)
            put(c, s, given, cid)
            d = c.download(("r", "v", "q", "L"))
            for key, w in zip(("r", "v", "q", "L"), want):
                np.testing.assert_array_equal(d[key], w.cpu().numpy().T)
