"""Context.download(keys): every array that comes back was filled by the library."""
import ctypes as C

import numpy as np
import pytest

from ls1amd import Context

NAMES = ("r", "v", "q", "L", "F", "M", "Vi", "ids")


class FakeLibrary:
    """mdx_download that fills each array it is given with its place in the call."""

    def mdx_download(self, h, n, *ptrs):
        self.given = [k for k, p in zip(NAMES, ptrs) if p is not None]
        for place, p in enumerate(ptrs):
            if p is None:
                continue
            typ = C.c_uint64 if NAMES[place] == "ids" else C.c_double
            width = {"ids": 1, "q": 4}.get(NAMES[place], 3)
            np.ctypeslib.as_array(C.cast(p, C.POINTER(typ)), (n * width,))[:] = place
        return 0

    def mdx_last_error(self, h):
        return b""


def context(n=3):
    c = Context.__new__(Context)
    c.L, c.h, c.n, c.open = FakeLibrary(), None, n, False
    c.close = lambda: None
    return c


@pytest.mark.parametrize("keys", [None, ("F",), ("ids", "q"), ["r", "Vi"], ()])
def test_every_array_is_filled(keys):
    c = context()
    d = c.download(keys)
    assert list(d) == list(NAMES if keys is None else keys)
    assert sorted(c.L.given) == sorted(d)
    for k, a in d.items():
        assert np.all(a == NAMES.index(k))


@pytest.mark.parametrize("keys", [("f",), ("F", "virial"), ["ids", "id"], "Fx"])
def test_an_unknown_array_is_refused(keys):
    with pytest.raises(ValueError, match="no arrays"):
        context().download(keys)
