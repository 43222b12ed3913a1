"""Uploads and downloads through the pinned ring at the sizes where their path
changes: straight into pinned memory (up to 256 KB in all), one batch and several
through the staging array, chunks that end inside an array, worker threads (from
32 MB), a state of the same shape and of another shape on one context, single
arrays, several contexts at once. Bytes are equal."""
import threading

import numpy as np
import pytest

import scenarios
from ls1amd import Context, MdxError

pytestmark = pytest.mark.gpu
KEYS = ("r", "v", "q", "L")


def state(n, seed):
    s = scenarios.small_mixture(n=150, seed=seed)
    rng = np.random.default_rng(seed)
    s.box = np.full(3, 40.0)
    s.r = rng.uniform(0.0, 40.0, (n, 3))
    s.v, s.L = rng.normal(size=(n, 3)), rng.normal(size=(n, 3))
    s.q = scenarios.random_quaternions(rng, n)
    s.cid = rng.integers(0, s.ncomp, n).astype(np.int32)
    return s


def put(c, s, ids=None):
    c.upload(s.r, s.v, s.q, s.L, s.cid, ids)


def same(c, s, ids=None):
    d = c.download()
    for key in KEYS:
        np.testing.assert_array_equal(d[key], getattr(s, key))
    for key in ("F", "M", "Vi"):
        assert not d[key].any()
    n = len(s.r)
    np.testing.assert_array_equal(d["ids"], np.arange(1, n + 1) if ids is None else ids)


# 1489 molecules: 256 KB for the 22 columns; 11915: the staging array is full;
# 190650: 32 MB
@pytest.mark.parametrize("n", [1, 63, 1489, 1490, 11915, 11916, 100003, 190649, 190651])
def test_round_trip(n):
    print("molecules", n, flush=True)
    s, t, u = state(n, 1), state(n, 2), state(max(1, n // 3), 3)
    t.cid = s.cid  # the same shape
    ids = np.random.default_rng(4).permutation(n).astype(np.uint64)
    with Context(0) as c:
        c.setup(s.ncomp, s.comp_desc, s.mix, s.eps_rf, s.box, s.rc, s.rc_lj, True, 0, 0)
        put(c, s, ids)
        same(c, s, ids)
        put(c, t)
        same(c, t)
        put(c, u)
        same(c, u)
        put(c, s)
        for key in KEYS:
            d = c.download((key,))
            assert list(d) == [key]
            np.testing.assert_array_equal(d[key], getattr(s, key))


def test_order_of_the_upload():
    """Columns come back in upload order once the molecules are sorted into cells."""
    s = state(30011, 5)
    with Context(0) as c:
        c.setup(s.ncomp, s.comp_desc, s.mix, s.eps_rf, s.box, s.rc, s.rc_lj, True, 0, 0)
        put(c, s)
        c.update_container()
        d = c.download()
    np.testing.assert_array_equal(d["r"], s.r)
    np.testing.assert_array_equal(d["v"], s.v)
    np.testing.assert_allclose(d["q"], s.q, rtol=0, atol=1e-15)


def test_a_refused_upload_keeps_the_state():
    s = state(500, 6)
    with Context(0) as c:
        c.setup(s.ncomp, s.comp_desc, s.mix, s.eps_rf, s.box, s.rc, s.rc_lj, True, 0, 0)
        put(c, s)
        bad = s.cid[:100].copy()
        bad[3] = s.ncomp
        with pytest.raises(MdxError):
            c.upload(s.r[:100], s.v[:100], s.q[:100], s.L[:100], bad)
        same(c, s)


def test_contexts_in_threads():
    err = []

    def one(k):
        try:
            s = state(200000 if k < 2 else 700, 10 + k)
            with Context(0) as c:
                c.setup(s.ncomp, s.comp_desc, s.mix, s.eps_rf, s.box, s.rc, s.rc_lj, True, 0, 0)
                for _ in range(3):
                    put(c, s)
                    same(c, s)
        except BaseException as e:  # reported by the test's own thread
            err.append(e)

    threads = [threading.Thread(target=one, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not err, err
