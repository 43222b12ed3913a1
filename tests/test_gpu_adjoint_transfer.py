"""The adjoint's arrays go as plain copies below 8 MB and through the pinned ring with
helping threads from there on: both sides of the line give the bits of
mdx_adjoint_noalloc, which always copies plainly, and the cotangent that was
given is not written."""
import numpy as np
import pytest

import scenarios
from ls1amd import PREC_FP64, Context

pytestmark = pytest.mark.gpu
LINE = (8 << 20) // 24  # molecules whose array is just below 8 MB


@pytest.mark.parametrize("n", [2, 63, 4001, LINE, LINE + 1, 500000])
def test_both_sides_of_the_line(n):
    print("molecules", n, flush=True)
    s = scenarios.binary_lj(n=max(n, 800), rho=0.6)
    s.r, s.v, s.q, s.L, s.cid = s.r[:n], s.v[:n], s.q[:n], s.L[:n], s.cid[:n]
    cot = np.random.default_rng(n).normal(size=(n, 3))
    kept = cot.copy()
    with Context(0) as c:
        c.setup_system(s, precision=PREC_FP64)
        c.update_container()
        ref = c.adjoint(cot, noalloc=True)
        for _ in range(2):
            out = c.adjoint(cot)
            for key in ref:
                np.testing.assert_array_equal(out[key], ref[key])
        assert ref["vjp"].shape == (n, 3)
        plain = c.adjoint()
        for key in plain:
            np.testing.assert_array_equal(plain[key], ref[key])
    np.testing.assert_array_equal(cot, kept)
