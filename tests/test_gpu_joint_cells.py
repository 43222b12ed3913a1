"""The quadrupole kernel takes two cells of an x row at a time. Which two depends on
the row alone: not on where a replica's cells begin in the batch (an odd number
of cells before it), nor on the cells per work item."""
import numpy as np
import pytest

import scenarios
from ls1amd import PREC_FP32_FP64ACC, PREC_FP64, Context

pytestmark = pytest.mark.gpu
KEYS = ("F", "M", "Vi")


def odd_box(seed):
    s = scenarios.mixture(n=11500, rho=0.3, seed=seed)
    assert int(s.box[0] // s.rc) == 11  # 1331 cells, rows of 11
    return s


@pytest.mark.parametrize("prec", [PREC_FP64, PREC_FP32_FP64ACC])
def test_replicas_behind_an_odd_number_of_cells(prec):
    reps = [odd_box(1), odd_box(2), scenarios.mixture(n=9000, rho=0.3, seed=3), odd_box(4)]
    with Context(0) as c:
        c.setup_replicas(reps, precision=prec)
        c.update_container()
        c.traverse()
        d = c.download()
    at = 0
    for k, s in enumerate(reps):
        print("replica", k, flush=True)
        with Context(0) as c:
            c.setup_system(s, precision=prec)
            c.update_container()
            c.traverse()
            alone = c.download()
        for key in KEYS:
            np.testing.assert_array_equal(d[key][at:at + s.n], alone[key])
        at += s.n


@pytest.mark.parametrize("shape", [(2, 0), (3, 0), (5, 16), (1, 8)])
def test_cells_per_item(shape):
    print("shape", shape, flush=True)
    s = odd_box(7)
    with Context(0) as c:
        c.setup_system(s, precision=PREC_FP32_FP64ACC)
        c.update_container()
        m_ref = c.traverse()
        ref = c.download()
        c.set_pair_config(*shape)
        m = c.traverse()
        d = c.download()
    for key in KEYS:
        np.testing.assert_array_equal(d[key], ref[key])
    np.testing.assert_allclose(m, m_ref, rtol=1e-12, atol=1e-12 * np.abs(m_ref).max())
