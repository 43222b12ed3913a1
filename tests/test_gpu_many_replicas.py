"""A batch of more replicas than a launch takes blocks on y or z (65535): every
replica's step records and forces are those of the system alone."""
import numpy as np
import pytest

import scenarios
from ls1amd import PREC_FP64, Context

pytestmark = pytest.mark.gpu


def test_more_replicas_than_a_grid_dimension():
    nrep, n, steps = 65536 + 700, 5, 3
    print("replicas", nrep, flush=True)
    s = scenarios.ljts_box(n, 0.035, 1.0, seed=3)  # 8 cells
    assert int(s.box[0] // s.rc) == 2
    with Context(0) as c:
        c.setup_system(s, precision=PREC_FP64)
        c.update_container()
        c.traverse()
        one = c.step(steps, s.dt, use_graph=True)
        alone = c.download(("r", "v", "F"))
    with Context(0) as c:
        c.setup(s.ncomp, s.comp_desc, s.mix, s.eps_rf, s.box, s.rc, s.rc_lj, True, 0, PREC_FP64)
        c.set_replicas(np.tile(s.box, (nrep, 1)), np.full(nrep, n), s.rc, s.rc_lj)
        c.upload(*(np.tile(a, (nrep, 1)) for a in (s.r, s.v, s.q, s.L)), np.tile(s.cid, nrep))
        c.update_container()
        mac = c.traverse()
        per = c.step(steps, s.dt, use_graph=True)
        d = c.download(("r", "v", "F"))
    assert mac.shape == (nrep, 4) and per.shape == (steps, nrep, 6)
    for key in d:
        np.testing.assert_array_equal(d[key].reshape(nrep, n, 3),
                                      np.broadcast_to(alone[key], (nrep, n, 3)))
    np.testing.assert_allclose(per, np.broadcast_to(one[:, None], per.shape), rtol=1e-12,
                               atol=1e-12 * np.abs(one).max())
