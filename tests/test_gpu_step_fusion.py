"""A step's fused passes (drift and binning, site sums and kicks, scans, the
reductions that end a step) against the separate calls of the same step, at the
sizes where their splits change: scans of one block and of several, block sums
that the adding blocks sum themselves and ones that are scanned first, one and
several blocks per reduction, replicas of different sizes.

The state must be equal bit for bit (the same operations in the same order);
the step records are the same sums, so they agree to rounding (1e-12)."""
import numpy as np
import pytest

import scenarios
from ls1amd import PREC_FP32_FP64ACC, PREC_FP64, Context

pytestmark = pytest.mark.gpu
KEYS = ("r", "v", "q", "L", "F", "M", "Vi")


def separate_steps(c, n, dt):
    rec = []
    for _ in range(n):
        c.leapfrog_pre(dt)
        c.update_container()
        macro = c.traverse()
        rec.append((macro, c.leapfrog_post(dt)))
    return rec


def check(setup, dt, steps=3):
    out = []
    for mode in ("separate", "graph", "plain"):
        with Context(0) as c:
            setup(c)
            c.update_container()
            c.traverse()
            if mode == "separate":
                rec = separate_steps(c, steps, dt)
            else:
                per = c.step(steps, dt, use_graph=mode == "graph")
                per = np.concatenate([per, c.step(1, dt, use_graph=mode == "graph")])
            if mode == "separate":
                rec += separate_steps(c, 1, dt)
                macro = np.array([np.atleast_2d(m) for m, _ in rec])
                sums = np.array([np.atleast_2d(s) for _, s in rec])
            else:
                per = per.reshape(steps + 1, -1, 6)
                u = macro[:, :, 0] / 6 + macro[:, :, 1] + macro[:, :, 3]
                np.testing.assert_allclose(per[:, :, 0], u, rtol=1e-12, atol=1e-12)
                np.testing.assert_allclose(per[:, :, 2:4], sums[:, :, :2], rtol=1e-12)
            out.append(c.download())
    for d in out[1:]:
        for key in KEYS:
            np.testing.assert_array_equal(d[key], out[0][key])


def thin_box(cells, n, seed):
    """n one-centre molecules spread over cells^3 cells."""
    s = scenarios.ljts_box(n, 0.3, 1.0, seed=seed)
    s.r = s.r * (cells + 0.01) * s.rc / s.box
    s.box = np.full(3, (cells + 0.01) * s.rc)
    return s


# 25^3 + 1 and 26^3 + 1 counts: one block, several; 162^3 + 1: more than 4096
# blocks, whose sums are scanned first; the reductions take 4, 5 and 64 blocks
@pytest.mark.parametrize("cells", [25, 26, 162])
def test_many_cells(cells):
    print("cells", cells, flush=True)
    s = thin_box(cells, 1501, seed=cells)
    check(lambda c: c.setup_system(s, precision=PREC_FP64), s.dt)


@pytest.mark.parametrize("n", [16383, 16384, 16385])
def test_site_scans(n):
    """The scans of the molecules' site counts at the edge of one block."""
    print("molecules", n, flush=True)
    s = scenarios.mixture(n=n, seed=n)
    check(lambda c: c.setup_system(s, precision=PREC_FP32_FP64ACC), s.dt, steps=2)


@pytest.mark.parametrize("system", ["one-centre", "multi-site"])
def test_replicas(system):
    print("replicas", system, flush=True)
    if system == "one-centre":
        reps = [scenarios.ljts_box(n, 0.4, 1.0, seed=n) for n in (300, 5000, 64, 1111)]
        reps[2:3] = [thin_box(17, 200, seed=1)]
    else:
        reps = [scenarios.mixture(n=n, seed=n) for n in (300, 2500, 1001)]
    check(lambda c: c.setup_replicas(reps, precision=PREC_FP64), reps[0].dt)
