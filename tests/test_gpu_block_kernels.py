"""The block pair kernels (boxes of few cells: four waves share a cell) at the
sizes where their split can go wrong, against the oracle: cells with fewer
sites than waves and with more than one pass or one list takes, one and two
cells per dimension (images of the same cells), several LJ ids in the LDS and
in the global parameter table, all site types, coincident molecules, and the
first box beyond the line, where the cell kernels run.

Bars as in test_gpu_parity.py: FP64 form 1e-12 relative to the largest value,
FP32 form relative RMS force error 1e-5, in-cutoff pair counts equal."""
import numpy as np
import pytest

import scenarios
from ls1amd import PREC_FP32_FP64ACC, PREC_FP64, Context
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu


def check(s, desc=None, cell_mode=0):
    desc = s.comp_desc if desc is None else desc
    o = Oracle(s.ncomp, desc, s.mix, s.eps_rf, s.rc, s.rc_lj, s.box, periodic=True,
               cell_mode=cell_mode)
    ref = o.forces(s.r, s.q, s.cid)
    for prec in (PREC_FP64, PREC_FP32_FP64ACC):
        with Context(0) as c:
            c.setup(s.ncomp, desc, s.mix, s.eps_rf, s.box, s.rc, s.rc_lj, True, cell_mode, prec)
            c.upload(s.r, s.v, s.q, s.L, s.cid)
            c.set_counting(True)
            out = c.forces()
            cnt = c.counters()
            kc = c.kernel_stats()[1]
        np.testing.assert_array_equal(cnt[1:], ref["counters"][1:])
        np.testing.assert_array_equal(kc.sum(0) // 2, cnt)
        for key in ("F", "M", "Vi"):
            top = np.abs(ref[key]).max()
            if top == 0:
                assert np.abs(out[key]).max() == 0
            elif prec == PREC_FP64:
                assert np.abs(out[key] - ref[key]).max() < 1e-12 * top, key
            else:
                e = np.sqrt(((out[key] - ref[key]) ** 2).sum() / (ref[key] ** 2).sum())
                assert e < 1e-5, (key, e)


@pytest.mark.parametrize("n,rho", [(90, 0.5), (300, 0.6), (700, 0.6), (500, 0.05), (1200, 0.85)])
def test_one_centre_boxes(n, rho):
    print("one centre", n, rho, flush=True)
    check(scenarios.ljts_box(n, rho, 1.0, seed=n))


@pytest.mark.parametrize("n", [150, 301, 800, 2500])
def test_all_site_types(n):
    print("all sites", n, flush=True)
    check(scenarios.small_mixture(n=n, seed=n))


@pytest.mark.parametrize("box", [(3.1, 6.3, 9.4), (12.5, 7.5, 3.1), (15.1, 12.6, 10.2)])
def test_rebuild_geometry(box):
    """cell_mode 1: one cell in a dimension is its own neighbour."""
    print("rebuild", box, flush=True)
    s = scenarios.small_mixture(n=120, seed=8)
    s.box = np.array(box)
    rng = np.random.default_rng(5)
    k = [int(b // 1.2) for b in box]
    g = np.stack(np.meshgrid(*[np.arange(x) for x in k], indexing="ij"), -1).reshape(-1, 3)
    r = (g + 0.5) * (s.box / np.array(k)) + rng.normal(scale=0.03, size=g.shape)
    keep = np.sort(rng.permutation(len(r))[:min(len(r), 400)])
    s.r = np.mod(r[keep], s.box)
    n = len(s.r)
    s.cid = rng.integers(0, s.ncomp, n).astype(np.int32)
    s.q = scenarios.random_quaternions(rng, n)
    s.v, s.L = np.zeros((n, 3)), np.zeros((n, 3))
    s.rc = s.rc_lj = 3.0
    check(s, cell_mode=1)


@pytest.mark.parametrize("ids", [3, 9])
def test_several_lj_ids(ids):
    """Two LJ sites per molecule, `ids` components (2 ids each): the LDS table
    (6 ids) and the global one (18 ids); also 1500 molecules in large cells:
    several passes and full hit lists per cell."""
    print("lj ids", 2 * ids, flush=True)
    parts = []
    for k in range(ids):
        d = 0.2 + 0.01 * k
        parts += [2, 0, 0, 0, 0, 0, d, 0.5, 1.0 + 0.02 * k, 0.8, 4.0, 0.0,
                  0, 0, -d, 0.5, 0.9, 0.85, 4.0, 0.0, 0, 0, 0]
    s = scenarios.small_mixture(n=1500, rho=0.55, rc=4.0, seed=ids, with_dipoles=False)
    rng = np.random.default_rng(ids)
    s.ncomp, s.comp_desc = ids, np.array(parts, np.float64)
    s.mix = np.tile([1.0, 1.0], (ids * (ids - 1) // 2, 1))
    s.cid = rng.integers(0, ids, s.n).astype(np.int32)
    check(s)


@pytest.mark.parametrize("n,cells", [(9000, 10), (11500, 11)])
def test_multisite_boxes_beyond_the_line(n, cells):
    """More than 512 cells."""
    print("cell kernels", n, flush=True)
    s = scenarios.mixture(n=n, rho=0.3, seed=6)
    assert int(s.box[0] // s.rc) == cells
    check(s)


def test_batch_of_small_and_large_boxes():
    """Replicas on both sides of the line in one batch, each as it is alone."""
    reps = [scenarios.mixture(n=n, rho=0.3, seed=n) for n in (9000, 700, 11500, 301)]
    for prec in (PREC_FP64, PREC_FP32_FP64ACC):
        with Context(0) as c:
            c.setup_replicas(reps, precision=prec)
            c.update_container()
            c.traverse()
            d = c.download()
        at = 0
        for s in reps:
            with Context(0) as c:
                c.setup_system(s, precision=prec)
                c.update_container()
                c.traverse()
                alone = c.download()
            for key in ("F", "M", "Vi"):
                np.testing.assert_array_equal(d[key][at:at + s.n], alone[key])
            at += s.n


def test_coincident_molecules_are_left_out():
    """Two molecules at the same place (distance 0) do not interact, as in
    SingleCellPolicy_. Their sums hold the same terms: in FP64 equal to rounding,
    in FP32 (partners summed in another order) within the FP32 bar."""
    print("coincident", flush=True)
    s = scenarios.ljts_box(200, 0.5, 1.0, seed=3)
    s.r = np.vstack([s.r, s.r[17:19]])
    n = len(s.r)
    s.v, s.L, s.q = np.zeros((n, 3)), np.zeros((n, 3)), np.tile([1.0, 0, 0, 0], (n, 1))
    s.cid = np.zeros(n, np.int32)
    out = {}
    for prec in (PREC_FP64, PREC_FP32_FP64ACC):
        with Context(0) as c:
            c.setup_system(s, precision=prec)
            out[prec] = c.forces()["F"]
        assert np.isfinite(out[prec]).all()
        top = np.abs(out[prec]).max()
        bar = 1e-12 if prec == PREC_FP64 else 1e-5
        assert np.abs(out[prec][200:] - out[prec][17:19]).max() < bar * top
