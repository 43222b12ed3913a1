"""Which boxes run the block pair kernels (four waves per cell): at most 512 cells
and, on average, at least 20 sites per cell and site type present, multi-site
molecules (cells larger than 1.5 rc^3 count by volume), or 15 sites of each type
and 13 molecules per rc^3. Every case says on which
side of the rule its box lies, so that none moves to the other kernel unseen:
dense boxes against the oracle where the block kernels' split can go wrong, and
sparse and one-centre ones, which lost time to them, for the time of a batch.

Bars as in test_gpu_parity.py: FP64 form 1e-12 relative to the largest value, FP32
form relative RMS force error 1e-5, in-cutoff pair counts equal."""
import numpy as np
import pytest

import scenarios
from ls1amd import PREC_FP32_FP64ACC, PREC_FP64, Context
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu


def cells(s):
    return np.floor(s.box / s.rc).astype(int)


def blocks(s):
    """The rule."""
    comps = scenarios.parse_components(s.comp_desc)
    n = [sum(len(comps[k][t]) * int((s.cid == k).sum()) for k in range(s.ncomp))
         for t in ("lj", "ch", "dp", "qp")]
    if all(len(c["lj"]) == 1 and not c["ch"] + c["dp"] + c["qp"]
           and not np.any(c["lj"][0][:3]) for c in comps):
        return False
    ncell = int(np.prod(cells(s)))
    if ncell > 512:
        return False
    volume, types = np.prod(s.box) / s.rc**3, sum(x > 0 for x in n)
    return (sum(n) >= 20 * types * max(ncell, volume / 1.5)
            or sum(n) >= 15 * types * volume and s.n >= 13 * volume)


def check(s, periodic=True, cell_mode=0):
    o = Oracle(s.ncomp, s.comp_desc, s.mix, s.eps_rf, s.rc, s.rc_lj, s.box, periodic=periodic,
               cell_mode=cell_mode)
    ref = o.forces(s.r, s.q, s.cid)
    for prec in (PREC_FP64, PREC_FP32_FP64ACC):
        with Context(0) as c:
            c.setup(s.ncomp, s.comp_desc, s.mix, s.eps_rf, s.box, s.rc, s.rc_lj, periodic,
                    cell_mode, prec)
            c.upload(s.r, s.v, s.q, s.L, s.cid)
            c.set_counting(True)
            out = c.forces()
            cnt, kc = c.counters(), c.kernel_stats()[1]
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


def dipolar(n, rho, seed, rc=3.0):
    """LJ site at the molecule's centre, a charge and a dipole beside it."""
    s = scenarios.mixture(n=n, rho=rho, seed=seed, rc=rc)
    s.ncomp, s.mix, s.eps_rf = 1, np.zeros((0, 2)), 5.0
    s.comp_desc = np.array([1, 1, 1, 0, 0, 0, 0, 1, 1, 1, rc, 1, 0, 0, -.1, 0, .3,
                            0, 0, .1, 0, 0, 1, 1.2, .02, .02, .01], np.float64)
    s.cid[:] = 0
    return s


def two_sites(ids, n, seed):
    """Two LJ sites per molecule, `ids` components of two LJ ids each."""
    s = scenarios.mixture(n=n, rho=0.8, seed=seed)
    parts = []
    for k in range(ids):
        d = 0.2 + 0.01 * k
        parts += [2, 0, 0, 0, 0, 0, d, 0.5, 1.0 + 0.02 * k, 0.8, 3.0, 0.0,
                  0, 0, -d, 0.5, 0.9, 0.85, 3.0, 0.0, 0, 0, 0]
    s.ncomp, s.comp_desc = ids, np.array(parts, np.float64)
    s.mix = np.tile([1.0, 1.0], (ids * (ids - 1) // 2, 1))
    s.cid = np.random.default_rng(seed).integers(0, ids, n).astype(np.int32)
    return s


def all_types(n, rho, seed, rc=3.0):
    s = scenarios.mixture(n=n, rho=rho, seed=seed, rc=rc)
    t = scenarios.small_mixture(n=150, rc=rc)
    s.ncomp, s.comp_desc, s.mix, s.eps_rf = t.ncomp, t.comp_desc, t.mix, t.eps_rf
    s.cid = np.random.default_rng(seed).integers(0, t.ncomp, n).astype(np.int32)
    return s


def crowd(s, corner, share, seed):
    """Some molecules of the whole box moved to `corner` of it: a dense cell beside
    thin and empty ones (sites that overlap are set apart by a small lattice)."""
    rng = np.random.default_rng(seed)
    k = np.sort(rng.permutation(s.n)[: int(share * s.n)])
    m = int(np.ceil(len(k) ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[: len(k)]
    s.r[k] = (g + 0.5) * (s.rc * corner / m)
    return s


@pytest.mark.parametrize("n,rho", [(500, .5), (1500, .5), (4000, .5), (9001, .5), (1777, .9),
                                   (3468, .5), (499, .49), (7000, .49)])
def test_mixture(n, rho):
    print("mixture", n, rho, flush=True)
    s = scenarios.mixture(n=n, rho=rho, seed=n)
    assert blocks(s)
    check(s)


@pytest.mark.parametrize("n", [800, 1301, 3001])
def test_all_site_types(n):
    print("all sites", n, flush=True)
    s = all_types(n, 0.9, n)
    assert blocks(s)
    check(s)


@pytest.mark.parametrize("ids", [1, 3, 9])
def test_lj_tables(ids):
    """One table entry, the LDS table (6 ids) and the global one (18)."""
    print("lj ids", 2 * ids, flush=True)
    s = two_sites(ids, 1100, seed=ids)
    assert blocks(s)
    check(s)


@pytest.mark.parametrize("n,rho", [(620, .8), (2000, .9)])
def test_lj_site_at_the_centre(n, rho):
    print("dipolar", n, rho, flush=True)
    s = dipolar(n, rho, n)
    assert blocks(s)
    check(s)


@pytest.mark.parametrize("share", [0.15, 0.4])
def test_a_dense_cell_beside_empty_ones(share):
    """A cell of more than 64 LJ sites, several passes of a wave over one staged
    neighbourhood (at most 672 sites, which a tile holds), idle waves elsewhere."""
    print("crowd", share, flush=True)
    s = crowd(dipolar(640, 0.75, 5), 0.9, share, 6)
    assert blocks(s) and int(np.prod(cells(s))) == 27
    idx = np.floor(s.r / (s.box / cells(s))).astype(int)
    per = np.bincount(idx @ np.array([9, 3, 1]), minlength=27)
    assert per.max() > 64 and s.n <= 672
    if share > 0.3:
        assert per.min() < 20
    check(s)


def test_open_boundaries():
    s = all_types(1500, 0.9, 3)
    s.r = 0.05 + s.r * (s.box - 0.1) / s.box
    assert blocks(s)
    check(s, periodic=False)


@pytest.mark.parametrize("box", [(3.1, 6.3, 9.4), (12.5, 7.5, 3.1)])
def test_one_cell_in_a_dimension(box):
    """cell_mode 1: a cell is its own neighbour."""
    print("box", box, flush=True)
    s = all_types(1200, 0.9, 8)
    s.box = np.array(box)
    rng = np.random.default_rng(5)
    k = [int(b // 0.8) for b in box]
    g = np.stack(np.meshgrid(*[np.arange(x) for x in k], indexing="ij"), -1).reshape(-1, 3)
    r = (g + 0.5) * (s.box / np.array(k)) + rng.normal(scale=0.02, size=g.shape)
    s.r = np.mod(r[np.sort(rng.permutation(len(r))[:1200])], s.box)
    n = len(s.r)
    s.cid, s.q = rng.integers(0, s.ncomp, n).astype(np.int32), scenarios.random_quaternions(rng, n)
    s.v, s.L = np.zeros((n, 3)), np.zeros((n, 3))
    assert blocks(s)
    check(s, cell_mode=1)


def test_coincident_molecules():
    """Two molecules at one place do not interact (SingleCellPolicy_): their sums
    hold the same terms."""
    s = scenarios.mixture(n=500, rho=0.6, seed=3)
    for key in ("r", "q", "cid", "v", "L"):
        a = getattr(s, key)
        setattr(s, key, np.concatenate([a, a[17:19]]))
    assert blocks(s)
    for prec, bar in ((PREC_FP64, 1e-12), (PREC_FP32_FP64ACC, 1e-5)):
        with Context(0) as c:
            c.setup_system(s, precision=prec)
            F = c.forces()["F"]
        assert np.isfinite(F).all()
        assert np.abs(F[500:] - F[17:19]).max() < bar * np.abs(F).max()


def test_batch_on_both_sides():
    """Small dense boxes between others in one batch, each as it is alone; then the
    same context with a state in which other boxes are dense."""
    dense = [scenarios.mixture(n=n, rho=.5, seed=n) for n in (500, 4000)]
    thin = [scenarios.mixture(n=n, rho=.3, seed=n) for n in (700, 9000)]
    assert all(map(blocks, dense)) and not any(map(blocks, thin))
    for prec in (PREC_FP64, PREC_FP32_FP64ACC):
        reps = [thin[1], dense[0], thin[0], dense[1]]
        with Context(0) as c:
            c.setup_replicas(reps, precision=prec)
            for water in (False, True):
                at = 0
                cid = np.concatenate([np.ones_like(s.cid) if water else s.cid for s in reps])
                c.upload(*(np.concatenate([getattr(s, k) for s in reps]) for k in "rvqL"), cid)
                c.update_container()
                c.traverse()
                d = c.download()
                for s in reps:
                    one = scenarios.dataclasses.replace(s, cid=np.ones_like(s.cid) if water else s.cid)
                    with Context(0) as b:
                        b.setup_system(one, precision=prec)
                        b.update_container()
                        b.traverse()
                        alone = b.download()
                    for key in ("F", "M", "Vi"):
                        np.testing.assert_array_equal(d[key][at:at + s.n], alone[key])
                    at += s.n


def pair_ms(setup):
    with Context(0) as c:
        setup(c)
        c.update_container()
        c.traverse()
        c.set_timing(True)
        t = []
        for _ in range(15):
            c.traverse()
            t.append(c.kernel_stats()[0].sum())
        return float(np.median(t))


@pytest.mark.parametrize("kind", ["one-centre", "one-centre-thin", "all-sites"])
@pytest.mark.parametrize("prec", [PREC_FP64, PREC_FP32_FP64ACC])
def test_a_batch_of_small_boxes_costs_what_one_large_box_does(kind, prec):
    """Per molecule, at the same density: within half as much again (the block
    kernels took 1.6 to 2.5 times here). Cell edges of both boxes are close to rc."""
    # f^3 boxes of k^3 cells, against a box f times as large
    k, f, rho = {"one-centre": (4, 8, .6), "one-centre-thin": (3, 10, .08),
                 "all-sites": (4, 5, .3)}[kind]
    rc = 2.5

    def make(n, edge, seed):
        if kind == "all-sites":
            return scenarios.small_mixture(n=n, rho=n / edge**3, rc=rc, seed=seed)
        return scenarios.ljts_box(n, n / edge**3, 1.0, rc, seed=seed)

    edge = k * rc * 1.005
    n = int(rho * edge**3)
    one, large = make(n, edge, 3), make(n * f**3, edge * f, 4)
    assert not blocks(one) and not blocks(large)
    few = pair_ms(lambda c: c.setup_replicas([one] * f**3, precision=prec))
    big = pair_ms(lambda c: c.setup_system(large, precision=prec))
    ratio = few / big
    print(kind, "batch / large box per molecule: %.2f" % ratio, flush=True)
    assert ratio < 1.5
