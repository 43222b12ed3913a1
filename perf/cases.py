"""Performance cases of the force path, through the Python entry points.

A user of this framework does four things with it, and every case is one of
them:

* ``steps``    a block of Leapfrog steps of one periodic system (or of a batch
               of replicas), then the state for a frame or a checkpoint;
* ``forces``   one force evaluation of a state in hand: re-bin, traversal,
               molecule forces, torques and virials back on the host;
* ``adjoint``  the derivatives of an LJ mixture with respect to its pair
               parameters, with or without the force vector-Jacobian product;
* ``fit``      one gradient step of a force-field fit through the autograd
               bridge (forward and backward).

Systems, densities and cutoffs are those of ``scenarios.py`` (the benchmark's
and the tests' workloads). Both precision forms appear; the frames of the
FP32-pair form are kept in single precision, which is what its pair
arithmetic carries, those of the FP64 form in double.
"""
import math
import pathlib
import sys

import numpy as np
import torch

sys.path.insert(0, str(pathlib.Path(__file__).resolve().parents[1] / "ls1-mardyn_amd"))

import ls1amd_torch  # noqa: E402
import scenarios  # noqa: E402
from ls1amd import PREC_FP32_FP64ACC, PREC_FP64, Context  # noqa: E402


def listed():
    return [
        # a small fluid box (teaching runs, unit checks, one of many state
        # points): a few cells per dimension, launches and latency count
        dict(name="steps_lj_500", kind="steps", system="lj", n=500, fp32=False, steps=50, mode="nve"),
        # the 32,000-molecule FCC LJ fluid in the FP64 form: the ordinary size
        dict(name="steps_lj_32k", kind="steps", system="lj", n=32000, fp32=False, steps=50,
             mode="nve"),
        # the multi-site mixture in an equilibration run with the thermostat;
        # an odd molecule count
        dict(name="steps_mixture_9k_nvt", kind="steps", system="mixture", n=9001, fp32=True,
             steps=20, mode="nvt"),
        # the headline: the multi-site mixture of the benchmark, 1 M molecules
        dict(name="steps_mixture_1m", kind="steps", system="mixture", n=1000000, fp32=True,
             steps=20, mode="nve"),
        # the same mixture in the FP64 form at a mid size, ragged count
        dict(name="steps_mixture_150k_f64", kind="steps", system="mixture", n=149993, fp32=False,
             steps=20, mode="nve"),
        # a vapour-liquid interface: dense cells beside nearly empty ones
        dict(name="steps_slab_1m", kind="steps", system="slab", n=990906, fp32=True, steps=25,
             mode="nve"),
        # the reduced-memory one-centre mode on a smaller interface, FP64
        dict(name="steps_slab_100k_rmm", kind="steps", system="slab", n=101463, fp32=False,
             steps=50, mode="rmm"),
        # a state-point sweep: independent systems stepped as one batch
        dict(name="steps_replicas_64", kind="steps", system="replicas", n=64, fp32=True, steps=25,
             mode="nve"),
        # one force call on every site kind (LJ, charge, dipole, quadrupole)
        dict(name="forces_allsites_3k", kind="forces", system="allsites", n=3001, fp32=False),
        # one force call on the mixture, as an external integrator makes it
        dict(name="forces_mixture_100k", kind="forces", system="mixture", n=100003, fp32=True),
        # differentiation of the binary LJ mixture with the force VJP
        dict(name="adjoint_binary_500k", kind="adjoint", system="binary", n=500000, fp32=False,
             vjp=True),
        # a force-field fit: one gradient step on the parameters of a charged mixture
        dict(name="fit_charged_4k", kind="fit", system="charged", n=4001, fp32=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["steps", "steps", "steps", "steps", "forces", "forces", "adjoint", "fit"])
    fp32 = rng.random() < 0.5
    if kind == "forces":
        system = rng.choice(["mixture", "allsites", "lj", "slab", "binary"])
        hi = 20000 if system == "allsites" else 300000
        return dict(kind=kind, system=system, n=_log_int(rng, 500, hi), fp32=fp32)
    if kind == "adjoint":
        return dict(kind=kind, system="binary", n=_log_int(rng, 2000, 500000), fp32=False,
                    vjp=rng.random() < 0.7)
    if kind == "fit":
        return dict(kind=kind, system="charged", n=_log_int(rng, 500, 20000), fp32=False)
    system = rng.choice(["lj", "mixture", "mixture", "slab", "replicas"])
    steps = rng.choice([10, 15, 20, 25])
    if system == "replicas":
        return dict(kind=kind, system=system, n=_log_int(rng, 4, 64), fp32=fp32, steps=steps,
                    mode=rng.choice(["nve", "nvt"]))
    modes = ["nve", "nve", "nvt"] + (["rmm"] if system != "mixture" else [])
    hi = {"lj": 500000, "mixture": 300000, "slab": 900000}[system]
    return dict(kind=kind, system=system, n=_log_int(rng, 500, hi), fp32=fp32, steps=steps,
                mode=rng.choice(modes))


# ------------------------------------------------------------------ inputs

def _charged(n, seed):
    """Water-like molecules (LJ oxygen, three charges) and one-centre LJ
    molecules, half and half: the site kinds the adjoint covers."""
    rng = np.random.default_rng(seed)
    k = int(math.ceil((n / 4.0) ** (1.0 / 3.0) - 1e-9))
    edge = (n / 0.4) ** (1.0 / 3.0)
    r = scenarios.fcc_lattice(k, edge / k)
    r = r[np.sort(rng.permutation(len(r))[:n])]
    r = np.mod(r + rng.normal(scale=0.02, size=r.shape), edge)
    r = np.minimum(r, np.nextafter(edge, 0.0))
    desc = np.array(scenarios.comp_water(2.5) + scenarios.comp_1clj(0.9, 1.05, 1.0, 2.5), np.float64)
    cid = np.zeros(n, np.int32)
    cid[rng.permutation(n)[: n // 2]] = 1
    q = scenarios.random_quaternions(rng, n)
    z = np.zeros((n, 3))
    return scenarios.System("charged", 2, desc, np.array([[0.98, 1.01]]), 1.0, 2.5, 2.5,
                            np.full(3, edge), r, z, q, z.copy(), cid, 1.0)


def _systems(case, seed):
    """The System records of a case (one, or one per replica)."""
    system, n = case["system"], int(case["n"])
    if system == "lj":
        k = int(math.ceil((n / 4.0) ** (1.0 / 3.0) - 1e-9))
        s = scenarios.lj_fcc(ncell=k, seed=seed)
        rng = np.random.default_rng(seed + 1)
        keep = np.sort(rng.permutation(s.n)[:n])
        r = np.mod(s.r[keep] + rng.normal(scale=0.05, size=(n, 3)), s.box)
        s.r = np.minimum(r, np.nextafter(s.box, 0.0))
        s.v, s.q, s.L, s.cid = s.v[keep], s.q[keep], s.L[keep], s.cid[keep]
        return [s]
    if system == "mixture":
        return [scenarios.mixture(n=n, seed=seed)]
    if system == "allsites":
        return [scenarios.small_mixture(n=n, seed=seed)]
    if system == "binary":
        return [scenarios.binary_lj(n=n, seed=seed)]
    if system == "charged":
        return [_charged(n, seed)]
    if system == "slab":
        # 3,962,880 molecules at scale 1; at least two cells per dimension
        return [scenarios.ljts_slab(scale=max((n / 3962880.0) ** (1.0 / 3.0), 0.04), seed=seed)]
    if system == "replicas":
        # the state points of the sweep (sizes, densities, temperatures) are
        # the benchmark's ranges, the same for every seed; positions are not
        rng = np.random.default_rng(1000 + n)
        ns = np.exp(rng.uniform(np.log(2000), np.log(40000), n)).astype(np.int64)
        rhos, ts = rng.uniform(0.05, 0.85, n), rng.uniform(0.7, 1.3, n)
        return [scenarios.ljts_box(int(ns[k]), float(rhos[k]), float(ts[k]), seed=10 * seed + k,
                                   name="replica%d" % k) for k in range(n)]
    raise ValueError(system)


def prepare(case, seed):
    seed = int(seed) % 1000003
    sys_ = _systems(case, seed)
    s = sys_[0]
    st = dict(case=case)
    if case["kind"] == "fit":
        eng = ls1amd_torch.ForceFieldEngine(s)
        st["engine"] = eng
        st["eps"] = torch.tensor(eng.eps0, dtype=torch.float64, requires_grad=True)
        st["sig"] = torch.tensor(eng.sig0, dtype=torch.float64, requires_grad=True)
        st["q"] = torch.tensor(eng.q0, dtype=torch.float64, requires_grad=True)
        st["r"] = torch.tensor(s.r, dtype=torch.float64)
        return st
    prec = PREC_FP32_FP64ACC if case["fp32"] else PREC_FP64
    ctx = Context(0)
    st["ctx"] = ctx
    if case["system"] == "replicas":
        ctx.setup_replicas(sys_, periodic=True, precision=prec)
    else:
        ctx.setup_system(s, periodic=True, precision=prec)
    st["dt"] = s.dt
    if case["kind"] == "adjoint":
        if case["vjp"]:
            st["cot"] = np.random.default_rng(seed + 7).normal(size=(s.n, 3))
        ctx.update_container()
        ctx.adjoint(st.get("cot"))
    if case["kind"] == "steps":
        if case["mode"] == "nvt":
            ctx.set_thermostat(np.array([x.temperature for x in sys_]), explosion_heuristics=False)
        ctx.update_container()
        ctx.traverse()
        if case["mode"] == "rmm":
            ctx.set_rmm(s.dt)
    return st


# -------------------------------------------------------------------- runs

def _frame(case, d, keys):
    out = {k: torch.from_numpy(d[k]) for k in keys}
    if case["fp32"]:
        out = {k: v.to(torch.float32) for k, v in out.items()}
    return out


def _records(case, x):
    t = torch.from_numpy(np.ascontiguousarray(x))
    return t.to(torch.float32) if case["fp32"] else t


def run(state):
    case = state["case"]
    rotates = case["system"] in ("mixture", "allsites")
    if case["kind"] == "steps":
        per = state["ctx"].step(case["steps"], state["dt"], use_graph=True)
        d = state["ctx"].download()
        keys = ["r", "v"] + ([] if case["mode"] == "rmm" else ["F"]) + (["q", "L", "M"] if rotates else [])
        return dict(_frame(case, d, keys), records=_records(case, per))
    if case["kind"] == "forces":
        d = state["ctx"].forces()
        return dict(_frame(case, d, ["F", "Vi"] + (["M"] if rotates else [])),
                    macro=_records(case, d["macro"]))
    if case["kind"] == "adjoint":
        return state["ctx"].adjoint(state.get("cot"))
    # one gradient step of a fit: loss, gradients, updated parameters
    eps, sig, q = state["eps"], state["sig"], state["q"]
    U, W, F = ls1amd_torch.force_field(eps, sig, q, state["r"], state["engine"])
    n = F.shape[0]
    loss = U / n + 0.1 * W / n
    g = torch.autograd.grad(loss, (eps, sig, q))
    with torch.no_grad():
        for k, x in zip(("eps", "sig", "q"), g):
            state[k] = (state[k] - 1e-6 * x).requires_grad_(True)
    return dict(loss=loss.detach(), F=F, g_eps=g[0], g_sig=g[1], g_q=g[2],
                eps=state["eps"].detach(), sig=state["sig"].detach(), q=state["q"].detach())


# -------------------------------------------------------------------- work

#: per molecule: site-pair flops (ls1's FlopCounter convention) at the system's
#: density, plus 8 per molecule pair inside the cutoff; neighbours rho 4/3 pi rc^3
_LJ1 = 41 + 8


def work(case):
    n, system = float(case["n"]), case["system"]
    if system == "replicas":
        n *= 12300.0  # log-uniform in [2,000, 40,000]
    nb = {"lj": 0.6 * 65.45, "slab": 0.6 * 65.45, "replicas": 0.45 * 65.45, "binary": 0.7 * 65.45,
          "mixture": 0.5 * 113.1, "allsites": 0.3 * 65.45, "charged": 0.4 * 65.45}[system]
    per_pair = {"lj": _LJ1, "slab": _LJ1, "replicas": _LJ1, "binary": _LJ1,
                # 2CLJQ / water, half and half: 9/4 LJ, 9/4 C-C, 3/2 C-Q, 1/4 Q-Q
                "mixture": 8 + 2.25 * 41 + 2.25 * 34 + 1.5 * 79 + 0.25 * 161,
                # a third each of 2CLJQ, water and LJ + charge + dipole
                "allsites": 8 + 1.78 * 41 + 1.78 * 34 + 0.89 * 62 + 0.11 * 135 + 0.89 * 79
                + 0.22 * 151 + 0.11 * 161,
                "charged": 8 + 41 + 2.25 * 34}[system]
    rot = system in ("mixture", "allsites", "charged")
    state = 8.0 * (13 if rot else 6)
    out = 8.0 * (9 if rot else 6)
    flops = 0.5 * n * nb * per_pair
    if case["kind"] == "steps":
        return dict(bytes=n * (2 * state + out), flops=flops * case["steps"])
    if case["kind"] == "forces":
        return dict(bytes=n * (state + out), flops=flops)
    if case["kind"] == "adjoint":
        return dict(bytes=n * (24 + (48 if case["vjp"] else 0)), flops=flops * (3 if case["vjp"] else 2))
    return dict(bytes=n * (state + out), flops=flops * 2)


# ------------------------------------------------------------------- exact
# The same quantities in plain torch, 64 bits: molecule pairs below the cutoff
# from padded cells, site energies, and autograd for forces, torques and
# parameter derivatives.

_DEV = "cuda" if torch.cuda.is_available() else "cpu"
_T64 = dict(dtype=torch.float64, device=_DEV)


def _pairs(r, box, rc):
    """(i, j, shift): every unordered pair of molecules closer than rc."""
    nc = np.maximum(np.floor(box / rc).astype(int), 1)
    if nc.min() < 3:  # too few cells: all pairs, nearest images
        i, j = torch.triu_indices(len(r), len(r), 1, device=_DEV)
        d = r[i] - r[j]
        b = torch.tensor(box, **_T64)
        sh = torch.round(d / b) * b
        m = ((d - sh) ** 2).sum(1) < rc * rc
        return i[m], j[m], sh[m]
    b, nt = torch.tensor(box, **_T64), torch.tensor(nc, device=_DEV)
    c3 = torch.minimum((r / b * nt).long(), nt - 1)
    c = (c3[:, 2] * nc[1] + c3[:, 1]) * nc[0] + c3[:, 0]
    order = torch.argsort(c, stable=True)
    cnt = torch.bincount(c, minlength=int(nc.prod()))
    width = int(cnt.max())
    start = torch.cumsum(cnt, 0) - cnt
    slot = torch.arange(len(r), device=_DEV) - start[c[order]]
    table = torch.full((len(cnt), width), -1, dtype=torch.long, device=_DEV)
    table[c[order], slot] = order
    cells = torch.arange(len(cnt), device=_DEV)
    xyz = torch.stack([cells % nc[0], cells // nc[0] % nc[1], cells // (nc[0] * nc[1])], 1)
    got = []
    for o in range(14):  # the cell itself and half of its neighbours
        off = torch.tensor([o % 3 - 1, o // 3 % 3 - 1, o // 9 - 1], device=_DEV)
        x = xyz + off
        sh = torch.where(x < 0, -b, torch.where(x >= nt, b, torch.zeros_like(b)))
        x = x % nt
        other = (x[:, 2] * nc[1] + x[:, 1]) * nc[0] + x[:, 0]
        own, oth = torch.nonzero(table >= 0, as_tuple=True), None
        i = table[own]
        for t in range(width):
            j = table[other[own[0]], t]
            ok = j >= 0
            if o == 13:
                ok = ok & (j > i)
            a, jj, s = i[ok], j[ok], sh[own[0][ok]]
            d2 = ((r[a] - r[jj] - s) ** 2).sum(1)
            m = d2 < rc * rc
            got.append((a[m], jj[m], s[m]))
    return tuple(torch.cat([g[k] for g in got]) for k in range(3))


def _rotate(q, d):
    w, u = q[..., :1], q[..., 1:]
    c = torch.cross(u, d, dim=-1)
    return d + 2 * (w * c + torch.cross(u, c, dim=-1))


class _Model:
    """Component records as tensors: sites per kind, masses, moments."""

    def __init__(self, s):
        self.s, self.comps = s, []
        p, desc = 0, [float(x) for x in s.comp_desc]
        for _ in range(s.ncomp):
            cnt = [int(x) for x in desc[p:p + 4]]
            p += 4
            rec = []
            for width, k in zip((8, 5, 7, 7), cnt):
                rec.append([desc[p + width * a:p + width * a + width] for a in range(k)])
                p += width * k
            mass = sum(x[3] for x in rec[0] + rec[1])
            inert = [sum(x[3] * (x[a] ** 2 + x[b] ** 2) for x in rec[0] + rec[1])
                     for a, b in ((1, 2), (0, 2), (0, 1))]
            rot = sum(v != 0 for v in inert)
            inert = [desc[p + d] if desc[p + d] > 0 else inert[d] for d in range(3)]
            p += 3
            self.comps.append(dict(lj=rec[0], c=rec[1], d=rec[2], q=rec[3], mass=mass,
                                   inertia=inert, rotdof=rot))
        self.cid = torch.tensor(s.cid, dtype=torch.long, device=_DEV)
        self.mass = torch.tensor([c["mass"] for c in self.comps], **_T64)[self.cid][:, None]
        self.inertia = torch.tensor([c["inertia"] for c in self.comps], **_T64)[self.cid]
        self.inv = torch.where(self.inertia != 0, 1 / torch.where(self.inertia != 0, self.inertia, 1.0),
                               torch.zeros_like(self.inertia))
        self.rotdof = float(sum(c["rotdof"] * int((self.cid == k).sum())
                                for k, c in enumerate(self.comps)))
        rc = s.rc
        self.rf = 2 * (s.eps_rf - 1) / (rc ** 3 * (2 * s.eps_rf + 1))

    def lj_pair(self, a, sa, b, sb):
        """(24 eps, sigma^2, shift6) of LJ sites sa of component a, sb of b."""
        x, y = self.comps[a]["lj"][sa], self.comps[b]["lj"][sb]
        if a == b:
            eps, sig = math.sqrt(x[4] * y[4]), 0.5 * (x[5] + y[5])
            sh = 0.0
            for z in (x, y):  # each side carries its own site's shift
                if z[7] != 0:
                    s6 = (z[5] / z[6]) ** 6
                    sh += 0.5 * 24 * z[4] * (s6 - s6 * s6)
            return 24 * eps, sig * sig, sh
        lo, hi = min(a, b), max(a, b)
        k = sum(self.s.ncomp - 1 - t for t in range(lo)) + hi - lo - 1
        xi, eta = (self.s.mix[k] if len(self.s.mix) else (1.0, 1.0))
        eps, sig = xi * math.sqrt(x[4] * y[4]), 0.5 * eta * (x[5] + y[5])
        s6 = (sig / self.s.rc_lj) ** 6
        return 24 * eps, sig * sig, 24 * eps * (s6 - s6 * s6)

    def forces(self, r, q):
        """F, M, Vi, macro of the state (molecule positions, unit quaternions)."""
        n = len(r)
        i, j, sh = _pairs(r, np.asarray(self.s.box), self.s.rc)
        F, Vi = torch.zeros(n, 3, **_T64), torch.zeros(n, 3, **_T64)
        M = torch.zeros(n, 3, **_T64)
        u6 = torch.zeros((), **_T64)
        ux, rf, vir = u6.clone(), u6.clone(), u6.clone()
        # site offsets and axes of every molecule, one leaf tensor per site
        leaf = {}
        for k, c in enumerate(self.comps):
            for kind in ("lj", "c", "d", "q"):
                for t, x in enumerate(c[kind]):
                    leaf[k, kind, t] = _rotate(q, torch.tensor(x[:3], **_T64).expand(n, 3).contiguous())
                    leaf[k, kind, t].requires_grad_(True)
                    if kind in "dq":
                        leaf[k, kind, t, "e"] = _rotate(q, torch.tensor(x[3:6], **_T64).expand(n, 3).contiguous())
                        leaf[k, kind, t, "e"].requires_grad_(True)
        chunk = 2_000_000
        grads = {k: torch.zeros(n, 3, **_T64) for k in leaf}
        for a in range(self.s.ncomp):
            for b in range(self.s.ncomp):
                sel = torch.nonzero((self.cid[i] == a) & (self.cid[j] == b))[:, 0]
                for lo in range(0, len(sel), chunk):
                    m = sel[lo:lo + chunk]
                    dm = (r[i[m]] - r[j[m]] - sh[m]).requires_grad_(True)
                    e6, ex, er = self._energy(a, b, leaf, i[m], j[m], dm)
                    used = [k for k in leaf if k[0] in (a, b)]
                    g = torch.autograd.grad((e6 / 6 + ex + er), [dm] + [leaf[k] for k in used],
                                            allow_unused=True)
                    f = -g[0]
                    F.index_add_(0, i[m], f)
                    F.index_add_(0, j[m], -f)
                    v = 0.5 * dm.detach() * f
                    Vi.index_add_(0, i[m], v)
                    Vi.index_add_(0, j[m], v)
                    vir = vir + 2 * v.sum()
                    u6, ux, rf = u6 + e6.detach(), ux + ex.detach(), rf + er.detach()
                    for k, x in zip(used, g[1:]):
                        if x is not None:
                            grads[k] += x
        for k, x in grads.items():
            M -= torch.cross(leaf[k].detach(), x, dim=1)
        return F, M, Vi, torch.stack([u6, ux, vir, rf])

    def _energy(self, a, b, leaf, i, j, dm):
        z = dm.sum() * 0
        e6, ex, er = z, z, z
        ca, cb = self.comps[a], self.comps[b]

        def site(k, kind, t, at):
            return leaf[k, kind, t][at]

        for s in range(len(ca["lj"])):
            for t in range(len(cb["lj"])):
                e24, s2, sh6 = self.lj_pair(a, s, b, t)
                d = dm + site(a, "lj", s, i) - site(b, "lj", t, j)
                l6 = (s2 / (d * d).sum(1)) ** 3
                e6 = e6 + (e24 * (l6 * l6 - l6) + sh6).sum()
        for s, x in enumerate(ca["c"]):
            for t, y in enumerate(cb["c"]):
                d = dm + site(a, "c", s, i) - site(b, "c", t, j)
                ex = ex + (x[4] * y[4] * (d * d).sum(1).rsqrt()).sum()
        # mixed pairs from both sides: (charge, dipole), (charge, quadrupole),
        # (dipole, quadrupole), with d from the second to the first
        for (k1, c1, at1), (k2, c2, at2), sg in (((a, ca, i), (b, cb, j), 1.0), ((b, cb, j), (a, ca, i), -1.0)):
            for s, x in enumerate(c1["c"]):
                for t, y in enumerate(c2["d"]):
                    d = sg * dm + site(k1, "c", s, at1) - site(k2, "d", t, at2)
                    e, r2 = leaf[k2, "d", t, "e"][at2], (d * d).sum(1)
                    ex = ex - (x[4] * y[6] * (d * e).sum(1) * r2 ** -1.5).sum()
                for t, y in enumerate(c2["q"]):
                    d = sg * dm + site(k1, "c", s, at1) - site(k2, "q", t, at2)
                    e, r2 = leaf[k2, "q", t, "e"][at2], (d * d).sum(1)
                    cos2 = (d * e).sum(1) ** 2 / r2
                    ex = ex + (0.5 * x[4] * y[6] * r2 ** -1.5 * (3 * cos2 - 1)).sum()
            for s, x in enumerate(c1["d"]):
                for t, y in enumerate(c2["q"]):
                    d = sg * dm + site(k1, "d", s, at1) - site(k2, "q", t, at2)
                    e1, e2 = leaf[k1, "d", s, "e"][at1], leaf[k2, "q", t, "e"][at2]
                    r2 = (d * d).sum(1)
                    ct1, ct2 = (d * e1).sum(1) * r2.rsqrt(), (d * e2).sum(1) * r2.rsqrt()
                    ex = ex + (1.5 * x[6] * y[6] * r2 ** -2 * (2 * ct2 * (e1 * e2).sum(1)
                                                              - ct1 * (5 * ct2 * ct2 - 1))).sum()
        for s, x in enumerate(ca["d"]):
            for t, y in enumerate(cb["d"]):
                d = dm + site(a, "d", s, i) - site(b, "d", t, j)
                e1, e2 = leaf[a, "d", s, "e"][i], leaf[b, "d", t, "e"][j]
                r2, ee = (d * d).sum(1), (e1 * e2).sum(1)
                ex = ex + (x[6] * y[6] * r2 ** -1.5 * (ee - 3 * (d * e1).sum(1) * (d * e2).sum(1) / r2)).sum()
                er = er - (x[6] * y[6] * self.rf * ee).sum()
        for s, x in enumerate(ca["q"]):
            for t, y in enumerate(cb["q"]):
                d = dm + site(a, "q", s, i) - site(b, "q", t, j)
                e1, e2 = leaf[a, "q", s, "e"][i], leaf[b, "q", t, "e"][j]
                r2 = (d * d).sum(1)
                c1, c2 = (d * e1).sum(1) * r2.rsqrt(), (d * e2).sum(1) * r2.rsqrt()
                term = (e1 * e2).sum(1) - 5 * c1 * c2
                ex = ex + (0.75 * x[6] * y[6] * r2 ** -2.5 * (1 + 2 * term ** 2 - 5 * (c1 ** 2 + c2 ** 2)
                                                              - 15 * (c1 * c2) ** 2)).sum()
        return e6, ex, er


def _unit(q):
    return q / q.norm(dim=1, keepdim=True)


def _conj(q):
    return torch.cat([q[:, :1], -q[:, 1:]], 1)


def _qdot(q, w):
    return 0.5 * torch.cat([-(q[:, 1:] * w).sum(1, keepdim=True),
                            q[:, :1] * w + torch.cross(q[:, 1:], w, dim=1)], 1)


def _exact_steps(case, s):
    m = _Model(s)
    t = lambda x: torch.tensor(np.asarray(x), **_T64)  # noqa: E731
    r, v, q, L, box = t(s.r), t(s.v), _unit(t(s.q)), t(s.L), t(s.box)
    dt = s.dt
    rotates = case["system"] == "mixture"
    F, M, _, _ = m.forces(r, q)
    if case["mode"] == "rmm":
        v = v + 0.5 * dt / m.mass * F
    per = []
    for _ in range(case["steps"]):
        if case["mode"] != "rmm":
            v = v + 0.5 * dt / m.mass * F
        r = r + dt * v
        if rotates:
            qh = _unit(q + 0.5 * dt * _qdot(q, _rotate(_conj(q), L) * m.inv))
            L = L + 0.5 * dt * M
            q = _unit(q + dt * _qdot(qh, _rotate(_conj(qh), L) * m.inv))
        r = torch.where(r < 0, r + box, torch.where(r >= box, r - box, r))
        F, M, _, mac = m.forces(r, q)
        v = v + (1.0 if case["mode"] == "rmm" else 0.5) * dt / m.mass * F
        mv2 = (v * v).sum() if case["mode"] == "rmm" else (m.mass * v * v).sum()
        iw2 = torch.zeros((), **_T64)
        if rotates:
            L = L + 0.5 * dt * M
            w = _rotate(_conj(q), L) * m.inv
            iw2 = (m.inertia * w * w).sum()
        per.append(torch.stack([mac[0] / 6 + mac[1] + mac[3], mac[2] + 3 * mac[3], mv2, iw2,
                                mac[0] / 6, mac[1] + mac[3]]))
        if case["mode"] == "nvt":
            v = v * (3 * len(r) * s.temperature / mv2) ** 0.4
            if rotates:
                L = L * (m.rotdof * s.temperature / iw2) ** 0.4
    out = dict(r=r, v=v, records=torch.stack(per))
    if case["mode"] != "rmm":
        out["F"] = F
    if rotates:
        out.update(q=q, L=L, M=M)
    return out


def _charge_table(s):
    comps = _Model(s).comps
    q = torch.zeros(s.ncomp, 8, **_T64)
    for k, c in enumerate(comps):
        for t, x in enumerate(c["c"]):
            q[k, t] = x[4]
    return q


def _parameter_energy(s, eps, sig, q, r):
    """U, W as functions of symmetric LJ pair parameters [nlj, nlj], charges
    [ncomp, 8] and positions; truncation shifts follow their pair's parameters
    (cross-component pairs; these systems shift no pair of a component)."""
    m = _Model(s)
    base = np.cumsum([0] + [len(c["lj"]) for c in m.comps])
    i, j, sh = _pairs(r.detach(), np.asarray(s.box), s.rc)
    rot = _unit(torch.tensor(s.q, **_T64))
    U = W = torch.zeros((), **_T64)
    for a in range(s.ncomp):
        for b in range(s.ncomp):
            sel = (m.cid[i] == a) & (m.cid[j] == b)
            ii, jj = i[sel], j[sel]
            dm = r[ii] - r[jj] - sh[sel]
            for kind in ("lj", "c"):
                for x, xs in enumerate(m.comps[a][kind]):
                    di = _rotate(rot[ii], torch.tensor(xs[:3], **_T64).expand(len(ii), 3))
                    for y, ys in enumerate(m.comps[b][kind]):
                        d = dm + di - _rotate(rot[jj], torch.tensor(ys[:3], **_T64).expand(len(jj), 3))
                        r2, dd = (d * d).sum(1), (dm * d).sum(1)
                        if kind == "lj":
                            e, g = eps[base[a] + x, base[b] + y], sig[base[a] + x, base[b] + y]
                            l6 = (g * g / r2) ** 3
                            U = U + (4 * e * (l6 * l6 - l6)).sum()
                            W = W + (24 * e * (2 * l6 * l6 - l6) / r2 * dd).sum()
                            if a != b:
                                s6 = (g / s.rc_lj) ** 6
                                U = U + len(ii) * 4 * e * (s6 - s6 * s6)
                        else:
                            qq = q[a, x] * q[b, y]
                            U = U + (qq * r2.rsqrt()).sum()
                            W = W + (qq * r2 ** -1.5 * dd).sum()
    return U, W


def _pair_tables(s):
    m = _Model(s)
    ids = [(k, t) for k, c in enumerate(m.comps) for t in range(len(c["lj"]))]
    n = len(ids)
    eps, sig = torch.zeros(n, n, **_T64), torch.zeros(n, n, **_T64)
    for x, (a, sa) in enumerate(ids):
        for y, (b, sb) in enumerate(ids):
            e24, s2, _ = m.lj_pair(a, sa, b, sb)
            eps[x, y], sig[x, y] = e24 / 24, math.sqrt(s2)
    return eps, sig


def _exact_adjoint(case, s, seed):
    eps, sig = _pair_tables(s)
    n = len(eps)
    up = torch.triu_indices(n, n, device=_DEV)

    def full(x):
        y = torch.zeros(n, n, **_T64).index_put((up[0], up[1]), x)
        return y + y.T - torch.diag(torch.diagonal(y))

    pe, ps = (x[up[0], up[1]].clone().requires_grad_(True) for x in (eps, sig))
    q = _charge_table(s).requires_grad_(True)
    r = torch.tensor(s.r, **_T64).requires_grad_(True)
    U, W = _parameter_energy(s, full(pe), full(ps), q, r)
    out = {}
    for key, x in (("U", U), ("W", W)):
        g = torch.autograd.grad(x, (pe, ps), retain_graph=True)
        out["d%s_deps" % key], out["d%s_dsig" % key] = full(g[0]), full(g[1])
        out["d%s_dq" % key] = torch.zeros(s.ncomp, 8, **_T64)
    if case["vjp"]:
        cot = torch.tensor(np.random.default_rng(seed + 7).normal(size=(s.n, 3)), **_T64)
        F = -torch.autograd.grad(U, r, create_graph=True)[0]
        out["vjp"] = torch.autograd.grad((F * cot).sum(), r)[0]
    return out


def _exact_fit(s):
    eps, sig = _pair_tables(s)
    n = len(eps)
    up = torch.triu_indices(n, n, device=_DEV)

    def full(x):
        y = torch.zeros(n, n, **_T64).index_put((up[0], up[1]), x)
        return y + y.T - torch.diag(torch.diagonal(y))

    pe, ps = (x[up[0], up[1]].clone().requires_grad_(True) for x in (eps, sig))
    q = _charge_table(s).requires_grad_(True)
    r = torch.tensor(s.r, **_T64).requires_grad_(True)
    U, W = _parameter_energy(s, full(pe), full(ps), q, r)
    loss = U / s.n + 0.1 * W / s.n
    g = torch.autograd.grad(loss, (pe, ps, q), retain_graph=True)
    F = -torch.autograd.grad(U, r)[0]
    new = [(x - 1e-6 * y).detach() for x, y in zip((pe, ps, q), g)]
    return dict(loss=loss.detach(), F=F, g_eps=g[0], g_sig=g[1], g_q=g[2], eps=new[0], sig=new[1],
                q=new[2])


def exact(case, seed):
    seed = int(seed) % 1000003
    n, kind, system = case["n"], case["kind"], case["system"]
    if kind == "steps":
        if system == "replicas" or n * case["steps"] > (2000000 if system != "mixture" else 460000):
            return None
        return _exact_steps(case, _systems(case, seed)[0])
    s = _systems(case, seed)[0]
    if kind == "forces":
        if n > 400000:
            return None
        F, M, Vi, mac = _Model(s).forces(torch.tensor(s.r, **_T64), _unit(torch.tensor(s.q, **_T64)))
        out = dict(F=F, Vi=Vi, macro=mac)
        if system in ("mixture", "allsites"):
            out["M"] = M
        return out
    if kind == "adjoint":
        return _exact_adjoint(case, s, seed)
    return _exact_fit(s)
