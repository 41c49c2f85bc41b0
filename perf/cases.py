"""The work a user of x2dhf_amd has the GPU do, as timed cases.

Each case is one call (or the short call sequence of one SCF step) through the
public entry points: the C ABI of include/x2gpu.h as x2dhf_amd.gpu binds it,
and the SCF driver of x2dhf_amd.scf.  `kind` selects the path:

  mcsor     x2g_mcsor, the drop-in for one padded function (FP64)
  relax     x2g_relax_batch: potentials (psi_i psi_j g sources, Coulomb and
            exchange, both parities) or orbitals (with their asymptotic tail)
            of one or more jobs, FP64 or mixed precision
  ordered   x2g_relax_batch with the reference's sequential schemes (SOR
            forward and backward, one-thread MCSOR) in a mesh ordering
  fock      x2g_lincomb_batch, x2g_normortho_batch and x2g_eahf_batch: the
            Fock operators, normalisation / orthogonalisation and orbital
            energies between two relaxations
  scf       whole SCF iterations (plain or batched schedule) of one or more
            jobs, with the orbitals read back

Grid sizes are those of the served stream (169x241 .. 505x901), of the
Poisson batch and of the decks (61x91 .. 481x901), all with n - 1 divisible
by 6.  `grids` is a text "nni x nmu * count + ...", one group per job: the
items of a group share its grid, its lhs and its orbitals, as the potentials
of one molecule do.
"""
import ctypes as C
import math

import numpy as np
import torch

from x2dhf_amd import gpu, scf

RINF = 40.0
_CTX = None


def _ctx():
    """One context per process, as a program keeps it."""
    global _CTX
    if _CTX is None:
        _CTX = gpu.Context(0)
    return _CTX


# ---------------------------------------------------------------------------
# the cases

def listed():
    return [
        # smallest call: one H2 orbital through the drop-in sweep
        dict(name="mcsor_h2_91x121", kind="mcsor", nni=91, nmu=121, bkind=0, isym=1, sweeps=10),
        # the same drop-in at the largest single-molecule deck (FH)
        dict(name="mcsor_fh_481x901", kind="mcsor", nni=481, nmu=901, bkind=1, isym=-1, sweeps=10),
        # the orbitals of one N2 job, FP64 (default precision of the driver)
        dict(name="orbitals_n2_fp64", kind="relax", what="orb", grids="331x601*6", prec=0, sweeps=10),
        # the potentials of one N2 job: FP64, and mixed precision
        dict(name="potentials_n2_fp64", kind="relax", what="pot", grids="331x601*22", prec=0, sweeps=10),
        dict(name="potentials_n2_mixed", kind="relax", what="pot", grids="331x601*22", prec=1, sweeps=10),
        # a served batch of different molecules, each on its own grid
        dict(name="potentials_stream_mixed", kind="relax", what="pot", prec=1, sweeps=10,
             grids="505x901*14+505x901*14+409x721*10+409x721*10+361x601*10+361x601*10+217x361*8+217x361*8+"
                   "169x241*8+169x241*8"),
        # sixteen N2 jobs stepped together: the largest relaxation served
        dict(name="potentials_16n2_mixed", kind="relax", what="pot", prec=1, sweeps=10,
             grids="+".join(["331x601*22"] * 16)),
        # the reference's default scheme: SOR in the middle ordering, the
        # potentials of one LiH job and the one potential of a He atom deck
        dict(name="sor_middle_lih_169x241", kind="ordered", nni=169, nmu=241, count=3, method=1, ordering=1,
             sweeps=10),
        dict(name="sor_middle_he_331x601", kind="ordered", nni=331, nmu=601, count=1, method=1, ordering=1,
             sweeps=10),
        # Fock operators, orthonormalisation and energies of eight N2 jobs
        dict(name="fock_8n2", kind="fock", nni=331, nmu=601, jobs=8, norb=6),
        # whole SCF iterations: one small job in the plain schedule (launch
        # bound), and a batch of served jobs in mixed precision, resumed from
        # the state of an FP64 run
        dict(name="scf_plain_h2_91x121", kind="scf", mol="h2", nni=91, nmu=121, jobs=1, schedule=0, prec=0, iters=4,
             warm=20),
        dict(name="scf_batched_mixed", kind="scf", mol="mix", nni=217, nmu=301, jobs=6, schedule=1, prec=1, iters=4,
             warm=600),
    ]


def _size(rng, lo, hi, aspect):
    """Grid sizes 6k+1, log-uniform in nni over [lo, hi], any residue mod 5."""
    n = int(math.exp(rng.uniform(math.log(lo), math.log(hi))))
    nni = 6 * (n // 6) + 1
    nmu = 6 * int(nni * rng.uniform(*aspect) / 6) + 1
    return max(nni, 61), max(nmu, 91)


def draw(rng):
    kind = rng.choice(["mcsor", "relax", "relax", "relax", "relax", "ordered", "fock", "scf"])
    if kind == "mcsor":
        nni, nmu = _size(rng, 61, 515, (1.3, 1.9))
        return dict(kind=kind, nni=nni, nmu=nmu, bkind=rng.randint(0, 1), isym=rng.choice([1, -1]),
                    sweeps=rng.choice([1, 4, 7, 10, 10, 20]))
    if kind == "relax":
        prec = rng.choice([0, 1, 1])
        what = "orb" if rng.random() < 0.25 else "pot"
        jobs = int(math.exp(rng.uniform(0.0, math.log(16.99 if prec else 8.99))))
        groups, points = [], 0
        for _ in range(jobs):
            nni, nmu = _size(rng, 91, 511, (1.4, 1.85))
            count = rng.randint(1, 6) if what == "orb" else rng.randint(1, 15)
            points += nni * nmu * count
            if groups and points > (40e6 if prec else 15e6):  # no dearer than the largest listed case
                break
            groups.append("%dx%d*%d" % (nni, nmu, count))
        return dict(kind=kind, what=what, grids="+".join(groups), prec=prec, sweeps=rng.choice([5, 8, 10, 10, 10, 15]))
    if kind == "ordered":
        nni, nmu = _size(rng, 61, 340, (1.3, 1.85))
        return dict(kind=kind, nni=nni, nmu=nmu, count=rng.randint(1, 6), method=rng.choice([1, 1, 2, 0]),
                    ordering=rng.choice([0, 1, 1, 3]), sweeps=rng.choice([5, 10]))
    if kind == "fock":
        nni, nmu = _size(rng, 91, 505, (1.4, 1.85))
        return dict(kind=kind, nni=nni, nmu=nmu, jobs=rng.randint(1, 3), norb=rng.randint(2, 6))
    nni, nmu = _size(rng, 91, 241, (1.3, 1.7))
    mol = rng.choice(["h2", "lih", "mix"])
    prec = 1 if mol == "mix" else 0
    return dict(kind=kind, mol=mol, nni=nni, nmu=nmu, jobs=rng.randint(2, 5) if mol == "mix" else 1,
                schedule=prec, prec=prec, iters=rng.randint(2, 5), warm=600 if prec else 20)


# ---------------------------------------------------------------------------
# inputs: smooth functions of the kind the relaxation meets, from the seed
# alone, formed with torch (on the GPU where there is one)

def _dev():
    return torch.device("cuda") if torch.cuda.is_available() else torch.device("cpu")


def _groups(text):
    out = []
    for part in text.split("+"):
        size, count = part.split("*")
        nni, nmu = size.split("x")
        out.append((int(nni), int(nmu), int(count)))
    return out


_D1 = [3.0, -32.0, 168.0, -672.0]
_D2 = [-9.0, 128.0, -1008.0, 8064.0]
_EX = [210.0 / 126, -120.0 / 126, 45.0 / 126, -10.0 / 126, 1.0 / 126]


class Axes:
    """The prolate-spheroidal mesh of (nni, nmu, r) in plain arithmetic: xi =
    cosh(mu), eta = cos(nu), fields indexed [mu, nu]."""

    def __init__(self, nni, nmu, r, z1, z2):
        dev, f8 = _dev(), torch.float64
        self.nni, self.nmu, self.r, self.z1, self.z2 = nni, nmu, r, z1, z2
        self.hni = math.pi / (nni - 1)
        x = 2.0 * RINF / r
        self.hmu = math.log(x + math.sqrt(x * x - 1.0)) / (nmu - 1)
        mu = torch.arange(nmu, dtype=f8, device=dev) * self.hmu
        nu = torch.arange(nni, dtype=f8, device=dev) * self.hni
        self.xi, self.sh = torch.cosh(mu)[:, None], torch.sinh(mu)[:, None]
        self.eta, self.sn = torch.cos(nu)[None, :], torch.sin(nu)[None, :]
        self.q = self.xi ** 2 - self.eta ** 2
        self.diag = -14350.0 / 5040.0 * (1.0 / self.hmu ** 2 + 1.0 / self.hni ** 2)
        self.f0 = r * (self.xi * (z1 + z2) + self.eta * (z2 - z1)).expand(nmu, nni)
        self.f1 = r * r * self.q / 2.0
        self.f2 = -r * self.q / self.xi
        self.f2[0] = 0.0
        self.f3 = (-2.0 / self.xi ** 2 + self.diag).expand(nmu, nni)
        self.f4 = (0.5 * r * self.xi).expand(nmu, nni)
        self.g = (-r ** 3 * math.pi * self.xi / 2.0) * self.q
        inner = torch.ones(nmu, dtype=f8, device=dev)[:, None]
        inner[0] = 0.0
        sh1, sn1 = self.sh.clone(), self.sn.clone()
        sh1[0] = 1.0
        sn1[:, 0] = 1.0
        sn1[:, -1] = 1.0
        edge = torch.ones(nni, dtype=f8, device=dev)[None, :]
        edge[:, 0] = 0.0
        edge[:, -1] = 0.0
        self.e = (-inner / sh1 ** 2 - 1.0 / sn1 ** 2) * edge
        self.borb = self.xi / sh1 * inner
        self.bpot = (self.xi / sh1 - 2.0 * self.sh / self.xi) * inner
        self.dnu = self.eta / sn1 * edge
        self.z = 0.5 * r * self.xi * self.eta
        self.rho2 = (0.5 * r) ** 2 * self.sh ** 2 * self.sn ** 2

    def weights(self):
        """(wgt1, wgt2): volume elements with the 7-point Newton-Cotes rule."""
        def rule(n, h):
            w = torch.tensor([82.0, 216.0, 27.0, 272.0, 27.0, 216.0], dtype=torch.float64, device=_dev())
            w = w[torch.arange(n, device=_dev()) % 6].clone()
            w[0] = w[-1] = 41.0
            return w * (h / 140.0)
        w = rule(self.nmu, self.hmu)[:, None] * rule(self.nni, self.hni)[None, :]
        s = self.sh * self.sn
        return (w * (-math.pi * self.r / 2.0) * s,
                w * (math.pi * self.r ** 2 / 2.0) * s * (self.sh ** 2 + self.sn ** 2) / self.xi)


def _embed(u, isym):
    """[k, mu, nu] -> [k, mu+8, nu+8] with mirror halos below mu = 1 and
    outside nu = 1..nni, zeros above the last row."""
    s = 1.0 if isym == 1 else -1.0
    k, nmu, nni = u.shape
    w = torch.zeros(k, nmu + 8, nni + 8, dtype=u.dtype, device=u.device)
    w[:, 4:-4, 4:-4] = u
    w[:, :4, 4:-4] = s * u[:, 1:5].flip(1)
    w[:, 4:-4, :4] = s * u[:, :, 1:5].flip(2)
    w[:, 4:-4, -4:] = s * u[:, :, -5:-1].flip(2)
    return w


def _operator(ax, w, b):
    """L of the 17-point cross without its diagonal, over the nni x nmu points."""
    nmu, nni = ax.nmu, ax.nni
    c = w[:, 4:4 + nmu, 4:4 + nni]
    out = torch.zeros_like(c)
    d1 = torch.zeros_like(c)
    for i, k in enumerate((4, 3, 2, 1)):
        m, p = w[:, 4 - k:4 - k + nmu, 4:4 + nni], w[:, 4 + k:4 + k + nmu, 4:4 + nni]
        out += _D2[i] / 5040.0 / ax.hmu ** 2 * (m + p)
        d1 += _D1[i] / 840.0 / ax.hmu * (m - p)
    out += b * d1
    d1.zero_()
    for i, k in enumerate((4, 3, 2, 1)):
        m, p = w[:, 4:4 + nmu, 4 - k:4 - k + nni], w[:, 4:4 + nmu, 4 + k:4 + k + nni]
        out += _D2[i] / 5040.0 / ax.hni ** 2 * (m + p)
        d1 += _D1[i] / 840.0 / ax.hni * (m - p)
    return out + ax.dnu * d1


def _rng(seed, k):
    return np.random.default_rng([int(seed) & 0x7FFFFFFF, k])


def _omegas(nni, nmu, zmax):
    rho = 0.5 * (math.cos(math.pi / nmu) + math.cos(math.pi / nni))
    pot = 2.0 * 0.603 / (1.0 + math.sqrt(1.0 - rho * rho)) + 0.79
    return (pot - 1.0) * pot - 0.001 * zmax, pot


def _axes(nni, nmu, seed, k):
    g = _rng(seed, 100 + k)
    return Axes(nni, nmu, float(g.uniform(1.2, 4.0)), float(g.integers(1, 10)), float(g.integers(1, 10)))


def _noise(ax, g):
    """1 + a smooth relative change of 1e-4: how far a potential or orbital
    moves in an iteration of a settling SCF."""
    a, b, ph = float(g.uniform(1, 6)), float(g.uniform(0.2, 1)), float(g.uniform(0, 6))
    return 1.0 + 1e-4 * torch.cos(a * ax.eta + ph) / ax.xi ** b


def _orbital(ax, g, m):
    """A two-centre hydrogenic orbital (m = 1: times rho, odd on the axis)."""
    h = 0.5 * ax.r
    za, zb, c = float(g.uniform(0.7, 3.0)), float(g.uniform(0.7, 3.0)), float(g.uniform(-1, 1))
    psi = torch.exp(-za * h * (ax.xi + ax.eta)) + c * torch.exp(-zb * h * (ax.xi - ax.eta))
    if m:
        psi = psi * torch.sqrt(ax.rho2)
    return psi


def _pairs(count):
    """(number of s orbitals, [(i, j)]) of `count` potentials; j = -1 pairs
    orbital i with the group's pi orbital (an odd exchange potential)."""
    ns = 1
    while ns * (ns + 1) // 2 + ns < count:
        ns += 1
    out = []
    for i in range(ns):
        out += [(i, i), (i, -1)] + [(i, j) for j in range(i + 1, ns)]
    return ns, out[:count]


def _potentials(ax, count, seed, k):
    """Orbitals [ns+1, mu, nu] (Gaussians, the last one pi) and, for each
    pair, (i, j, isym, converged potential).  psi_i psi_j is a Gaussian (or
    rho times one) at the product's centre, whose potential is closed-form."""
    g = _rng(seed, 200 + k)
    ns, pairs = _pairs(count)
    alpha, cen = g.uniform(0.15, 3.0, ns + 1), g.uniform(-0.6, 0.6, ns + 1) * ax.r
    psi = torch.stack([torch.exp(-alpha[i] * (ax.rho2 + (ax.z - cen[i]) ** 2)) * (2 * alpha[i] / math.pi) ** 0.75
                       for i in range(ns + 1)])
    psi[ns] *= torch.sqrt(ax.rho2) * math.sqrt(2.0 * alpha[ns])
    out = []
    for i, j in pairs:
        jj = ns if j < 0 else j
        p = alpha[i] + alpha[jj]
        zc = (alpha[i] * cen[i] + alpha[jj] * cen[jj]) / p
        amp = math.exp(-alpha[i] * alpha[jj] / p * (cen[i] - cen[jj]) ** 2)
        amp *= (2 * alpha[i] / math.pi) ** 0.75 * (2 * alpha[jj] / math.pi) ** 0.75
        if j < 0:
            amp *= math.sqrt(2.0 * alpha[jj])
        rr = torch.sqrt(ax.rho2 + (ax.z - zc) ** 2).clamp_min(1e-6)
        t = math.sqrt(p) * rr
        q = amp * (math.pi / p) ** 1.5
        if j >= 0:
            v = q * torch.erf(t) / rr
        else:  # x exp(-p r^2) = -1/(2p) d/dx exp(-p r^2)
            h = torch.where(t < 0.05, (4.0 / (3.0 * math.sqrt(math.pi)) * p ** 1.5 * (1.0 - 0.6 * t * t)),
                            torch.erf(t) / rr ** 3 - 2.0 * math.sqrt(p / math.pi) * torch.exp(-t * t) / rr ** 2)
            v = q / (2.0 * p) * h * torch.sqrt(ax.rho2)
        out.append((i, jj, 1 if j >= 0 else -1, ax.f4 * v))
    return psi, out


def _relax_group(case, nni, nmu, count, seed, k):
    """One job's relaxation inputs as [count, nmu, nni] fields:
    dict(u, lhs list, rhs, isym, bkind, omega, psi, pairs, fock1)."""
    ax = _axes(nni, nmu, seed, k)
    om_orb, om_pot = _omegas(nni, nmu, max(ax.z1, ax.z2))
    g = _rng(seed, 300 + k)
    if case.get("what") == "orb":
        us, lhss, rhss, focks, isyms = [], [], [], [], []
        for i in range(count):
            m = 1 if i % 3 == 2 else 0
            psi = _orbital(ax, g, m)
            fock1 = 0.3 * ax.f0 - float(g.uniform(0.3, 2.0)) * ax.f1 + m * ax.e
            isym = -1 if m else 1
            lhs = fock1 + ax.diag
            rhss.append(_operator(ax, _embed(psi[None], isym), ax.borb)[0] + lhs * psi)
            us.append(psi * _noise(ax, g))
            lhss.append(lhs)
            focks.append(fock1)
            isyms.append(isym)
        return dict(ax=ax, u=torch.stack(us), lhs=torch.stack(lhss), lhs_of=list(range(count)),
                    rhs=torch.stack(rhss), fock1=torch.stack(focks), isym=isyms, bkind=0, omega=om_orb, psi=None)
    psi, pots = _potentials(ax, count, seed, k)
    lhs = torch.stack([ax.f3, ax.f3 + ax.e])
    u = torch.stack([v * _noise(ax, g) for _, _, _, v in pots])
    u[:, -4:] = torch.stack([v[-4:] for _, _, _, v in pots])
    return dict(ax=ax, u=u, lhs=lhs, lhs_of=[0 if s == 1 else 1 for _, _, s, _ in pots], rhs=None,
                pairs=[(i, j) for i, j, _, _ in pots], psi=psi, isym=[s for _, _, s, _ in pots], bkind=1,
                omega=om_pot, fock1=None)


def _rhs(d):
    """The right-hand sides of a group as one [count, mu, nu] field."""
    if d["rhs"] is not None:
        return d["rhs"]
    return torch.stack([d["psi"][i] * d["psi"][j] * d["ax"].g for i, j in d["pairs"]])


def _mcsor_inputs(case, seed):
    nni, nmu = case["nni"], case["nmu"]
    ax = _axes(nni, nmu, seed, 0)
    om_orb, om_pot = _omegas(nni, nmu, max(ax.z1, ax.z2))
    g = _rng(seed, 1)
    m = 0 if case["isym"] == 1 else 1
    if case["bkind"] == 0:
        u = _orbital(ax, g, m)
        lhs = 0.3 * ax.f0 - float(g.uniform(0.3, 2.0)) * ax.f1 + m * ax.e + ax.diag
        b, om = ax.borb, om_orb
    else:
        _, pots = _potentials(ax, 2, seed, 0)
        u = pots[m][3]
        lhs = ax.f3 + m * ax.e
        b, om = ax.bpot, om_pot
    rhs = _operator(ax, _embed(u[None], case["isym"]), b)[0] + lhs * u
    return ax, u * _noise(ax, g), lhs, rhs, om


# ---------------------------------------------------------------------------
# what a program holds before the call

def _grid(ax):
    """The device grid from the package's own grid builder."""
    coef, suppl, vxi, veta = scf.grid_build(ax.nni, ax.nmu, ax.z1, ax.z2, ax.r, RINF)
    return gpu.Grid(_ctx(), ax.nni, ax.nmu, coef, suppl, vxi, veta)


class State(dict):
    """A case's buffers and handles; the grids and jobs go with it."""

    def __del__(self):
        if torch is None or not (self.get("grids") or self.get("jobs")):
            return
        torch.cuda.synchronize()
        for g in self.get("grids", ()):
            g.destroy()
        for j in self.get("jobs", ()):
            j.close()


def _handles(grids):
    return (gpu._vp * len(grids))(*[g.h.value for g in grids])


def _suppl(g, k):
    return g.suppl_ptr(k)


def _prepare_relax(case, seed, groups):
    grids, items, outs, keep = [], [], [], []
    for k, (nni, nmu, count) in enumerate(groups):
        d = _relax_group(case, nni, nmu, count, seed, k)
        g = _grid(d["ax"])
        grids.append(g)
        u = d["u"].contiguous()
        lhs = d["lhs"].contiguous()
        mixed_pot = d["psi"] is not None and case.get("prec") == 1
        rhs = torch.zeros_like(u) if mixed_pot else _rhs(d).contiguous()
        nb = nni * nmu * 8
        psi = d["psi"].contiguous() if d["psi"] is not None else None
        fock1 = d["fock1"].contiguous() if d["fock1"] is not None else None
        keep += [lhs, rhs, psi, fock1]
        outs.append(u)
        for q in range(count):
            it = gpu.RelaxItem(u.data_ptr() + q * nb, lhs.data_ptr() + d["lhs_of"][q] * nb, rhs.data_ptr() + q * nb,
                               fock1.data_ptr() + q * nb if fock1 is not None else None, d["omega"], d["isym"][q],
                               d["bkind"], case.get("prec", 0), k)
            if mixed_pot:
                i, j = d["pairs"][q]
                it.rhs_f1_d, it.rhs_f2_d = psi.data_ptr() + i * nb, psi.data_ptr() + j * nb
                it.rhs_f3_d = _suppl(g, 9)
            it.method, it.ordering = case.get("method", 0), case.get("ordering", 0)
            items.append(it)
    s = State(kind="relax", grids=grids, keep=keep, outs=outs, gh=_handles(grids),
              items=(gpu.RelaxItem * len(items))(*items), n=len(items), sweeps=case["sweeps"])
    torch.cuda.synchronize()
    return s


def _prepare_fock(case, seed):
    """`jobs` jobs of `norb` orbitals (s Gaussians and hydrogenic functions)
    with their potentials: the operators' term lists as the SCF loop makes
    them, one exchange slot per orbital pair."""
    ctx = _ctx()
    nni, nmu, norb, jobs = case["nni"], case["nmu"], case["norb"], case["jobs"]
    n = nni * nmu
    nb = 8 * n
    grids, bufs = [], []
    ops1, terms1, ops2, terms2, eahf = [], [], [], [], []
    no = [[] for _ in range(norb)]
    outs = {"orb": [], "fock": []}
    scal = torch.zeros(2, jobs, norb, dtype=torch.float64, device=_dev())
    for q in range(jobs):
        d = _fock_inputs(case, seed, q)
        g = _grid(d["ax"])
        grids.append(g)
        orb, coul, exch = d["orb"].contiguous(), d["coul"].contiguous(), d["exch"].contiguous()
        # cpot, xpot, fock1, lhs of every orbital
        f = torch.zeros(4, norb, nmu, nni, dtype=torch.float64, device=orb.device)
        bufs += [coul, exch]
        outs["orb"].append(orb)
        outs["fock"].append(f)

        def at(t, k):
            return t.data_ptr() + k * nb
        cpot, xpot, f1, lo = (f[i] for i in range(4))
        for i in range(norb):
            ops1.append(gpu.LincombOp(at(cpot, i), None, 0.0, len(terms1), norb, q))
            terms1 += [gpu.Term(d["coo"][i][j], at(coul, j), None, None) for j in range(norb)]
            tx = [gpu.Term(1.0, at(exch, d["slot"][i][j]), at(orb, j), None) for j in range(norb) if j != i]
            ops1.append(gpu.LincombOp(at(xpot, i), None, 0.0, len(terms1), len(tx), q))
            terms1 += tx
            t1 = [gpu.Term(d["eps"][i], _suppl(g, 5), None, None)]
            if d["m"][i]:
                t1.append(gpu.Term(1.0, _suppl(g, 3), None, None))
            t1.append(gpu.Term(1.0, _suppl(g, 6), at(cpot, i), None))
            ops2.append(gpu.LincombOp(at(f1, i), _suppl(g, 4), 1.0, len(terms2), len(t1), q))
            terms2 += t1
            t1 = t1 + [gpu.Term(d["ax"].diag, d["ones"].data_ptr(), None, None)]
            ops2.append(gpu.LincombOp(at(lo, i), _suppl(g, 4), 1.0, len(terms2), len(t1), q))
            terms2 += t1
            others = [j for j in range(i + 1, norb) if d["m"][j] == d["m"][i]]
            it = gpu.NormOrthoItem(at(orb, i), (gpu._vp * gpu.MAX_ORTHO)(*[at(orb, j) for j in reversed(others)]),
                                   len(others), 0, 1, q, scal[0, q, i].data_ptr())
            no[norb - 1 - i].append(it)
            eahf.append(gpu.EaHFItem(at(orb, i), at(cpot, i), at(xpot, i), -1 if d["m"][i] else 1, d["m"][i], q,
                                     scal[1, q, i].data_ptr()))
        bufs.append(d["ones"])

    def arr(t, v):
        return (t * len(v))(*v)
    s = State(kind="fock", grids=grids, keep=bufs, gh=_handles(grids), ctx=ctx, outs=outs, scal=scal,
              ops1=arr(gpu.LincombOp, ops1), terms1=arr(gpu.Term, terms1), ops2=arr(gpu.LincombOp, ops2),
              terms2=arr(gpu.Term, terms2), no=[arr(gpu.NormOrthoItem, v) for v in no],
              eahf=arr(gpu.EaHFItem, eahf))
    torch.cuda.synchronize()
    return s


def _fock_inputs(case, seed, q):
    nni, nmu, norb = case["nni"], case["nmu"], case["norb"]
    ax = _axes(nni, nmu, seed, q)
    g = _rng(seed, 400 + q)
    m = [1 if norb > 2 and i == 0 else 0 for i in range(norb)]
    orb = torch.stack([_orbital(ax, g, mm) for mm in m])
    npair = norb * (norb - 1) // 2
    _, pots = _potentials(ax, norb + npair + norb + 1, seed, q)
    even = [v for _, _, s, v in pots if s == 1]
    coul = torch.stack([even[i % len(even)] * float(g.uniform(0.5, 1.5)) for i in range(norb)])
    exch = torch.stack([even[i % len(even)] * float(g.uniform(0.05, 0.5)) for i in range(npair)])
    slot = [[0] * norb for _ in range(norb)]
    k = 0
    for i in range(norb):
        for j in range(i + 1, norb):
            slot[i][j] = slot[j][i] = k
            k += 1
    coo = [[(4.0 if m[j] else 2.0) - (1.0 if i == j else 0.0) for j in range(norb)] for i in range(norb)]
    return dict(ax=ax, m=m, orb=orb, coul=coul, exch=exch, slot=slot, coo=coo,
                eps=[-float(g.uniform(0.3, 15.0)) for _ in range(norb)],
                ones=torch.ones(nmu, nni, dtype=torch.float64, device=orb.device))


_MOLS = {"h2": [scf.h2_spec], "lih": [scf.lih_spec], "mix": [scf.lih_spec, scf.bh_spec, scf.h2_spec]}


def _jobs(case, seed, prec):
    """Jobs with stop thresholds out of reach, on slightly different R."""
    g = _rng(seed, 7)
    jobs = []
    for k in range(case["jobs"]):
        f = _MOLS[case["mol"]][k % len(_MOLS[case["mol"]])]
        r = {scf.h2_spec: 1.4, scf.lih_spec: 3.015, scf.bh_spec: 2.3289}[f] * float(g.uniform(0.95, 1.05))
        spec = f(nni=case["nni"] + 48 * (k % 2 if case["mol"] == "mix" else 0), nmu=case["nmu"], r=r,
                 schedule=case["schedule"], prec=prec, maxscf=1 << 30, ienterm=40, inoterm=40,
                 conv=(1 << 30, 1 << 30, 1 << 30))
        jobs.append(scf.Job(spec, ctx=_ctx()))
    return jobs


def _prepare_scf(case, seed):
    """FP64 jobs some iterations into their SCF; a mixed-precision case
    resumes from the orbitals and potentials of such jobs."""
    first = State(jobs=_jobs(case, seed, 0), schedule=case["schedule"])
    for j in first["jobs"]:
        j.prep()
    _advance(first, case["warm"])
    first.update(kind="scf", iters=case["iters"])
    if case["prec"] == 0:
        torch.cuda.synchronize()
        return first
    jobs = _jobs(case, seed, case["prec"])
    for old, new in zip(first["jobs"], jobs):
        norb = old.spec.norb
        for kind, count in ((0, norb), (1, norb), (2, norb * (norb - 1) // 2)):
            for i in range(1, count + 1):
                new.put(kind, i, old.get(kind, i))
        new.prep_restart(np.diag(old.result()["eps"]))
    s = State(kind="scf", jobs=jobs, schedule=case["schedule"], iters=case["iters"])
    torch.cuda.synchronize()
    return s


def _advance(s, iters):
    if s["schedule"] == 0:
        for j in s["jobs"]:
            j.iterate(iters)
    else:
        for _ in range(iters):
            scf.iterate_batched(s["jobs"])


def prepare(case, seed):
    kind = case["kind"]
    if kind == "relax":
        return _prepare_relax(case, seed, _groups(case["grids"]))
    if kind == "ordered":
        return _prepare_relax(case, seed, [(case["nni"], case["nmu"], case["count"])])
    if kind == "fock":
        return _prepare_fock(case, seed)
    if kind == "scf":
        return _prepare_scf(case, seed)
    ax, u, lhs, rhs, om = _mcsor_inputs(case, seed)
    g = _grid(ax)
    s = State(kind="mcsor", grids=[g], work=_embed(u[None], case["isym"])[0].contiguous(), lhs=lhs.contiguous(),
              rhs=rhs.contiguous(), omega=om, isym=case["isym"], bkind=case["bkind"], sweeps=case["sweeps"])
    torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------------------
# one pass

def run(s):
    ctx = _ctx()
    lib = ctx.lib
    kind = s["kind"]
    if kind == "mcsor":
        gpu.check(lib.x2g_mcsor(s["grids"][0].h, s["isym"], s["bkind"], s["work"].data_ptr(), s["lhs"].data_ptr(),
                                s["rhs"].data_ptr(), s["omega"], s["sweeps"]))
        return s["work"]
    if kind == "relax":
        gpu.check(lib.x2g_relax_batch(ctx.h, s["gh"], s["items"], s["n"], 1, s["sweeps"]))
        return s["outs"]
    if kind == "fock":
        gh = s["gh"]
        for ops, terms in ((s["ops1"], s["terms1"]), (s["ops2"], s["terms2"])):
            gpu.check(lib.x2g_lincomb_batch(ctx.h, gh, ops, len(ops), terms, len(terms)))
        for no in s["no"]:
            gpu.check(lib.x2g_normortho_batch(ctx.h, gh, no, len(no)))
        gpu.check(lib.x2g_eahf_batch(ctx.h, gh, s["eahf"], len(s["eahf"])))
        return {"orb": s["outs"]["orb"], "fock": s["outs"]["fock"], "scal": s["scal"]}
    _advance(s, s["iters"])
    res = [j.result() for j in s["jobs"]]
    return {"eps": [r["eps"] for r in res], "norm": [r["norm"] for r in res],
            "orb": [j.get(0, i + 1) for j in s["jobs"] for i in range(j.spec.norb)]}


# ---------------------------------------------------------------------------
# the same in plain 64-bit torch

def _colours(ax):
    nni, nmu = ax.nni, ax.nmu
    ca = (nni - 2) % 5 or 4
    mu = torch.arange(nmu, device=_dev())[:, None] - 1
    nu = torch.arange(nni, device=_dev())[None, :] - 1
    col = (nu + ca * mu) % 5
    inner = (mu >= 0) & (mu <= nmu - 6) & (nu >= 0) & (nu <= nni - 3)
    return [inner & (col == c) for c in range(5)]


def _boundary(ax, w, isym):
    nmu, nni = ax.nmu, ax.nni
    if isym != 1:
        w[:, 4, 5:nni + 3] = 0.0
        w[:, 4:nmu, 4] = 0.0
        w[:, 4:nmu, nni + 3] = 0.0
        return
    w[:, 4, 5:nni + 3] = sum(_EX[k] * w[:, 5 + k, 5:nni + 3] for k in range(5))
    w[:, 4:nmu, 4] = sum(_EX[k] * w[:, 4:nmu, 5 + k] for k in range(5))
    w[:, 4:nmu, nni + 3] = sum(_EX[k] * w[:, 4:nmu, nni + 2 - k] for k in range(5))


def _mcsor(ax, w, lhs, rhs, b, isym, omega, sweeps):
    cols = _colours(ax)
    u = w[:, 4:-4, 4:-4]
    for _ in range(sweeps):
        for c in cols:
            new = omega * (rhs - _operator(ax, w, b)) / lhs + (1.0 - omega) * u
            u.copy_(torch.where(c, new, u))
        _boundary(ax, w, isym)


def _order(ax, ordering):
    """Relaxed points (padded row, column) in mesh ordering 0 col-wise,
    1 middle, 3 row-wise."""
    nni, nmu = ax.nni, ax.nmu
    rows, cols = list(range(5, nmu)), list(range(5, nni + 3))
    if ordering == 1:
        rm, cm = (nmu + 7) // 2 - 1, (nni + 7) // 2 - 1
        rows = [rm - i + 5 if i <= rm else i for i in rows]
        cols = [cm - i + 5 if i <= cm else i for i in cols]
    if ordering == 3:
        return [(r, c) for c in cols for r in rows]
    return [(r, c) for r in rows for c in cols]


def _sequential(ax, w, lhs, rhs, b, isym, omega, sweeps, method, ordering):
    """The sequential schemes, one set of mutually independent points at a
    time (w [k, mu+8, nu+8], lhs / rhs [k, mu, nu])."""
    nni = ax.nni
    n8 = nni + 8
    seq = _order(ax, ordering)
    if method == 2:
        seq = seq[::-1]
    passes = [seq[c::5] for c in range(5)] if method == 0 else [seq]
    nb = [d for k in (1, 2, 3, 4) for d in (k, -k, k * n8, -k * n8)]
    sets = []
    for pts in passes:
        lev, by = {}, []
        for r, c in pts:
            p = r * n8 + c
            got = -1
            for d in nb:
                v = lev.get(p + d, -1)
                if v > got:
                    got = v
            lev[p] = got + 1
            if got + 1 == len(by):
                by.append([])
            by[got + 1].append(p)
        sets += by
    a = w.cpu().numpy().reshape(w.shape[0], -1).copy()
    lh = np.stack([x.cpu().numpy() for x in lhs])
    rh = rhs.cpu().numpy()
    bb = b.expand(ax.nmu, nni).cpu().numpy()
    dd = ax.dnu.expand(ax.nmu, nni).cpu().numpy()
    idx = []
    for s in sets:
        p = np.array(s)
        mu, nu = p // n8 - 4, p % n8 - 4
        idx.append((p, lh[:, mu, nu], rh[:, mu, nu], bb[mu, nu], dd[mu, nu]))
    c1m, c2m = [x / 840.0 / ax.hmu for x in _D1], [x / 5040.0 / ax.hmu ** 2 for x in _D2]
    c1n, c2n = [x / 840.0 / ax.hni for x in _D1], [x / 5040.0 / ax.hni ** 2 for x in _D2]
    for _ in range(sweeps):
        for p, l, rr, bp, dp in idx:
            acc = 0.0
            for i, k in enumerate((4, 3, 2, 1)):
                m, q = a[:, p - k * n8], a[:, p + k * n8]
                acc = acc + c2m[i] * (m + q) + bp * (c1m[i] * (m - q))
                m, q = a[:, p - k], a[:, p + k]
                acc = acc + c2n[i] * (m + q) + dp * (c1n[i] * (m - q))
            a[:, p] = omega * (rr - acc) / l + (1.0 - omega) * a[:, p]
        t = torch.from_numpy(a.reshape(w.shape))
        for q, s in enumerate(isym):
            _boundary(ax, t[q:q + 1], s)
    return torch.from_numpy(a.reshape(w.shape))


def _exact_group(case, d):
    ax, count = d["ax"], d["u"].shape[0]
    b = ax.borb if d["bkind"] == 0 else ax.bpot
    rhs, u = _rhs(d), d["u"].clone()
    lhs = [d["lhs"][k] for k in d["lhs_of"]]
    if case["kind"] == "ordered":
        w = torch.stack([_embed(u[q][None], d["isym"][q])[0] for q in range(count)])
        w = _sequential(ax, w, lhs, rhs, b, d["isym"], d["omega"], case["sweeps"], case["method"], case["ordering"])
        return w[:, 4:-4, 4:-4]
    for s in (1, -1):
        sel = [q for q in range(count) if d["isym"][q] == s]
        if not sel:
            continue
        w = _embed(u[sel], s)
        _mcsor(ax, w, torch.stack([lhs[q] for q in sel]), rhs[sel], b, s, d["omega"], case["sweeps"])
        u[sel] = w[:, 4:-4, 4:-4]
    if d["fock1"] is not None:  # the asymptotic tail of an orbital
        nmu = ax.nmu
        fa = (d["fock1"] / ax.f1)[:, -5:]
        rr = torch.sqrt(ax.xi ** 2 + ax.eta ** 2 - 1.0)[-5:]
        for k in range(4):
            ed = (fa[:, k + 1] / fa[:, k]).abs() ** 0.25 * torch.exp(fa[:, k].abs().sqrt() * (rr[k] - rr[k + 1]))
            u[:, nmu - 4 + k] = u[:, nmu - 5 + k] * ed
    return u


def _exact_fock(case, seed):
    out = {"orb": [], "fock": [], "scal": None}
    norb = case["norb"]
    scal = torch.zeros(2, case["jobs"], norb, dtype=torch.float64)
    for q in range(case["jobs"]):
        d = _fock_inputs(case, seed, q)
        ax, orb = d["ax"], d["orb"].clone()
        wgt1, wgt2 = ax.weights()
        f = torch.zeros(4, *orb.shape, dtype=torch.float64, device=orb.device)
        for i in range(norb):
            for j in range(norb):
                f[0, i] += d["coo"][i][j] * d["coul"][j]
                if j != i:
                    f[1, i] += d["exch"][d["slot"][i][j]] * d["orb"][j]
            f[2, i] = ax.f0 + d["eps"][i] * ax.f1 + d["m"][i] * ax.e + ax.f2 * f[0, i]
            f[3, i] = f[2, i] + ax.diag
        w = wgt2 * ax.f4
        for i in reversed(range(norb)):
            s = (w * orb[i] ** 2).sum()
            scal[0, q, i] = s
            others = [j for j in range(i + 1, norb) if d["m"][j] == d["m"][i]]
            ov = [(w * orb[i] * orb[j]).sum() / s.sqrt() for j in others]
            a = sum((o * o for o in ov), torch.zeros_like(s))
            new = orb[i] / s.sqrt() - sum((o * orb[j] for o, j in zip(ov, others)), torch.zeros_like(orb[i]))
            orb[i] = torch.sqrt(1.0 + a) / (1.0 - a * a) * new
        for i in range(norb):
            m, psi = d["m"][i], orb[i]
            t = _operator(ax, _embed(psi[None], -1 if m else 1), ax.borb)[0] + ax.diag * psi + m * ax.e * psi
            scal[1, q, i] = ((wgt1 * psi * (t + ax.f0 * psi)).sum() +
                             (wgt2 * (psi * f[0, i] * psi - psi * f[1, i])).sum())
        out["orb"].append(orb)
        out["fock"].append(f)
    out["scal"] = scal
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "mcsor":
        ax, u, lhs, rhs, om = _mcsor_inputs(case, seed)
        w = _embed(u[None], case["isym"])
        _mcsor(ax, w, lhs[None], rhs[None], ax.borb if case["bkind"] == 0 else ax.bpot, case["isym"], om,
               case["sweeps"])
        return w[0]
    if kind == "relax":
        return [_exact_group(case, _relax_group(case, *g, seed, k)) for k, g in enumerate(_groups(case["grids"]))]
    if kind == "ordered":
        return [_exact_group(case, _relax_group(case, case["nni"], case["nmu"], case["count"], seed, 0))]
    if kind == "fock":
        return _exact_fock(case, seed)
    return None  # a whole SCF: no closed form in reach


# ---------------------------------------------------------------------------
# what one pass cannot do without

_POINT = 36  # operations of one point update of the 17-point cross


def work(case):
    kind = case["kind"]
    if kind == "mcsor":  # read the function, lhs, rhs; write the function
        n = case["nni"] * case["nmu"]
        return {"bytes": 32.0 * n, "flops": float(_POINT * n * case["sweeps"])}
    if kind in ("relax", "ordered"):
        groups = _groups(case["grids"]) if kind == "relax" else [(case["nni"], case["nmu"], case["count"])]
        by = fl = 0.0
        for nni, nmu, count in groups:
            n = nni * nmu
            fl += _POINT * n * case["sweeps"] * count
            # each function once in and out; a job's lhs (one per |dm|) and
            # its orbitals once, or an array rhs per item
            by += 16.0 * n * count
            if case.get("what") == "orb":
                by += 16.0 * n * count
            else:
                ns, pairs = _pairs(count)
                by += 8.0 * n * (1 + any(j < 0 for _, j in pairs))
                by += 8.0 * n * (ns + 2 if case.get("prec") == 1 else count)
        return {"bytes": by, "flops": fl}
    if kind == "fock":
        n, norb = case["nni"] * case["nmu"], case["norb"]
        arrays = 2 * norb + norb + norb * (norb - 1) // 2 + 4 * norb + 8  # orbitals in/out, J, K, operators, grid
        flops = norb * (2 * norb + 3 * norb + 12 + 8 * norb + 60)
        return {"bytes": 8.0 * n * arrays * case["jobs"], "flops": float(flops * n * case["jobs"])}
    n = case["nni"] * case["nmu"] * case["jobs"] * case["iters"]
    norb = {"h2": 1, "lih": 2, "mix": 2}[case["mol"]]
    npot = norb * (norb + 1) // 2
    return {"bytes": 8.0 * n * (2 * norb + 2 * npot + 4), "flops": float(_POINT * 10 * n * (norb + npot))}
