"""Performance cases of the propagator: what a user of the library runs, through
its public entry points (madwave3_amd.lib and madwave3_amd.leps).

Kinds of case:
  run       one loop of a propagation: mw3_cheby_begin with the initial packet,
            `steps` damped Chebyshev steps (the configurations' ntimes is 500),
            then the analysis of that loop: P(E), the reactant and product
            S-matrix sums and the state pair of the continuation files
  batch     the same for several total angular momenta stepped together
  hphi      one H psi on host arrays, the drop-in for the reference's difs
  spectrum  the photodissociation spectrum of an autocorrelation

Surfaces and grids come from the synthetic LEPS generator; boxes are in bohr.
A seed changes the initial packet (and the autocorrelation of a spectrum); the
surface, the grid and the operator tables are the program's set-up.
"""
import functools
import math

import numpy as np
import torch

from madwave3_amd import consts, leps
from madwave3_amd import lib as mw3

ANG = 1.0 / 0.529177  # bohr per angstrom


def _run(name, n1, n2, na, precision, steps, **kw):
    d = dict(kind="run", npun1=n1, npun2=n2, nangu=na, precision=precision, steps=steps,
             box1=8.0, box2=15.0, Jtot=0, nelec=1, products=False, netot=500)
    d.update(kw)
    if name:
        d["name"] = name
    return d


def listed():
    return [
        # the reference's own example: HD + H, J = 0, a 20 angstrom box on a
        # coarse grid (most of its modes lie below the kinetic cut)
        _run("hdh_mixed", 256, 256, 140, "mixed", 500, box1=20 * ANG, box2=20 * ANG,
             products=True),
        # the smallest production grid, product states resolved
        _run("small_mixed", 128, 256, 60, "mixed", 500, products=True),
        # the benchmark's grid in both precisions, product states resolved
        _run("bench_mixed", 256, 512, 120, "mixed", 500, products=True),
        _run("bench_fp64", 256, 512, 120, "fp64", 500, products=True),
        # J = 12 with seven Coriolis-coupled helicity blocks
        _run("coriolis_mixed", 192, 384, 96, "mixed", 500, Jtot=12),
        _run("coriolis_fp64", 192, 384, 96, "fp64", 250, Jtot=12),
        # photodissociation on three coupled states (autocorrelation kept),
        # on a grid with an odd number of r points
        _run("photo_mixed", 171, 256, 64, "mixed", 500, nelec=3),
        # FFT-friendly odd sizes (the reference asks for 2^a 3^b 5^c ... only),
        # J = 1 with two helicity blocks
        _run("ragged_fp64", 105, 225, 45, "fp64", 500, Jtot=1),
        # a convergence test's grid: every step is launches and latency
        _run("tiny_fp64", 32, 64, 16, "fp64", 500, products=True, netot=200),
        # several total J on one GPU
        dict(name="batch_mixed", kind="batch", npun1=160, npun2=320, nangu=80,
             precision="mixed", steps=250, Js="0,1,2,3", box1=8.0, box2=15.0, netot=500),
        # one operator application on host arrays
        dict(name="hphi_fp64", kind="hphi", npun1=128, npun2=256, nangu=60, precision="fp64",
             Jtot=0, nelec=1, products=False, box1=8.0, box2=15.0, netot=500),
        # cheby-spectra after a photodissociation run of 30000 steps
        dict(name="spectrum", kind="spectrum", kmax=30000, ne=2000),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["run"] * 8 + ["batch", "hphi", "spectrum"])
    if kind == "spectrum":
        return dict(kind=kind, kmax=_logint(rng, 500, 60000), ne=_logint(rng, 100, 2000))
    n1, n2, na = _logint(rng, 32, 256), _logint(rng, 64, 512), _logint(rng, 16, 140)
    box1, box2 = 8.0, 15.0
    if min(n1, n2) >= 128 and rng.random() < 0.3:
        box1 = box2 = rng.uniform(18.0, 38.0)
    precision = rng.choice(["mixed", "fp64"])
    netot = rng.choice([100, 200, 500])
    if kind == "batch":
        n1, n2, na = min(n1, 160), min(n2, 320), min(na, 80)
        return dict(kind=kind, npun1=n1, npun2=n2, nangu=na, precision=precision,
                    steps=rng.randint(20, 250), Js=rng.choice(["0,1", "0,1,2", "1,2"]),
                    box1=8.0, box2=15.0, netot=netot)
    nelec = 1
    Jtot = rng.choice([0, 0, 0, 1, 2, 4, 12])
    if Jtot == 0 and rng.random() < 0.25:
        nelec, n1, n2, na = 3, min(n1, 171), min(n2, 256), min(na, 64)
    elif Jtot:
        n1, n2, na = min(n1, 192), min(n2, 384), min(na, 96)
    products = nelec == 1 and Jtot == 0 and rng.random() < 0.6
    if kind == "hphi":
        return dict(kind=kind, npun1=n1, npun2=n2, nangu=na, precision=precision, Jtot=Jtot,
                    nelec=nelec, products=False, box1=box1, box2=box2, netot=netot)
    return _run(None, n1, n2, na, precision, rng.randint(20, 250), box1=box1, box2=box2,
                Jtot=Jtot, nelec=nelec, products=products, netot=netot)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _params(npun1, npun2, nangu, box1, box2, Jtot, nelec, products, netot):
    if nelec == 3:
        p = leps.config(5)
    elif Jtot:
        p = leps.config(4, J=Jtot)
        p.update(Jtot=Jtot, iommin=Jtot % 2 if Jtot > 1 else 0, iommax=min(Jtot, 6), iomref=-1)
        if Jtot == 1:
            p.update(iparity=-1)  # Omega = 0 and 1
    else:
        p = leps.config(1)
    p.update(npun1=npun1, npun2=npun2, nangu=nangu, rfin1_bohr=box1, rfin2_bohr=box2,
             npun1min=min(32, npun1 // 2), netot=netot, iprod=2 if products else 0,
             width_bohr=0.6, absorb_bohr=4.5)  # a packet that reaches the analysis line
    p["jmax"] = min(p["jmax"], nangu - 1)
    p["jmaxprod"] = min(p["jmaxprod"], nangu - 1)
    if box1 > 9.0:  # the 20 angstrom example: absorb over the outer part
        p.update(absorb_bohr=0.6 * box1, nexpo=2, R0_bohr=5.2 * ANG, ecol_eV=0.62,
                 Rbalinprod_bohr=min(6.0 * ANG, 0.4 * box1), r1flux_bohr=4.0 * ANG, nvmax=5,
                 jmax=min(39, nangu - 1), nvmaxprod=10, jmaxprod=min(20, nangu - 1))
    return p


@functools.lru_cache(maxsize=6)
def _built(*key):
    return leps.build(_params(*key))


def _cases(case):
    Js = [int(j) for j in case["Js"].split(",")] if case["kind"] == "batch" else [case["Jtot"]]
    return [_built(case["npun1"], case["npun2"], case["nangu"], case["box1"], case["box2"], J,
                   case.get("nelec", 1), case.get("products", False), case["netot"]) for J in Js]


def _packet(c, seed):
    """The case's initial packet with a seeded long-wave modulation along r, R
    and gamma, normalised."""
    rng = np.random.default_rng(seed)
    q = rng.uniform(0.5, 3.0, 3)
    ph = rng.uniform(0.0, 2.0 * math.pi, 3)
    w = []
    for sl in range(c.nangu):
        ia = int(c.indangreal[sl]) - 1
        n = int(c.npunreal[ia])
        m = 1.0 + 0.3 * np.cos(q[0] * 2 * math.pi * c.indr1[ia, :n] / c.npun1 + ph[0])
        m = m + 0.3 * np.cos(q[1] * 2 * math.pi * c.indr2[ia, :n] / c.npun2 + ph[1])
        m = m * (1.0 + 0.2 * math.cos(q[2] * 2 * math.pi * ia / c.nangu + ph[2]))
        w += [m] * c.ncan
    x = np.ascontiguousarray(c.rpaq0 * np.concatenate(w))
    return x / math.sqrt(float(np.sum(x * x)))


def _autocorrelation(case, seed):
    """A decaying autocorrelation of a few levels, and the spectrum's energies."""
    rng = np.random.default_rng(seed)
    k = np.arange(case["kmax"] + 1)
    th = rng.uniform(0.4, 2.6, 12)
    a = rng.uniform(0.1, 1.0, 12)
    auto = (a[:, None] * np.cos(th[:, None] * k)).sum(0) / a.sum()
    auto *= np.exp(-3.0 * k / case["kmax"])
    emindlt, delta2 = 1.1, 2.3
    e = np.linspace(emindlt - 0.9 * delta2, emindlt + 0.9 * delta2, case["ne"])
    return auto, e, emindlt, delta2, 1.0 / case["kmax"]


def prepare(case, seed):
    if case["kind"] == "spectrum":
        return dict(kind="spectrum", args=_autocorrelation(case, seed))
    prec = mw3.MW3_MIXED if case["precision"] == "mixed" else mw3.MW3_FP64
    cs = _cases(case)
    st = dict(kind=case["kind"], props=[mw3.Propagator(c, prec) for c in cs])
    if case["kind"] == "hphi":
        st["psi"] = np.random.default_rng(seed).standard_normal(cs[0].ntot)
        return st
    st["steps"] = case["steps"]
    st["psi0"] = [_packet(c, seed + 7919 * i) for i, c in enumerate(cs)]
    return st


def _results(p):
    tot, elec = p.flux_result()
    out = dict(P=tot, Pelec=elec, zs2=p.zs2())
    if mw3.has_prod_tables(p.case):
        out["zs2prod"] = p.zs2prod()
    out["psim1"], out["psi"], _ = p.state()
    return out


def run(state):
    if state["kind"] == "spectrum":
        auto, e, emindlt, delta2, xk = state["args"]
        return mw3.cheby_spectrum(auto, emindlt, delta2, consts.hbr, xk, e)
    if state["kind"] == "hphi":
        return state["props"][0].hphi(state["psi"])
    for p, x in zip(state["props"], state["psi0"]):
        p.begin(x)
    if state["kind"] == "batch":
        norms = mw3.steps_batch(state["props"], state["steps"])
        return [dict(_results(p), norms=norms[i]) for i, p in enumerate(state["props"])]
    p = state["props"][0]
    photo = p.case.iphoto >= 1
    norms, auto = p.steps(state["steps"], want_auto=photo)
    out = dict(_results(p), norms=norms)
    if photo:
        out["auto"] = auto
    return out


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _fft_size(span, nmax, nmin):
    n = span
    while n <= nmax:
        m = n
        for f in (2, 3, 5, 7, 11):
            while m % f == 0:
                m //= f
        if m == 1:
            break
        n += 1
    return max(min(n, nmax), nmin)


def _momenta(n, ah, mu):
    p = math.pi * np.arange(1, n + 1) / ((n + 1) * ah)
    return 0.5 * consts.hbr ** 2 / mu * p * p


def _step_work(c, precision):
    """(bytes, flops) of one step: psi_k, psi_{k-1} and V read and psi_{k+1}
    written at the kept points; the low-mode kinetic products at the kept
    points and the (folded) angular products over the kept columns."""
    sv = 4 if precision == "mixed" else 8
    nk = int(c.npunreal.sum())
    k1 = int((_momenta(c.npun1, c.ah1, c.xm1red) < c.radcutmax).sum())
    k2 = int((_momenta(c.npun2, c.ah2, c.xm2red) < c.radcutmax).sum())
    cols = np.zeros(c.npun1 * c.npun2, dtype=bool)
    for ia in range(c.nangu):
        n = int(c.npunreal[ia])
        cols[(c.indr1[ia, :n].astype(np.int64) - 1) * c.npun2 + c.indr2[ia, :n] - 1] = True
    fold = 2 if c.nangu % 2 == 0 else 1
    kmin = min(k1 * c.npun1, k2 * c.npun2) / (c.npun1 if k1 * c.npun1 <= k2 * c.npun2
                                              else c.npun2)
    flops = c.ncan * (4.0 * nk * kmin + 4.0 * c.nangu * k1 * c.npun2 * k2 / 2
                      + 4.0 * c.nangu * c.nangu * int(cols.sum()) / fold + 12.0 * nk)
    byts = c.ncan * nk * 24.0 + c.nelecmax ** 2 * nk * sv
    if mw3.has_prod_tables(c):
        byts += nk * sv
        flops += 2.0 * nk
    return byts, flops


def work(case):
    if case["kind"] == "spectrum":
        n = float(case["kmax"]) * case["ne"]
        return dict(bytes=8.0 * (case["kmax"] + 2 * case["ne"]), flops=20.0 * n)
    cs = _cases(case)
    if case["kind"] == "hphi":
        c = cs[0]
        b, f = _step_work(c, case["precision"])
        return dict(bytes=b, flops=f)
    byts = flops = 0.0
    for c in cs:
        b, f = _step_work(c, case["precision"])
        nfl = c.ncan * c.nangu * c.npun2 * 0.5
        byts += case["steps"] * b + 3 * 8.0 * c.ntot
        flops += case["steps"] * (f + 12.0 * nfl * c.netot)
    return dict(bytes=byts, flops=flops)


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------
class _Exact:
    """The operator and the recursion as plain dense products in float64."""

    def __init__(self, c, dev):
        self.c, self.dev = c, dev
        T = functools.partial(torch.as_tensor, dtype=torch.float64, device=dev)
        self.T = T
        n1, n2, na, nc, ne = c.npun1, c.npun2, c.nangu, c.ncan, c.nelecmax
        hb, mu1, mu2 = consts.hbr, c.xm1red, c.xm2red
        pl = n1 * n2
        idx, mask = [], np.zeros((na, pl), dtype=bool)
        V = np.zeros((ne, ne, na, pl))
        groups = {}
        for sl in range(na):
            ia = int(c.indangreal[sl]) - 1
            n = int(c.npunreal[ia])
            i1 = c.indr1[ia, :n].astype(np.int64)
            p = (i1 - 1) * n2 + c.indr2[ia, :n].astype(np.int64) - 1
            mask[ia, p] = True
            V[:, :, ia, p] = c.VVV[:, :, sl, :n]
            idx += [(ch * na + ia) * pl + p for ch in range(nc)]
            groups.setdefault(_fft_size(int(i1.max() - i1.min()) + 1, n1, c.npun1min),
                              []).append(ia)
        self.idx = torch.as_tensor(np.concatenate(idx), device=dev)
        self.mask = T(mask).reshape(na, n1, n2)
        self.V = T(V).reshape(ne, ne, na, n1, n2)

        def dst(n):
            m = np.outer(np.arange(1, n + 1), np.arange(1, n + 1)) % (2 * (n + 1))
            return T(2.0 * np.sin(math.pi * m / (n + 1)))
        self.SR = dst(n2)
        p2 = _momenta(n2, c.ah2, mu2)
        self.rad = []
        for n, ias in sorted(groups.items()):
            e = np.minimum(_momenta(n, c.ah1, mu1)[:, None] + p2, c.radcutmax)
            self.rad.append((n, torch.as_tensor(ias, device=dev), dst(n),
                             T(e / (4.0 * (n + 1) * (n2 + 1)))))
        # angular functions and coefficients
        nJ = (na - 1) * c.inc + 1
        r1 = c.rmis1 + np.arange(n1) * c.ah1
        r2 = c.rmis2 + np.arange(n2) * c.ah2
        self.D = T(np.stack([c.Djmmp[c.iombas[h], c.nelebas[h] - 1, :nJ] for h in range(nc)]))
        a = np.zeros((nc, nJ, n1))
        for h in range(nc):
            om = int(c.iomdiat[c.nelebas[h] - 1])
            for k in range(int(c.nojbas[h])):
                j = int(c.jbas[h, k])
                if j < nJ:
                    x = (j * (j + 1.0) - om * om) * hb * hb * 0.5 / (mu1 * r1 * r1)
                    a[h, j] += np.minimum(x, c.rotcutmax)
        chan = {(int(c.nelebas[h]), int(c.iombas[h])): h for h in range(nc)}
        b = {}
        J, par = c.Jtot, 1 if c.Jtot % 2 == 0 else -1
        for e in range(1, ne + 1):
            sig = -1 if c.sigdiat[e - 1] == -1.0 or c.sigatom[e - 1] == -1.0 else 1
            for j in range(c.j0, nJ, c.inc):
                lo = 1 if c.iparity != sig * par and c.iommin == 0 else c.iommin
                hi = min(j, c.iommax)
                if lo > hi:
                    continue
                om = np.arange(lo, hi + 1)
                m = np.diag(j * (j + 1.0) + J * (J + 1) - 2.0 * om * om)
                for q in range(len(om) - 1):
                    w = om[q] * om[q + 1]
                    x = -math.sqrt((J * (J + 1.0) - w) * (j * (j + 1.0) - w))
                    m[q, q + 1] = m[q + 1, q] = x * (math.sqrt(2.0) if w == 0 else 1.0)
                m = m * (hb * hb * 0.5 / mu2)
                ev = np.linalg.eigvalsh(m)
                mean = 0.5 * (ev[0] + ev[-1])
                re2 = np.where(mean / (r2 * r2) > c.rotcutmax, abs(mean / c.rotcutmax), r2 * r2)
                for x in range(len(om)):
                    for y in range(max(0, x - 1), min(len(om), x + 2)):
                        t, s = chan.get((e, int(om[x]))), chan.get((e, int(om[y])))
                        if t is None or s is None or abs(m[x, y]) <= 1e-8:
                            continue
                        b.setdefault((t, s), np.zeros((nJ, n2)))[j] += np.where(
                            re2 > 1e-6, m[x, y] / re2, 0.0)
        self.a = T(a)
        self.b = {k: T(v) for k, v in b.items()}
        self.f = T(c.absfr1)[:, None] * T(c.absfr2)[None, :]

    def dense(self, a0):
        c = self.c
        x = torch.zeros(c.ncan * c.nangu * c.npun1 * c.npun2, dtype=torch.float64,
                        device=self.dev)
        x[self.idx] = self.T(a0)
        return x.reshape(c.ncan, c.nangu, c.npun1, c.npun2)

    def packed(self, x):
        return x.reshape(-1)[self.idx].cpu().numpy()

    def h(self, x):
        c = self.c
        nc, na, n1, n2 = x.shape
        out = torch.empty_like(x)
        y = x.reshape(-1, n2).matmul(self.SR).reshape(x.shape)
        for n, ias, S, kin in self.rad:
            z = torch.matmul(S, y[:, ias, :n]) * kin
            z = torch.matmul(S, z)
            out[:, ias, :n] = z.reshape(-1, n2).matmul(self.SR).reshape(z.shape)
            if n < n1:
                out[:, ias, n:] = x[:, ias, n:]
        F = [self.D[h].matmul(x[h].reshape(na, -1)).reshape(-1, n1, n2) for h in range(nc)]
        for h in range(nc):
            G = self.a[h][:, :, None] * F[h]
            for s in range(nc):
                if (h, s) in self.b:
                    G += self.b[h, s][:, None, :] * F[s]
            out[h] += self.D[h].t().matmul(G.reshape(G.shape[0], -1)).reshape(na, n1, n2)
            for s in range(nc):
                if c.iombas[s] == c.iombas[h]:
                    out[h] += self.V[c.nelebas[h] - 1, c.nelebas[s] - 1] * x[s]
        return out * self.mask

    def propagate(self, psi0, steps):
        """begin, steps and the analysis, laid out as _results returns them."""
        c, T = self.c, self.T
        nc, na, n1, n2 = c.ncan, c.nangu, c.npun1, c.npun2
        # flux line: d/dr by a Fourier derivative at the last r <= r1flux
        r1 = c.rmis1 + np.arange(n1) * c.ah1
        i4 = int((r1 <= c.r1flux).sum())
        m = np.arange(n1)
        xk = 2.0 * math.pi * np.where(m + 1 <= n1 // 2, m, m - n1) / (n1 * c.ah1)
        arg = xk[None, :] * ((i4 - 1 - m) * c.ah1)[:, None]
        zar = T(np.stack([-(xk * np.sin(arg)).sum(1), (xk * np.cos(arg)).sum(1)]) / (2.0 * n1))
        fl, pot, fe = [], [], []
        for sl in range(na):
            ia = int(c.indangreal[sl]) - 1
            n = int(c.npunreal[ia])
            i1 = c.indr1[ia, :n]
            ok = (i1 - 1) * c.ah1 + c.rmis1 <= c.r1flux
            sel = np.nonzero(i1 == (i1[ok].max() if ok.any() else -1))[0]
            for h in range(nc):
                e = int(c.nelebas[h]) - 1
                fl += [((h * na + ia), int(i1[q]) - 1, int(c.indr2[ia, q]) - 1) for q in sel]
                pot += list(c.VVV[e, e, sl, sel])
                fe += [e] * len(sel)
        fl = torch.as_tensor(np.array(fl, dtype=np.int64).reshape(-1, 3), device=self.dev)
        # reactant states
        nj, nv = c.jmax - c.jini + 1, c.nvmax - c.nvini + 1
        dj, fd = np.zeros((nc, nj, na)), np.zeros((nc, nj, nv, n1))
        late = np.zeros((nc, nj, nv), dtype=bool)
        for h in range(nc):
            e = int(c.nelebas[h]) - 1
            for j in range(int(c.j00[h]), c.jmax + 1, c.inc):
                if j < c.jini:
                    continue
                dj[h, j - c.jini] = c.Djmmp[c.iombas[h], e, j]
                for v in range(c.nvini, min(c.nvmax, int(c.noBCstates[e, j - c.jini])) + 1):
                    fd[h, j - c.jini, v - c.nvini] = c.fd[e, j - c.jini, v - c.nvini]
                    late[h, j - c.jini, v - c.nvini] = (
                        v == c.nvref and j == c.jref and c.iphoto == 0 and c.iprod != 1
                        and (c.iomref < 0 or h + 1 == c.icanref))
        dj, fd = T(dj), T(fd)
        prod = mw3.has_prod_tables(c)
        if prod:
            a0, a1 = c.nangproj0 - 1, c.nangproj1
            b0, b1 = c.n2prod0 - 1, c.n2prod1
            tr = self.dense(c.transRgjac)
            L = (a1 - a0) * (b1 - b0)
            nom, njp, nvp = mw3.prod_shape(c)
            dt = T(c.dtrans).reshape(nc, nom, L)
            wf = np.array(c.prodwf, dtype=np.float64).reshape(nom, njp, nvp, c.nelecmax, L)
            for o in range(nom):
                for j in range(njp):
                    for v in range(nvp):
                        if (j + c.jiniprod < o + c.iomminprod
                                or v + c.nviniprod > c.noBCprod[j]):
                            wf[o, j, v] = 0.0
            wf = T(wf)
        p0 = self.dense(psi0)
        pm, p = p0, (self.h(p0) - c.emindlt * p0) / c.delta2
        norms, autoc, zr, zd, cv, cp = [], [], [], [], [], []
        for _ in range(steps):
            hn = (self.h(p) - c.emindlt * p) / c.delta2
            pm, p = p, (2.0 * hn - self.f * pm) * self.f * self.mask
            norms.append((p * p).sum())
            autoc.append((p0 * p).sum())
            q = p.reshape(nc * na, n1, n2)
            zr.append(q[fl[:, 0], fl[:, 1], fl[:, 2]])
            s = torch.matmul(zar, q)
            zd.append(s[fl[:, 0], :, fl[:, 2]])
            x = torch.matmul(dj, p[:, :, :, c.ir2abs - 1]) / math.sqrt(c.ah2)
            cv.append((fd * x[:, :, None, :]).sum(-1))
            if prod:
                fp = (tr * p).sum(2)[:, a0:a1, b0:b1].reshape(nc, 1, L) * dt
                fe_ = torch.stack([sum(fp[h] for h in range(nc) if c.nelebas[h] - 1 == e)
                                   for e in range(c.nelecmax)], 1)
                cp.append((wf * fe_[:, None, None]).sum((-1, -2)))
        E = T(c.etotS2)
        es = (E - c.emindlt) / c.delta2
        k = torch.arange(2, steps + 2, dtype=torch.float64, device=self.dev)
        ck = 2.0 * consts.hbr / c.delta2 / torch.sqrt(1.0 - es * es)
        ph = k[:, None] * torch.acos(es)
        C, S = ck * torch.cos(ph), -ck * torch.sin(ph)
        out = dict(norms=torch.stack(norms), auto=torch.stack(autoc))
        zr, zd = torch.stack(zr), torch.stack(zd)
        ar, ai = zr.t().matmul(C), zr.t().matmul(S)
        dr, di = zd[:, :, 0].t(), zd[:, :, 1].t()
        br, bi = dr.matmul(C) - di.matmul(S), dr.matmul(S) + di.matmul(C)
        v = (ar * bi - ai * br) * (E > T(np.array(pot))[:, None])
        f = T(c.reacfct) / c.ah1
        fe = torch.as_tensor(np.array(fe, dtype=np.int64), device=self.dev)
        out["Pelec"] = torch.stack([(v * (fe == e)[:, None]).sum(0) * f
                                    for e in range(c.nelecmax)])
        out["P"] = v.sum(0) * f
        cv = torch.stack(cv).reshape(steps, -1)
        skip = torch.as_tensor(late.reshape(-1), device=self.dev)[None, :] * (
            k < c.kminelastic)[:, None]
        cv = torch.where(skip, torch.zeros_like(cv), cv)
        out["zs2"] = torch.complex(cv.t().matmul(C), cv.t().matmul(S)).reshape(nc, nj, nv, -1)
        if prod:
            cp = torch.stack(cp).reshape(steps, -1)
            out["zs2prod"] = torch.complex(cp.t().matmul(C),
                                           cp.t().matmul(S)).reshape(nom, njp, nvp, -1)
        out = {n: t.cpu().numpy() for n, t in out.items()}
        out["psim1"], out["psi"] = self.packed(pm), self.packed(p)
        if c.iphoto < 1:
            del out["auto"]
        return out


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if case["kind"] == "spectrum":
        auto, e, emindlt, delta2, xk = _autocorrelation(case, seed)
        k = torch.arange(1, case["kmax"] + 1, dtype=torch.float64, device=dev)
        a = 2.0 * consts.hbr * torch.exp(-k * xk) * torch.as_tensor(auto[1:], device=dev)
        es = (torch.as_tensor(e, device=dev) - emindlt) / delta2
        th = torch.acos(es)
        s = torch.stack([(a * torch.cos(k * t)).sum() for t in th])
        s = (auto[0] * consts.hbr + s) / (torch.sqrt(1.0 - es * es) * delta2)
        return s.cpu().numpy()
    cs = _cases(case)
    if case["kind"] == "hphi":
        x = _Exact(cs[0], dev)
        psi = np.random.default_rng(seed).standard_normal(cs[0].ntot)
        return x.packed(x.h(x.dense(psi)))
    res = []
    for i, c in enumerate(cs):
        x = _Exact(c, dev)
        res.append(x.propagate(_packet(c, seed + 7919 * i), case["steps"]))
        del x
    return res if case["kind"] == "batch" else res[0]
