"""The update's sums over r per strip segment, added up over the waves of a block
and over a strip's segments: flux-line samples and derivatives of one step against
the same sums of the state it leaves, whole strips in one block and strips cut
over waves and blocks, one and two R per lane, in both precisions (the state is
FP64 in both, so the sums agree to their rounding: n1 2^-53 of the terms' sizes,
1e-13 with C_k(E))."""
import numpy as np
import pytest

from madwave3_amd import leps
from madwave3_amd.lib import MW3_FP64, MW3_MIXED, Propagator
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

# npun1, npun2, nangu, Jtot
SIZES = [
    (64, 64, 4, 0),
    (150, 96, 6, 0),
    (48, 512, 40, 0),
    (96, 512, 60, 0),
    (70, 333, 50, 0),
    (100, 160, 44, 1),
]


def wanted(c, o, psi, k):
    """zCR, zCdR of one step whose new psi is `psi`, and the size of zCdR's terms."""
    t = o.tables()
    za, ck = t["zAR1flux"], o.coef_echeby(k, c.etotS2)
    zr, zd, size, at = [], [], [], 0
    for sl in range(c.nangu):
        ia = int(c.indangreal[sl]) - 1
        n = int(c.npunreal[ia])
        i1, i2 = c.indr1[ia, :n].astype(int), c.indr2[ia, :n].astype(int)
        line = np.nonzero(i1 == t["ir1flux"][ia])[0]
        for _ in range(c.ncan):
            p = psi[at:at + n]
            at += n
            s, a = np.zeros(c.npun2 + 1, complex), np.zeros(c.npun2 + 1)
            np.add.at(s, i2, za[i1 - 1] * p)
            np.add.at(a, i2, np.abs(za[i1 - 1] * p))
            zr.append(p[line])
            zd.append(s[i2[line]])
            size.append(a[i2[line]])
    zr, zd = np.concatenate(zr), np.concatenate(zd)
    return (zr[:, None] * ck, zd[:, None] * ck,
            np.max(np.concatenate(size)) * np.max(np.abs(ck)))


@pytest.mark.parametrize("prec", [MW3_FP64, MW3_MIXED])
@pytest.mark.parametrize("n1,n2,na,J", SIZES)
def test_segment_sums(n1, n2, na, J, prec):
    p = leps.config(4, J=J) if J else leps.config(1)
    p.update(npun1=n1, npun2=n2, nangu=na, npun1min=8, jmax=min(5, na - 1), nvmax=2, netot=10,
             iprod=0, kminelastic=4, width_bohr=0.6, absorb_bohr=4.5)
    if J:
        p.update(Jtot=J, iommin=0, iommax=J, iomref=-1, iparity=-1)
    c = leps.build(p)
    print("case", (n1, n2, na, J, prec), c, flush=True)
    o = Oracle(c)
    psi0 = np.random.default_rng(n2).standard_normal(c.ntot)
    g = Propagator(c, prec)
    g.flux_energy_test(0)
    g.begin(psi0 / np.linalg.norm(psi0))
    norm = g.steps(1)[0]
    _, psi, k = g.state()
    a, b = g.flux_accum()
    wa, wb, size = wanted(c, o, psi, k)
    assert a.shape == wa.shape and np.max(np.abs(wa)) > 0.0
    assert np.max(np.abs(a - wa)) <= 1e-13 * np.max(np.abs(wa))
    assert np.max(np.abs(b - wb)) <= 1e-13 * size
    assert abs(norm[0] - np.sum(psi * psi)) <= 1e-12 * norm[0]
