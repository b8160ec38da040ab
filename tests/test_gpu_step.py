"""The update with the radial r products and its R-product kernel
(madwave3_amd/csrc/mw3_step.h) at the edges of their tiles: r sizes one off a
16-row tile, odd and unaligned R sizes, one and several mode tiles, a block per
strip and runs over many strips, and a grid whose low modes do not fit (batched
GEMMs).  Bars as in test_gpu_parity: FP64 to rounding (1e-11 on H psi, 1e-10 on
the recursion, 1e-9 on the energy sums), mixed 2e-5 on H psi."""
import numpy as np
import pytest

from madwave3_amd import leps
from madwave3_amd.lib import MW3_FP64, MW3_MIXED, MW3_OPT_RADIAL, Propagator
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


def rel(a, b):
    a, b = np.asarray(a), np.asarray(b)
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300))


# npun1, npun2, nangu, Jtot, box (bohr, both), radial kernels (else GEMMs)
SIZES = [
    (16, 32, 4, 0, None, 1),
    (17, 48, 5, 0, None, 1),
    (31, 50, 6, 0, None, 1),
    (33, 37, 7, 2, None, 1),
    (48, 64, 4, 0, None, 1),
    (64, 75, 5, 1, None, 1),
    (80, 272, 4, 0, None, 1),
    (20, 320, 60, 0, None, 1),
    (100, 96, 4, 0, 12.0, 1),
]


@pytest.mark.parametrize("n1,n2,na,J,box,radial", SIZES)
def test_step_matches_oracle(n1, n2, na, J, box, radial):
    p = leps.config(4, J=J) if J else leps.config(1)
    p.update(npun1=n1, npun2=n2, nangu=na, npun1min=8, jmax=min(5, na - 1), nvmax=2, netot=30,
             iprod=0, kminelastic=4, width_bohr=0.6, absorb_bohr=4.5)
    if J:
        p.update(Jtot=J, iommin=0, iommax=J, iomref=-1, iparity=1 if J % 2 == 0 else -1)
    if box:
        p.update(rfin1_bohr=box)
    c = leps.build(p)
    print("case", (n1, n2, na, J, box), c, flush=True)
    o = Oracle(c)
    rng = np.random.default_rng(n1 * 1000 + n2)
    psi = rng.standard_normal(c.ntot)
    h = o.hphi(psi)
    g = Propagator(c, MW3_FP64)
    assert g.get_option(MW3_OPT_RADIAL) == radial
    assert rel(g.hphi(psi), h) < 1e-11
    m = Propagator(c, MW3_MIXED)
    assert m.get_option(MW3_OPT_RADIAL) == radial
    assert rel(m.hphi(psi), h) < 2e-5
    o.begin(c.rpaq0)
    g.begin(c.rpaq0)
    n_o = o.steps(20)[0]
    n_g = np.concatenate([g.steps(1)[0], g.steps(19)[0]])  # G formed anew, then left by the update
    assert rel(n_g, n_o) < 1e-10
    assert rel(g.state()[1], o.state()[1]) < 1e-10
    assert rel(g.flux_result()[0], o.flux_result()[0]) < 1e-9
    assert rel(g.zs2(), o.zs2()) < 1e-9


@pytest.mark.parametrize("n1,n2", [(2048, 16), (2049, 18), (4096, 16)])
def test_longest_r(n1, n2):
    """The factors of the r rows in LDS: the longest r with the r products in the
    update, the first without, and the longest there is."""
    p = leps.config(1)
    p.update(npun1=n1, npun2=n2, nangu=2, npun1min=8, jmax=1, nvmax=2, netot=30, iprod=0,
             kminelastic=4, width_bohr=0.6, absorb_bohr=4.5)
    c = leps.build(p)
    o = Oracle(c)
    psi = np.random.default_rng(n1).standard_normal(c.ntot)
    h = o.hphi(psi)
    o.begin(c.rpaq0)
    n_o = o.steps(20)[0]
    for prec, bar in ((MW3_FP64, 1e-11), (MW3_MIXED, 2e-5)):
        g = Propagator(c, prec)
        assert rel(g.hphi(psi), h) < bar
        g.begin(c.rpaq0)
        assert rel(g.steps(20)[0], n_o) < 10 * bar
        assert rel(g.state()[1], o.state()[1]) < 10 * bar


@pytest.mark.parametrize("n1,n2,na", [(12, 12, 2), (32, 64, 16), (64, 128, 60)])
def test_begin_sums(n1, n2, na):
    """psi.H psi, psi.psi and H psi.H psi of the initial packet: fewer points than
    a block, than the whole launch, and more (sums of n products: n 2^-53)."""
    p = leps.config(1)
    p.update(npun1=n1, npun2=n2, nangu=na, npun1min=8, jmax=min(5, na - 1), nvmax=2, netot=0,
             iprod=0, kminelastic=4, width_bohr=0.6, absorb_bohr=4.5)
    c = leps.build(p)
    psi = np.random.default_rng(n1).standard_normal(c.ntot)
    g = Propagator(c, MW3_FP64)
    h = g.hphi(psi)
    size = np.array([np.abs(psi * h).sum(), (psi * psi).sum(), (h * h).sum()])
    want = np.array([(psi * h).sum(), (psi * psi).sum(), (h * h).sum()])
    assert np.all(np.abs(g.begin(psi) - want) <= 2.0 * c.ntot * 2.0**-53 * size)


# npun1, npun2, nangu, box r, box R (bohr), radial kernels (else GEMMs)
BEYOND = [
    (120, 256, 4, 20.0, 15.0, 1),   # more low r modes than the update takes: FP64 R passes in LDS
    (128, 256, 4, 20.0, 10.0, 1),
    (112, 320, 4, 20.0, 22.0, 1),
    (96, 384, 5, 18.0, 6.0, 1),
    (100, 512, 4, 18.0, 15.0, 1),
    (2064, 256, 2, 8.0, 15.0, 1),   # more r rows than the update's products take
    (128, 128, 4, 20.0, 15.0, 0),   # neither update nor R passes: GEMMs
    (90, 100, 5, 20.0, 15.0, 0),
    (700, 64, 6, 8.0, 15.0, 1),     # strips cut into many segments, vectorised and not
    (705, 50, 6, 8.0, 15.0, 1),
]


@pytest.mark.parametrize("n1,n2,na,b1,b2,radial", BEYOND)
def test_grids_beyond_the_update(n1, n2, na, b1, b2, radial):
    p = leps.config(1)
    p.update(npun1=n1, npun2=n2, nangu=na, npun1min=8, jmax=1, nvmax=1, netot=30, iprod=0,
             kminelastic=4, width_bohr=0.6, absorb_bohr=4.5, rfin1_bohr=b1, rfin2_bohr=b2)
    c = leps.build(p)
    print("case", (n1, n2, na, b1, b2), c, flush=True)
    o = Oracle(c)
    psi = np.random.default_rng(n1 * 1000 + n2).standard_normal(c.ntot)
    h = o.hphi(psi)
    o.begin(c.rpaq0)
    n_o = o.steps(20)[0]
    for prec, bar in ((MW3_FP64, 1e-11), (MW3_MIXED, 2e-5)):
        g = Propagator(c, prec)
        if prec == MW3_FP64:
            assert g.get_option(MW3_OPT_RADIAL) == radial
        assert rel(g.hphi(psi), h) < bar
        g.begin(c.rpaq0)
        assert rel(g.steps(20)[0], n_o) < 10 * bar
        # (of the packet's size at the start: some boxes have absorbed most of it by now)
        d = np.max(np.abs(g.state()[1] - o.state()[1]))
        assert d < 10 * bar * np.max(np.abs(c.rpaq0))
        g.close()
