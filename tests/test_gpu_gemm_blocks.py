"""The batched GEMMs' block lists (results and k ranges limited to the kept
points) against the oracle: the radial and angular terms as GEMMs on grids whose
kept points fill them, are few, or lie in part of an angle's rows, with sizes the
vector kernel takes and sizes it does not.  Bars as in test_gpu_parity: 1e-11 in
FP64, 2e-5 mixed, on H psi, and 10 times that on 12 steps."""
import numpy as np
import pytest

from madwave3_amd import leps
from madwave3_amd.lib import (MW3_FP64, MW3_MIXED, MW3_OPT_ANGULAR, MW3_OPT_RADIAL, Propagator)
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.max(np.abs(a - b)) / np.max(np.abs(b)))


# npun1, npun2, nangu, Jtot, box r, box R (bohr)
SIZES = [
    (64, 64, 8, 0, None, None),
    (96, 128, 20, 0, 30.0, 30.0),
    (72, 100, 70, 0, 36.0, 30.0),
    (81, 75, 9, 0, 25.0, 30.0),
    (64, 64, 12, 2, 25.0, 25.0),
    (45, 50, 7, 3, None, None),
]


@pytest.mark.parametrize("n1,n2,na,J,b1,b2", SIZES)
def test_gemm_blocks(n1, n2, na, J, b1, b2):
    p = leps.config(4, J=J) if J else leps.config(1)
    p.update(npun1=n1, npun2=n2, nangu=na, npun1min=8, jmax=min(5, na - 1), nvmax=2, netot=0,
             iprod=0, kminelastic=4, width_bohr=0.6, absorb_bohr=4.5)
    if J:
        p.update(Jtot=J, iommin=0, iommax=J, iomref=-1, iparity=1 if J % 2 == 0 else -1)
    if b1:
        p.update(rfin1_bohr=b1)
    if b2:
        p.update(rfin2_bohr=b2)
    c = leps.build(p)
    print("case", (n1, n2, na, J, b1, b2), c, c.ntot / (c.ncan * n1 * n2 * na), flush=True)
    o = Oracle(c)
    psi = np.random.default_rng(n1 + n2).standard_normal(c.ntot)
    h = o.hphi(psi)
    o.begin(c.rpaq0)
    n_o = o.steps(12)[0]
    for prec, bar in ((MW3_FP64, 1e-11), (MW3_MIXED, 2e-5)):
        g = Propagator(c, prec)
        for radial, angular in ((0, 2), (1, 2), (0, 0)):
            g.set_option(MW3_OPT_RADIAL, radial)
            g.set_option(MW3_OPT_ANGULAR, angular)
            assert rel(g.hphi(psi), h) < bar, (prec, radial, angular)
            g.begin(c.rpaq0)
            assert rel(g.steps(12)[0], n_o) < 10 * bar, (prec, radial, angular)
        g.close()
