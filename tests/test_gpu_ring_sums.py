"""The sums of a ring of steps where what the updates leave is kept for fewer steps
than a ring (128 MB: 16 steps at seven blocks of 48 x 512 x 64, 32 at 64 x 256 x 64,
64 or 128 at 24 x 512 x 64, and other depths for segments and slices):
one long call against many short ones, whose steps are summed as they come, by
graphs and kernel by kernel.  Norms and per-step records are bitwise the same; the
energy sums, added up in other groups, to the rounding of 300 terms."""
import numpy as np
import pytest

from madwave3_amd import leps
from madwave3_amd.lib import MW3_FP64, MW3_MIXED, MW3_OPT_GRAPHS, Propagator

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.max(np.abs(a - b)) / np.max(np.abs(b)))


def run(c, prec, calls, graphs):
    g = Propagator(c, prec)
    g.set_option(MW3_OPT_GRAPHS, graphs)
    g.records(True)
    g.begin(c.rpaq0)
    norms = np.concatenate([g.steps(n)[0] for n in calls])
    it, cvj, cvjp = g.take_records()
    out = norms, it, cvj, cvjp, g.flux_accum(), g.zs2(), g.zs2prod() if cvjp is not None else None
    g.close()
    return out


@pytest.mark.parametrize("n1,n2,na,J,prec,prod", [(64, 256, 64, 12, MW3_FP64, False),
                                                  (48, 512, 64, 12, MW3_MIXED, False),
                                                  (24, 512, 64, 0, MW3_FP64, True),
                                                  (24, 512, 64, 0, MW3_MIXED, True)])
def test_ring_places(n1, n2, na, J, prec, prod):
    p = leps.config(4, J=J) if J else leps.config(1)
    p.update(npun1=n1, npun2=n2, nangu=na, npun1min=8, jmax=5, nvmax=2, netot=20,
             iprod=2 if prod else 0, nvmaxprod=2, jmaxprod=4, kminelastic=4, width_bohr=0.6,
             absorb_bohr=4.5)
    if J:
        p.update(Jtot=J, iommin=0, iommax=6, iomref=-1)
    c = leps.build(p)
    print("case", (n1, n2, na, J, prec, prod), c, flush=True)
    a = run(c, prec, [300], 1)
    for calls, graphs in (([1] * 20 + [16, 37, 2, 225], 1), ([7, 293], 0)):
        b = run(c, prec, calls, graphs)
        for x, y in zip(a[:4], b[:4]):
            assert x is None if y is None else np.array_equal(x, y)
        assert rel(b[4][0], a[4][0]) < 1e-12 and rel(b[4][1], a[4][1]) < 1e-12
        assert rel(b[5], a[5]) < 1e-12
        assert b[6] is None or rel(b[6], a[6]) < 1e-12
    assert np.all(a[0] > 0.0) and a[1].tolist() == list(range(2, 302))
