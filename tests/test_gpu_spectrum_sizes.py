"""The spectrum where its kernels change (one term per thread and turns, blocks
for four energies and one energy per thread) and with tens of thousands of terms,
against extended precision.  Bar, per term and energy: the angle th = acos(Es) is
an ulp off at most, so k th is off by kmax ulp(th); a rounded k th by half an ulp of
kmax th; a rotation of 512 terms by two roundings a turn."""
import numpy as np
import pytest

from madwave3_amd import consts as C
from madwave3_amd.lib import cheby_spectrum

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kmax,ne", [(1, 16384), (31, 16383), (31, 16384), (32, 16384), (63, 7),
                                     (64, 40959), (65, 40960), (512, 40961), (895, 40960),
                                     (896, 40959), (896, 40960), (897, 40960), (30000, 24),
                                     (60000, 18), (100001, 6)])
def test_spectrum_sizes(kmax, ne):
    rng = np.random.default_rng(kmax + ne)
    a = rng.standard_normal(kmax + 1)
    emindlt, delta2, xk = 0.4, 1.7, 0.5 / kmax
    es = rng.uniform(-0.97, 0.97, ne)
    es[::2] = np.cos(rng.uniform(0.005, 0.02, es[::2].size))  # a small ulp(th)
    e = emindlt + delta2 * es
    got = cheby_spectrum(a, emindlt, delta2, C.hbr, xk, e)
    assert got.shape == (ne,)
    at = np.unique(np.concatenate([rng.integers(0, ne, 100), np.arange(max(0, ne - 6), ne), [0]]))
    es = (e[at] - emindlt) / delta2  # as the library forms it
    k = np.arange(1, kmax + 1, dtype=np.longdouble)
    ak = 2.0 * C.hbr * np.exp(-k * xk) * a[1:]
    th = np.arccos(es.astype(np.longdouble))
    want = np.array([(a[0] * C.hbr + np.sum(ak * np.cos(k * t))) for t in th])
    want = want / (np.sqrt(1 - es.astype(np.longdouble) ** 2) * delta2)
    size = (abs(a[0]) * C.hbr + np.sum(np.abs(ak))) / (np.sqrt(1.0 - es ** 2) * delta2)
    t = th.astype(float)
    bar = kmax * np.spacing(t) + 0.5 * np.spacing(kmax * t) + (kmax / 512 + 1) * 4.4e-16 + 2e-15
    err = np.abs(got[at] - want).astype(float) / size.astype(float)
    print("kmax %d ne %d: err %.1e, of its bar %.2f" % (kmax, ne, err.max(), (err / bar).max()))
    assert np.all(err <= bar)
