"""What libmw3 asks of the HIP runtime, on a runtime without a device
(tests/fakehip.c, loaded in a process of its own): device memory of a context, blocks
of the update, what the autotuner times, what an option without effect costs."""
import json
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
PRELUDE = """
import ctypes as ct, json, sys
fake = ct.CDLL(sys.argv[1], mode=ct.RTLD_GLOBAL)
fake.fake_log.restype = ct.c_char_p
fake.fake_bytes.restype = ct.c_size_t
sys.path.insert(0, sys.argv[2])
from madwave3_amd import leps, lib as L
def log():
    s = fake.fake_log().decode()
    fake.fake_log_clear()
    return s
def case(n1, n2, na, J=0, **kw):
    p = leps.config(4, J=J) if J else leps.config(1)
    p.update(npun1=n1, npun2=n2, nangu=na, npun1min=min(16, n1 // 2), jmax=min(5, na - 1),
             nvmax=2, netot=100, iprod=0, kminelastic=4, width_bohr=0.6, absorb_bohr=4.5)
    if J:
        p.update(Jtot=J, iommin=J % 2 if J > 1 else 0, iommax=min(J, 6), iomref=-1)
    p.update(kw)
    return leps.build(p)
out = {}
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "fakehip.so")
    subprocess.run(["gcc", "-O1", "-w", "-shared", "-fPIC", "-o", so,
                    os.path.join(HERE, "fakehip.c")], check=True)

    def run(script):
        r = subprocess.run([sys.executable, "-c", PRELUDE + script + "\nprint(json.dumps(out))",
                            so, os.path.dirname(HERE)], capture_output=True, text=True,
                           timeout=300)
        assert r.returncode == 0, r.stderr
        return json.loads(r.stdout.splitlines()[-1])
    return run


MEMORY = """
for i, (n1, n2, na, J, prec, prod) in enumerate([(64, 256, 64, 12, 0, 0), (64, 256, 64, 12, 1, 0),
                                                 (64, 256, 64, 0, 1, 1), (32, 64, 16, 0, 0, 0)]):
    c = case(n1, n2, na, J, **(dict(iprod=2, nvmaxprod=2, jmaxprod=5) if prod else {}))
    g = L.Propagator(c, prec, prod=False)
    b0 = fake.fake_bytes()
    if prod:
        g.prod_attach()
    b = fake.fake_bytes()
    out[i] = dict(bytes=b, attach=b - b0, nc=c.ncan, n1=n1, n2=n2, na=na, prec=prec, ntot=c.ntot,
                  nflux=g.nflux, netot=c.netot, ncvj=c.ncan * (c.jmax - c.jini + 1) * 3)
    if prod:
        L_ = (c.nangproj1 - c.nangproj0 + 1) * (c.n2prod1 - c.n2prod0 + 1)
        nvj = L.prod_shape(c)[1] * L.prod_shape(c)[2]
        out[i]["prod"] = 8 * (L_ * (1 + nvj + 256) + 256 * nvj * 600)
    g.close()
out["left"] = fake.fake_bytes()
"""


def test_device_memory_of_a_context(fake):
    """Within the slabs, accumulators and tables a propagation needs; what the
    updates leave for the ring's sums (segments, slices) takes at most 128 MB each, or
    16 steps'."""
    out = fake(MEMORY)
    assert out.pop("left") == 0
    for r in out.values():
        s = 4 if r["prec"] else 8
        grid = r["nc"] * r["na"] * r["n1"] * r["n2"]
        cols = r["nc"] * r["na"] * (r["n2"] + 32)
        state = 5 * 8 * grid + (3 * 4 * grid if r["prec"] else 0)  # psi, psi_{k-1}, psi0, H psi, input
        work = 5 * s * grid + s * grid / r["nc"] + 2 * 8 * r["ntot"]
        accum = r["nflux"] * (32 * r["netot"] + 24 * 256) + r["ncvj"] * (16 * r["netot"] + 8 * 256)
        seg = cols * 4 * 8 * 1.25  # (strips cut in segments: 1.25)
        slices = 8 * r["nc"] * r["na"] * r["n1"]
        rings = sum(min(256 * x, max(128 << 20, 16 * x)) for x in (seg, slices))
        low = 0 if r["prec"] else 2.5 * 8 * 48 * cols  # G, G2
        tables = 0.5 * 8 * grid + (4 << 20)
        limit = state + work + accum + rings + low + tables + r.get("prod", 0) + (
            s * grid if "prod" in r else 0)
        print(r, "limit %.1f MB" % (limit / 1e6))
        assert r["bytes"] <= limit, (r, limit)


BLOCKS = """
for i, (n1, n2, na) in enumerate([(16, 32, 4), (128, 64, 8), (1200, 64, 16), (3500, 64, 16),
                                  (256, 256, 60)]):
    c = case(n1, n2, na, jmax=0, nvmax=0)
    for prec in (0, 1):
        g = L.Propagator(c, prec)
        g.begin(c.rpaq0)
        out["%d %d" % (i, prec)] = [n1, fake.fake_grid(b"k_update")]
        g.close()
"""


def test_update_fills_the_chip(fake):
    """The update's blocks (256 CUs, two blocks on each, one with more than 80 KB of
    LDS): long strips are shared out, and no more blocks run than are resident."""
    out = fake(BLOCKS)
    for k, (n1, blocks) in out.items():
        print(k, n1, blocks)
        assert 0 < blocks <= (256 if 24 * n1 > 80 * 1024 else 512)
        assert n1 < 1000 or blocks > 200


TUNE = """
for prec in (0, 1):
    for first in (0, 1):
        for n in (2, 4, 16, 20, 48):
            g = L.Propagator(case(32, 64, 16), prec)
            g.begin(g.case.rpaq0)
            if first:
                g.steps(1)
            log()
            g.autotune(n)
            out["%d %d %d" % (prec, first, n)] = log()
            g.close()
"""


def test_autotuner_times_steps_only(fake):
    """No capture between a trial's events, and the graph trials of 16 steps and
    more time the runs of 16 that a long call is made of."""
    for key, s in fake(TUNE).items():
        n = int(key.split()[-1])
        parts = s.split("T")
        assert len(parts) % 2 == 1 and len(parts) > 8
        timed = parts[1::2]
        assert not any(c in t for t in timed for c in "CIk"), (key, timed)
        graphs = "K" + "G" * (n // 16 if n >= 16 else n)  # (K: the ring slot of the first)
        assert graphs in timed and all(t == graphs or "G" not in t for t in timed), (key, timed)


OPTION = """
for prec in (0, 1):
    g = L.Propagator(case(32, 64, 16), prec)
    g.begin(g.case.rpaq0)
    g.steps(40)
    log()
    for v in (2, 4, 1):
        g.set_option(L.MW3_OPT_RADIAL_GRID, v)
    g.steps(32)
    s = log()
    out[prec] = s
    bad = 0
    try:
        g.set_option(L.MW3_OPT_RADIAL_GRID, 3)
    except L.Mw3Error:
        bad = 1
    out["%d bad" % prec] = bad
    g.close()
"""


def test_option_without_effect_keeps_graphs(fake):
    """MW3_OPT_RADIAL_GRID takes 1, 2 and 4 (and refuses others), and the steps after
    it run as the graphs captured before it."""
    out = fake(OPTION)
    for prec in "01":
        assert "C" not in out[prec] and "I" not in out[prec] and "G" in out[prec], out[prec]
        assert out[prec + " bad"] == 1


FORK = """
for name, size in dict(one_pass=(24, 48, 12, 0), parts=(100, 225, 46, 1), gemms=(105, 225, 45, 1),
                       gemms_small=(80, 160, 41, 1), low=(100, 256, 41, 1),
                       parts_large=(90, 300, 48, 12)).items():
    c = case(*size, **(dict(iparity=-1) if size[3] == 1 else {}))
    for prec in (0, 1):
        g = L.Propagator(c, prec)
        g.begin(c.rpaq0)
        log()
        g.steps(40)
        out["%s %d" % (name, prec)] = [c.ntot, log().count("w")]
        g.close()
"""


def test_captured_steps_fork_only_where_it_pays(fake):
    """One stream in FP64, with the low-mode R passes, an angular term of one launch,
    as GEMMs below 500 000 points and as folded Coriolis parts below 1.5 M; a fork and
    a join (two waits) in each captured step otherwise."""
    out = fake(FORK)
    assert out["parts_large 1"][0] >= 1500000 > out["parts 1"][0] > 500000
    assert out["gemms 1"][0] >= 500000 > out["gemms_small 1"][0]
    for k, (_, waits) in out.items():
        assert (waits > 0) == (k in ("gemms 1", "parts_large 1")), out
        assert waits % 2 == 0
