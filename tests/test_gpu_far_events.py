"""Events outside the layer, at its edges, with a first column far away and
with coordinates that are not finite: every photon's fate, pixel and detection
point against the oracle, bit for bit.  The short arithmetic of the in-column
pass holds for distances of ordinary size only; a distance beyond them (a
quotient that overflows, an infinite coordinate) has to end the photon as IEEE
arithmetic does."""
import numpy as np
import pytest

from hybridmantis_amd import events as E

pytestmark = pytest.mark.gpu

Z = [75.0, -75.0, 75.00001, 80.0, -80.0, 1e3, -1e3, 1e10, -1e10, 2.0 ** 59, 2.0 ** 61, 1e30, -1e30,
     1e37, 1e38, -1e38, 3e38, -3e38, np.inf, -np.inf, 1e-30, -1e-30, 0.0]
XY = [0.0, 1e-6, 9e-6, -1.0, 909.0, 909.1, 1e10, 1e30, 3e38, -3e38, np.inf, -np.inf]
DX = [1.0, 5.1, 5.09999, -5.1, 6.0, -20.0, 1e5, 1e10, 1e18, 1e30, -1e30, np.inf]


def far_events():
    at = [(454.5, 454.5, z, 0.0) for z in Z]
    at += [(x, 454.5, 10.0, 0.0) for x in XY] + [(454.5, y, 10.0, 0.0) for y in XY]
    at += [(454.5, 454.5, z, c) for c in DX for z in (10.0, 75.0)]
    ev = np.zeros(len(at), E.EVENT_DTYPE)
    for e, (x, y, z, c) in zip(ev, at):
        e["x"], e["y"], e["z"], e["col_dx"] = x, y, z, c
    ev["N"] = 40
    ev["hist"] = np.arange(len(ev)) + 1
    return ev


@pytest.mark.parametrize("kw", [
    dict(), dict(H=500.0, R=2.55, xdet=1001.0, ydet=1001.0), dict(H=0.016), dict(R=0.01),
    dict(beta=0.0, sensor_refl=0.0), dict(bulk=1e-2)],
    ids=["150um", "500um", "flat", "thin", "smooth", "absorbing"])
def test_far_events_match_oracle(fd2lib, oracle, kw):
    ev = far_events()
    p = dict(R=5.1, xdet=909.0, ydet=909.0, lbx=0.0, lby=0.0, ubx=909.0, uby=909.0, pixel=9,
             sensor_refl=0.25)
    p.update(kw)
    p = E.params(num_hist=len(ev), **p)
    o = oracle.run(p, ev, len(ev), rng=oracle.RNG_COUNTER, math=oracle.MATH_DEVICE, record=True)
    print(f"[far] {kw}", flush=True)
    with fd2lib.Transport(p) as tr:
        rec = tr.submit_record(ev)
        bad = np.flatnonzero((rec["fate"] != o.photons["fate"]) | (rec["pix"] != o.photons["pix"]))
        assert len(bad) == 0, ev[np.unique(bad // 40)]
        for c in "xy":
            assert np.array_equal(rec[c].view(np.uint32), o.photons[c].view(np.uint32))
        tr.reset()
        tr.submit(ev)
        assert np.array_equal(tr.prf(), o.prf)
        assert np.array_equal(tr.hist_counts(), o.hist_count)
