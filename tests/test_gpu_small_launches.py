"""Launches of few photons per wave (a few lanes of a wave take photons) in every
form of the transport: tallies, records, radial histograms, the allocation-free
submit and a graph, with one and with several geometries and long runs of empty
events.  Photon counts around the plan's steps for 1,024 waves (one per SIMD of 256
compute units): 1 photon, below and just above 16, 32 and 64 per wave, and 128.
Tallies and records against the oracle, bit for bit; radial histograms against
the same events at the head of a launch that uses whole waves."""
import numpy as np
import pytest

from hybridmantis_amd import events as E

pytestmark = pytest.mark.gpu

GEOMS = [(100.0, 2.55), (150.0, 5.1), (300.0, 4.0)]


def events(photons, n_geoms, empty, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    n = max(1, photons // 60)
    ev = np.zeros(n, E.EVENT_DTYPE)
    ev["x"] = 454.5 + rng.normal(0, 3, n)
    ev["y"] = 454.5 + rng.normal(0, 3, n)
    ev["z"] = rng.uniform(-45, 45, n)
    ev["geom"] = rng.integers(0, n_geoms, n)
    ev["hist"] = np.arange(n) // 7 + 1
    full = np.ones(n, bool)
    if empty:
        full = rng.random(n) < 0.4
        full[n // 4:3 * n // 4] = False
        full[-1] = True
    ev["N"][full] = photons // full.sum()
    ev["N"][np.flatnonzero(full)[:photons - int(ev["N"].sum())]] += 1
    assert int(ev["N"].sum()) == photons
    return ev


@pytest.mark.parametrize("n_geoms", [1, 3])
@pytest.mark.parametrize("photons,empty", [
    (1, False), (1023, True), (17 * 1024 - 1024, False), (17 * 1024, True), (33 * 1024 - 1024, False),
    (33 * 1024, True), (64 * 1024 - 1, False), (64 * 1024 + 1, True), (128 * 1024, False)])
def test_every_form(fd2lib, oracle, n_geoms, photons, empty):
    ev = events(photons, n_geoms, empty, photons + n_geoms)
    n, nh = len(ev), int(ev["hist"].max())
    pl = [E.params(num_hist=nh, H=h, R=r, xdet=909.0, ydet=909.0, lbx=0.0, lby=0.0, ubx=909.0,
                   uby=909.0, pixel=9, sensor_refl=0.25) for h, r in GEOMS[:n_geoms]]
    want, owner = [], np.repeat(ev["geom"], ev["N"])
    fate = np.empty(photons, np.int32)
    pix = np.empty(photons, np.int32)
    for g, p in enumerate(pl):
        one = ev.copy()
        one["N"][ev["geom"] != g] = 0
        o = oracle.run(p, one, nh, rng=oracle.RNG_COUNTER, math=oracle.MATH_DEVICE, record=True)
        fate[owner == g], pix[owner == g] = o.photons["fate"], o.photons["pix"]
        want.append((o.prf, o.hist_count, {k: o.counter(k) for k in oracle.COUNTER_NAMES}))
    print(f"[small] {photons} photons, {n} events, {n_geoms} geometries", flush=True)

    def same(tr):
        tr.sync()
        for g, (prf, hist, counters) in enumerate(want):
            assert np.array_equal(tr.prf(g), prf)
            assert np.array_equal(tr.hist_counts(g), hist)
            have = tr.counters(g)
            assert {k: have[k] for k in counters} == counters
        tr.reset()

    with fd2lib.Transport(pl) as tr:
        tr.submit(ev)
        same(tr)
        rec = tr.submit_record(ev)
        assert np.array_equal(rec["fate"], fate) and np.array_equal(rec["pix"], pix)
        same(tr)
        radial = fd2lib.submit_radial(tr, ev)
        same(tr)
        buf = tr.upload_events(ev)
        tr.submit_device_noalloc(buf, n)
        same(tr)
        with tr.graph(buf, n) as graph:
            for _ in range(2):
                graph.launch()
                same(tr)
        buf.free()
        more = np.concatenate([ev, ev[:1]])
        more["N"][n] = 300000
        assert np.array_equal(fd2lib.submit_radial(tr, more)[:n], radial)
