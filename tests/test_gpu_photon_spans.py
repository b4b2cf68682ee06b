"""Work-queue spans over many small events: per-photon records against the
oracle at the queue build's edges (one block / several), with long runs of
empty events, and at launches of fewer photons than one per SIMD, a few lanes
per wave, and more than 64 per wave."""
import numpy as np
import pytest

from hybridmantis_amd import events as E

pytestmark = pytest.mark.gpu


def small_events(n, mean, empty, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    ev = np.zeros(n, E.EVENT_DTYPE)
    ev["x"] = 454.5 + rng.normal(0, 3, n)
    ev["y"] = 454.5 + rng.normal(0, 3, n)
    ev["z"] = rng.uniform(-70, 70, n)
    ev["N"] = rng.poisson(mean, n)
    ev["N"][rng.random(n) < empty] = 0
    if empty > 0:
        ev["N"][n // 3: n // 3 + n // 2] = 0  # a long empty run inside a span
    ev["hist"] = np.arange(n) // 7 + 1
    return ev


@pytest.mark.parametrize("n,mean,empty,chunk", [
    (1, 1, 0.0, 128), (2, 500, 0.0, 128), (70, 1, 0.5, 128), (300, 40, 0.0, 1),
    (4096, 2, 0.0, 128), (4097, 2, 0.3, 16), (9001, 0.02, 0.9, 128), (20000, 3, 0.95, 64),
    (40000, 25, 0.2, 128)])
def test_spans_match_oracle(fd2lib, oracle, n, mean, empty, chunk):
    ev = small_events(n, mean, empty, n + chunk)
    p = E.params(num_hist=int(ev["hist"].max()), R=5.1, xdet=909.0, ydet=909.0, lbx=0.0, lby=0.0,
                 ubx=909.0, uby=909.0, pixel=9, sensor_refl=0.25)
    total = int(ev["N"].sum())
    print(f"[spans] {n} events, {total} photons, chunk {chunk}", flush=True)
    o = oracle.run(p, ev, p["num_hist"], rng=oracle.RNG_COUNTER, math=oracle.MATH_DEVICE,
                   record=True)
    with fd2lib.Transport(p, tuning=dict(chunk=chunk)) as tr:
        rec = tr.submit_record(ev)
        assert np.array_equal(rec["fate"], o.photons["fate"])
        assert np.array_equal(rec["pix"], o.photons["pix"])
        tr.reset()
        tr.submit(ev)
        assert tr.counters()["generated"] == total
        assert np.array_equal(tr.prf(), o.prf)
    # the same events in device memory through the allocation-free submit, and
    # with waiting photons kept in their lanes
    with fd2lib.Transport(p, tuning=dict(chunk=chunk, wall_queue=-1, park_lanes=5)) as tr:
        buf = tr.upload_events(ev)
        tr.submit_device_noalloc(buf, n)
        assert np.array_equal(tr.prf(), o.prf)
        buf.free()
