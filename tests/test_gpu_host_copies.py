"""Events and results through the pinned ring: sizes at the edges of one slice,
of one slice per slot and beyond, the same answers as events already in device
memory or in smaller calls, and the first invalid event's status."""
import numpy as np
import pytest

from hybridmantis_amd import events as E

pytestmark = pytest.mark.gpu

KB64, SLICE, RING = (64 << 10) // 32, (512 << 10) // 32, (16 << 20) // 32  # in events


def events(n, every):
    rng = np.random.Generator(np.random.PCG64(n))
    ev = np.zeros(n, E.EVENT_DTYPE)
    ev["x"] = 454.5 + rng.normal(0, 3, n)
    ev["y"] = 454.5 + rng.normal(0, 3, n)
    ev["z"] = rng.uniform(-70, 70, n)
    ev["N"][::every] = 2
    ev["hist"] = np.arange(n) % 97 + 1
    return ev


def params():
    return E.params(num_hist=97, R=5.1, xdet=909.0, ydet=909.0, lbx=0.0, lby=0.0, ubx=909.0,
                    uby=909.0, pixel=9)


@pytest.mark.parametrize("n", [1, KB64, KB64 + 1, SLICE, SLICE + 1, 8 * SLICE + 3,
                               RING + SLICE + 5])
def test_submitted_events_arrive(fd2lib, n):
    ev = events(n, max(1, n // 3000))
    print(f"[copies] {n} events", flush=True)
    with fd2lib.Transport(params()) as tr:
        buf = tr.upload_events(ev)
        tr.submit_device(buf, n)
        tr.sync()
        want = tr.prf(), tr.hist_counts(), tr.counters()
        buf.free()
        for _ in range(2):
            tr.reset()
            tr.submit(ev)
            tr.sync()
            assert np.array_equal(tr.prf(), want[0])
            assert np.array_equal(tr.hist_counts(), want[1])
            assert tr.counters() == want[2]


@pytest.mark.parametrize("many,negative,geom,code", [
    (5, None, None, "photons"), (None, 5, None, "invalid"), (3 * SLICE, 2, None, "invalid"),
    (2, 3 * SLICE, None, "photons"), (9 * SLICE, 9 * SLICE + 1, 9 * SLICE - 1, "invalid"),
    (9 * SLICE + 7, None, 9 * SLICE + 8, "photons")])
def test_first_invalid_event_is_reported(fd2lib, many, negative, geom, code):
    ev = events(9 * SLICE + 9, 400)
    bad = ev.copy()
    if many is not None:
        bad["N"][many] = 900001
    if negative is not None:
        bad["N"][negative] = -1
    if geom is not None:
        bad["geom"][geom] = 1
    with fd2lib.Transport(params()) as tr:
        tr.submit(ev)
        tr.sync()
        want = tr.prf()
        tr.reset()
        with pytest.raises(fd2lib.Fd2Error, match=code):
            tr.submit(bad)
        assert tr.counters()["generated"] == 0
        tr.submit(ev)
        tr.sync()
        assert np.array_equal(tr.prf(), want)


@pytest.mark.parametrize("photons", [1, 65535, 65537, 300001, 1200007])
def test_records_of_one_call_and_of_two(fd2lib, photons):
    """16 bytes a record: below 1 MB, around it, one slice per slot, several."""
    ev = events(max(2, photons // 100), 1)
    ev["N"] = 0
    ev["N"][: len(ev) // 2 + 1] = photons // (len(ev) // 2 + 1)
    ev["N"][0] += photons - int(ev["N"].sum())
    half = len(ev) // 4 + 1
    print(f"[copies] {photons} records", flush=True)
    with fd2lib.Transport(params()) as tr:
        whole = tr.submit_record(ev)
        tr.reset()
        parts = np.concatenate([tr.submit_record(ev[:half]), tr.submit_record(ev[half:])])
    assert len(whole) == photons
    assert np.array_equal(whole.view(np.uint8), parts.view(np.uint8))


def test_forward_of_one_call_and_of_many(fd2lib):
    """65 floats a row: within one copy, several slices, several batches."""
    rng = np.random.Generator(np.random.PCG64(5))
    x = rng.uniform(0, 1, (70001, 5)).astype(np.float32)
    net = fd2lib.Mlp(seed=3)
    whole = net.forward(x)
    parts = [net.forward(x[a:b]) for a, b in
             ((0, 1), (1, 4033), (4033, 8066), (8066, 20000), (20000, 70001))]
    assert np.array_equal(whole, np.concatenate(parts))


def test_radial_histograms_of_one_call_and_of_two(fd2lib):
    """256 bytes an event: more than the events' own ring holds, on a new context."""
    ev = events(9001, 1)
    with fd2lib.Transport(params()) as tr:
        whole = fd2lib.submit_radial(tr, ev)
    with fd2lib.Transport(params()) as tr:
        parts = [fd2lib.submit_radial(tr, ev[a:b]) for a, b in ((0, 3000), (3000, 6001), (6001, 9001))]
    assert whole.sum() > 0 and np.array_equal(whole, np.concatenate(parts))
