"""The transport's short root, reciprocal, quotient and azimuth on the GPU:
correctly rounded, and the azimuth bit for bit that of fd2_sincos_turns; and
the in-column step's general branch, which a geometry of unusual size always
takes, against the oracle photon by photon."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def floats(lo, hi):
    """Every float in [lo, hi)."""
    a, b = (np.float32(v).view(np.uint32) for v in (lo, hi))
    return np.arange(a, b, dtype=np.uint32).view(np.float32)


@pytest.mark.parametrize("lo", [2.0 ** -96, 2.0 ** -24, 0.25, 1.0, 2.0 ** 98])
@pytest.mark.parametrize("fn", ["sqrt_01", "sqrt_pos"])
def test_roots(fd2lib, fn, lo):
    x = floats(lo, 4 * lo)  # both exponent parities
    print(f"[short-math] {fn} {lo} n={len(x)}", flush=True)
    assert np.array_equal(fd2lib.debug_math(fn, x).view(np.uint32), np.sqrt(x).view(np.uint32))
    if fn == "sqrt_01":
        z = np.array([0.0, -0.0], np.float32)
        assert np.array_equal(fd2lib.debug_math(fn, z).view(np.uint32), z.view(np.uint32))


@pytest.mark.parametrize("lo", [2.0 ** -100, 2.0 ** -32, 0.5, 1.0, 2.0 ** 99])
def test_reciprocal_and_quotient(fd2lib, lo):
    x = floats(lo, 2 * lo)
    x = np.concatenate([x, -x])
    print(f"[short-math] recip/div {lo} n={len(x)}", flush=True)
    one = np.float32(1.0) / x
    assert np.array_equal(fd2lib.debug_math("recip", x).view(np.uint32), one.view(np.uint32))
    if 2.0 ** -60 <= lo <= 2.0 ** 59:
        q = np.float32(0.7310586) / x
        assert np.array_equal(fd2lib.debug_math("div", x).view(np.uint32), q.view(np.uint32))


@pytest.mark.parametrize("fn", ["sin", "cos"])
def test_azimuth_of_every_draw(fd2lib, fn):
    u = (np.arange(1, (1 << 24) + 1, dtype=np.float64) / (1 << 24)).astype(np.float32)
    print(f"[short-math] {fn} of {len(u)} draws", flush=True)
    a, b = fd2lib.debug_math(fn + "_quarters", u), fd2lib.debug_math(fn + "_turns", u)
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("R,H", [(0.003, 150.0), (2.55, 0.007)])
def test_unusual_geometry_matches_oracle(fd2lib, oracle, R, H):
    from hybridmantis_amd import events as E

    p = E.params(num_hist=4, R=R, H=H)
    ev = np.zeros(4, E.EVENT_DTYPE)
    ev["x"] = ev["y"] = 500.5
    ev["z"] = np.array([-0.4, -0.1, 0.2, 0.45], np.float32) * H
    ev["hist"] = np.arange(4) + 1
    ev["N"] = 24
    print(f"[short-math] R={R} H={H}", flush=True)
    with fd2lib.Transport(p) as tr:
        rec = tr.submit_record(ev)
    o = oracle.run(p, ev, 4, rng=oracle.RNG_COUNTER, math=oracle.MATH_DEVICE, record=True)
    assert np.array_equal(rec["fate"], o.photons["fate"])
    assert np.array_equal(rec["pix"], o.photons["pix"])
