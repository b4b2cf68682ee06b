"""Timed cases of the fastDETECT2 transport and its surrogate.

Each case is one call (or the few calls that belong together) that a program
using this package makes, from the data it holds to the results it reads:

  host      events in host memory -> fd2_submit -> PRF, per-history counts,
            counters (what penEasy's tally does with a full event buffer)
  device    the same on events already in device memory
  noalloc   the same through the allocation-free submit
  graph     the same through a captured HIP graph (several geometries)
  record    one record per photon instead of tallies
  radial    log-radial detection histograms per event (training targets)
  surrogate network + Monte Carlo fallback, tallies and audit
  forward   network inference on host rows
  gradients loss and gradients of one batch
  train     Adam steps from given weights, losses and updated weights

All inputs are synthetic and made from the seed.  Tallies are reset at the
start of a pass, so every pass of a state transports the same photons.
"""
import math

import numpy as np
import torch

from hybridmantis_amd import events as E
from hybridmantis_amd import fd2
from hybridmantis_amd import surrogate as S

# largest event buffer of the reference's driver
BUFFER = 2304000
# arithmetic of one optical photon in a 150-um layer (one FP32 operation per
# +, -, *, / and elementary function), and per network row
PHOTON_FLOP = 1.0e4
ROW_FLOP = 2.0 * (5 * 256 + 2 * 256 * 256 + 256 * 65)


def listed():
    return [
        # one deposition event at a time, the reference's example detector
        # (9-um pixels, R = 5.1 um, partly reflecting sensor): latency
        dict(name="one_event", kind="host", events=1, photons=1375, H=150.0, R=5.1, pixel=9,
             refl=0.25, bulk=1e-4, top=0.1, energy=25.0),
        # a short run inside a caller that may not allocate
        dict(name="noalloc_200", kind="noalloc", hist=200, H=300.0, R=4.0, pixel=2, refl=0.0,
             bulk=1e-4, top=0.1, energy=60.0),
        # the reference case that a CPU still runs: 2,000 histories at 25 keV
        dict(name="mono25", kind="host", hist=2000, H=150.0, R=2.55, pixel=1, refl=0.0,
             bulk=1e-4, top=0.1, energy=25.0),
        # the headline workload: 100,000 histories at 25 keV
        dict(name="mono25x50", kind="device", hist=100000, H=150.0, R=2.55, pixel=1, refl=0.0,
             bulk=1e-4, top=0.1, energy=25.0),
        # the reference driver's full event buffer at its example run's two
        # photons per event (electron tracks give many small deposits)
        dict(name="ede_buffer", kind="host", events=BUFFER, photons=2.06, H=150.0, R=5.1, pixel=9,
             refl=0.25, bulk=1e-4, top=0.1, energy=25.0),
        # four detectors, 15-90 keV, one graph launch
        dict(name="batched_poly", kind="graph", hist=5000),
        # surrogate training targets: 20 detectors, 1e5 photons per grid point
        dict(name="radial_grid", kind="radial", depths=7, offsets=3, photons=100000),
        # per-photon records for an analysis program
        dict(name="record_501", kind="record", hist=501, H=150.0, R=2.55, pixel=1, refl=0.0,
             bulk=1e-4, top=0.1, energy=40.0),
        # surrogate production run, a fifth of 1e6 histories at 50 keV
        dict(name="surrogate_mono50", kind="surrogate", hist=200000, H=500.0, R=5.0, energy=50.0),
        # network inference, a ragged number of rows
        dict(name="forward_50001", kind="forward", rows=50001),
        # one training batch's gradients for an outside optimiser
        dict(name="gradients_4096", kind="gradients", rows=4096),
        # a stretch of training at the network's own batch size
        dict(name="train_4096", kind="train", rows=4096, steps=60, data=65536),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["host", "host", "small", "device", "noalloc", "ede", "graph", "record",
                       "radial", "surrogate", "forward", "gradients", "train"])
    if kind == "graph":
        return dict(kind="graph", hist=_log(rng, 20, 5000))
    if kind == "radial":
        return dict(kind="radial", depths=rng.randint(1, 9), offsets=rng.randint(1, 3),
                    photons=_log(rng, 1000, 70000))
    if kind == "forward":
        return dict(kind="forward", rows=_log(rng, 1, 70000))
    if kind == "gradients":
        return dict(kind="gradients", rows=16 * _log(rng, 2, 512))
    if kind == "train":
        return dict(kind="train", rows=16 * _log(rng, 8, 256), steps=rng.randint(5, 60),
                    data=_log(rng, 5000, 65536))
    if kind == "surrogate":
        H, R = rng.choice(E.BATCH_GEOMS)
        return dict(kind="surrogate", hist=_log(rng, 300, 150000), H=H, R=R,
                    energy=float(rng.randint(25, 60)))
    c = dict(H=round(rng.uniform(100.0, 500.0), 1), R=round(rng.uniform(2.55, 5.1), 2),
             pixel=rng.choice([1, 2, 3, 9]), refl=rng.choice([0.0, 0.25]),
             bulk=rng.choice([0.0, 1e-4, 1e-3]), top=rng.choice([0.0, 0.1, 0.5]),
             energy=float(rng.randint(15, 90)))
    if kind == "small":
        n = _log(rng, 2, 2000)
        return dict(c, kind="host", events=n, photons=_log(rng, 4, 4000))
    if kind == "ede":
        return dict(c, kind="host", events=_log(rng, 20000, 1500000),
                    photons=round(rng.uniform(0.5, 6.0), 2))
    # photons of a history: 0.8 * 55 per keV, about 69 steps each in 150 um
    most = {"host": 4e7, "device": 4e7, "noalloc": 2e6, "record": 2e6}[kind]
    hist = _log(rng, 5, most / (44.0 * c["energy"]) * min(1.0, 150.0 / c["H"]))
    return dict(c, kind=kind, hist=hist)


def _photons(case):
    """Mean number of optical photons of a pass."""
    k = case["kind"]
    if k == "graph":
        return 4 * case["hist"] * 44.0 * 52.5
    if k == "radial":
        return 20.0 * case["depths"] * case["offsets"] * case["photons"]
    if "events" in case:
        return float(case["events"]) * case["photons"]
    return 44.0 * case["energy"] * case["hist"]


def _events(case):
    k = case["kind"]
    if k == "radial":
        return 20.0 * case["depths"] * case["offsets"]
    if "events" in case:
        return float(case["events"])
    return 2.0 * case["hist"] * (4 if k == "graph" else 1)


def work(case):
    k = case["kind"]
    if k in ("forward", "gradients", "train"):
        n = case["rows"]
        if k == "forward":
            return {"bytes": n * 4.0 * (5 + 65) + 6.4e5, "flops": n * ROW_FLOP}
        steps = case.get("steps", 1)
        return {"bytes": steps * n * 4.0 * (5 + 65) + 1.3e6, "flops": 3.0 * steps * n * ROW_FLOP}
    ph, ev = _photons(case), _events(case)
    out = 8.0 * 501 * 501 * (4 if k == "graph" else 1) if k != "radial" else 256.0 * ev
    if k == "record":
        out = 16.0 * ph
    flops = ph * PHOTON_FLOP
    if k == "surrogate":  # two thin surface layers and one event in a hundred take the transport
        share = 0.01 + 10.0 / case["H"]
        flops = share * flops + ev * ROW_FLOP
    return {"bytes": 32.0 * ev + out, "flops": flops}


def _params(case, num_hist):
    side = 909.0 if case["pixel"] == 9 else 1001.0
    lo, hi = (0.0, 909.0) if case["pixel"] == 9 else (250.0, 751.0)
    return E.params(num_hist=num_hist, H=case["H"], R=case["R"], pixel=case["pixel"],
                    sensor_refl=case["refl"], bulk=case["bulk"], top_absfrac=case["top"],
                    xdet=side, ydet=side, lbx=lo, lby=lo, ubx=hi, uby=hi)


def _small_events(case, side, seed):
    """`events` deposits with `photons` photons each on average: histories of
    up to 461 deposits around one interaction point, photon counts Poisson of
    an exponential deposit energy."""
    rng = np.random.Generator(np.random.PCG64(seed))
    n, H = case["events"], case["H"]
    hist = np.arange(n) // 461
    nh = int(hist[-1]) + 1
    depth = rng.exponential(150.0, nh) % H
    ev = np.zeros(n, E.EVENT_DTYPE)
    ev["x"] = np.clip(0.5 * side + rng.normal(0.0, 3.0, n), 0.01, side - 0.01)
    ev["y"] = np.clip(0.5 * side + rng.normal(0.0, 3.0, n), 0.01, side - 0.01)
    ev["z"] = np.clip(H / 2 - depth[hist] + rng.normal(0.0, 3.0, n), -H / 2 + 0.01, H / 2 - 0.01)
    mean = case["photons"] * (rng.exponential(1.0, n) if n > 1 else np.ones(n))
    ev["N"] = rng.poisson(mean)
    ev["E"] = mean / 0.055
    ev["hist"] = hist + 1
    return ev, nh


def _rows(n, rng):
    """Feature rows and targets over the network's training range."""
    x = np.empty((n, 5), np.float32)
    geom = np.array(E.BATCH_GEOMS, np.float32)[rng.integers(0, 4, n)]
    x[:, 0] = rng.random(n)
    x[:, 1] = rng.random(n)
    x[:, 2] = geom[:, 0] / 500.0
    x[:, 3] = geom[:, 1] / 5.0
    x[:, 4] = rng.uniform(0.5, 0.95, n)
    y = np.empty((n, 65), np.float32)
    y[:, 0] = 0.3 + 0.5 * x[:, 0] + 0.05 * rng.standard_normal(n)
    k = np.arange(64, dtype=np.float32)
    q = np.exp(-0.5 * ((k - (12 + 36 * x[:, :1])) / (5 + 4 * x[:, 1:2])) ** 2)
    q *= rng.uniform(0.8, 1.2, q.shape)
    y[:, 1:] = q / q.sum(1, keepdims=True)
    y[rng.random(n) < 0.01, 1:] = 0.0  # no photon detected
    return x, y


SHAPES = [(32, 256), (256, 256), (256, 256), (256, 80)]
REAL = [(5, 256), (256, 256), (256, 256), (256, 65)]


def _weights(rng):
    """Glorot-uniform weights with small biases, in the network's order:
    W0 [32x256], b0, W1 [256x256], b1, W2, b2, W3 [256x80], b3 (the rows and
    columns past 5 inputs and 65 outputs are zero)."""
    out = []
    for (r, c), (rr, cc) in zip(SHAPES, REAL):
        w = np.zeros((r, c), np.float32)
        lim = math.sqrt(6.0 / (rr + cc))
        w[:rr, :cc] = rng.uniform(-lim, lim, (rr, cc))
        b = np.zeros(c, np.float32)
        b[:cc] = rng.normal(0.0, 0.02, cc)
        out += [w.ravel(), b]
    return np.concatenate(out)


def _network_inputs(case, seed):
    rng = np.random.default_rng(seed)
    w = _weights(rng)
    x, y = _rows(case["data"] if case["kind"] == "train" else case["rows"], rng)
    return w, x, y


def prepare(case, seed):
    k = case["kind"]
    s = dict(case, seed=seed)
    if k in ("forward", "gradients", "train"):
        w, x, y = _network_inputs(case, seed)
        s["net"] = fd2.Mlp(seed=1)
        if k == "train":
            s["w"] = w
            s["net"].set_data(x, y)
        else:
            s["net"].set_params(w)
            s["x"], s["y"] = x, y
        return s
    if k == "graph":
        plist, ev = E.batched_workload(scale=case["hist"] / 50000.0, seed=seed)
        s["tr"] = fd2.Transport(plist, seed=seed)
        s["buf"] = s["tr"].upload_events(ev)
        s["graph"] = s["tr"].graph(s["buf"], len(ev))
        return s
    if k == "radial":
        rng = np.random.default_rng(seed)
        ev, _, _ = S.grid_events(case["depths"], case["offsets"], case["photons"])
        H = np.array([g[0] for g in E.BATCH_GEOMS])[ev["geom"] // 5]
        ev["z"] = np.clip(ev["z"] + rng.uniform(-2.0, 2.0, len(ev)), -H / 2 + 0.1, H / 2 - 0.1)
        s["tr"] = fd2.Transport(S.grid_params(), seed=seed)
        s["ev"] = ev
        return s
    if k == "surrogate":
        p = E.params(num_hist=case["hist"], H=case["H"], R=case["R"], max_ph=5000, num_bins=1000)
        lam = float(E.attenuation_length_um(case["energy"]))
        s["ev"] = E.generate(case["hist"], case["H"], case["energy"], lam, seed)
        s["tr"] = fd2.Transport(p, seed=seed)
        s["net"] = S.load()
        return s
    side = 909.0 if case["pixel"] == 9 else 1001.0
    if "events" in case:
        ev, hist = _small_events(case, side, seed)
    else:
        hist = case["hist"]
        lam = float(E.attenuation_length_um(case["energy"]))
        # a record per photon: the number of photons is the case's, the
        # deposits' places the seed's
        ev = E.generate(hist, case["H"], case["energy"], lam,
                        0x5EED0005 if k == "record" else seed, beam=(side / 2, side / 2),
                        xdet=side, ydet=side)
        if k == "record":
            rng = np.random.Generator(np.random.PCG64(seed))
            ev["x"] += rng.normal(0.0, 1.0, len(ev)).astype(np.float32)
            ev["y"] += rng.normal(0.0, 1.0, len(ev)).astype(np.float32)
            ev["z"] = rng.permutation(ev["z"])
    s["tr"] = fd2.Transport(_params(case, hist), seed=seed)
    if k in ("device", "noalloc"):
        s["buf"] = s["tr"].upload_events(ev)
        s["n"] = len(ev)
    else:
        s["ev"] = ev
    return s


def _tallies(tr, geom=0):
    return {"prf": tr.prf(geom), "hist": tr.hist_counts(geom), "counters": tr.counters(geom)}


def run(s):
    k = s["kind"]
    if k == "forward":
        return s["net"].forward(s["x"])
    if k == "gradients":
        loss, g = s["net"].gradients(s["x"], s["y"])
        return {"loss": loss, "grads": g}
    if k == "train":
        net = s["net"]
        net.set_params(s["w"])
        losses, _ = net.train(s["steps"], batch=s["rows"], lr=1e-3, seed=s["seed"])
        return {"losses": losses, "params": net.params()}
    tr = s["tr"]
    tr.reset()
    if k == "radial":
        return fd2.submit_radial(tr, s["ev"])
    if k == "record":
        rec = tr.submit_record(s["ev"])
        return {f: rec[f] for f in rec.dtype.names}
    if k == "graph":
        s["graph"].launch()
        tr.sync()
        return [_tallies(tr, g) for g in range(len(tr.params))]
    if k == "surrogate":
        st = fd2.surrogate_submit(tr, s["net"], s["ev"], seed=s["seed"] & 0xFFFFFFFF)
        out = _tallies(tr)
        out["routing"] = {f: st[f] for f in ("n_events", "n_mc", "n_surrogate", "n_audit",
                                             "photons_mc", "photons_surrogate")}
        out["audit"] = {f: st[f] for f in ("audit_detected_mc", "audit_detected_pred",
                                           "audit_radial_l1")}
        return out
    if k == "device":
        tr.submit_device(s["buf"], s["n"])
        tr.sync()
    elif k == "noalloc":
        tr.submit_device_noalloc(s["buf"], s["n"])
    else:
        tr.submit(s["ev"])
    return _tallies(tr)


# ---- network outputs in 64 bits ------------------------------------------------------

def _unpack(w):
    out, at = [], 0
    for r, c in SHAPES:
        out.append((w[at:at + r * c].view(r, c), w[at + r * c:at + r * c + c]))
        at += r * c + c
    return out


def _logits(layers, x):
    a = torch.nn.functional.pad(x, (0, 27))
    for i, (w, b) in enumerate(layers):
        a = a @ w + b
        if i < 3:
            a = torch.nn.functional.gelu(a, approximate="tanh")
    return a


def _loss(z, y):
    bce = torch.nn.functional.binary_cross_entropy_with_logits(z[:, 0], y[:, 0], reduction="none")
    q = y[:, 1:]
    ce = -(q * torch.log_softmax(z[:, 1:65], 1)).sum(1)
    return (bce + (q.sum(1) > 0).double() * ce).mean()


def _grad(w, x, y):
    w = w.detach().requires_grad_(True)
    loss = _loss(_logits(_unpack(w), x), y)
    g, = torch.autograd.grad(loss, w)
    mask = torch.ones_like(g)
    mask[-15:] = 0.0  # the output padding's biases are not parameters
    return float(loss.detach()), g * mask


def exact(case, seed):
    k = case["kind"]
    if k not in ("forward", "gradients", "train"):
        return None  # whole numbers and per-photon records: nothing to compute in 64 bits
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    w, x, y = (torch.from_numpy(v).to(dev, torch.float64)
               for v in _network_inputs(case, seed))
    if k == "forward":
        z = _logits(_unpack(w), x)
        out = torch.cat([torch.sigmoid(z[:, :1]), torch.softmax(z[:, 1:65], 1)], 1)
        return out.cpu().numpy()
    if k == "gradients":
        loss, g = _grad(w, x, y)
        return {"loss": loss, "grads": g.cpu().numpy()}
    # Adam on the minibatches that the training call draws (xorshift64*)
    mask, n, B = (1 << 64) - 1, case["data"], case["rows"]
    s = (0xD1B54A32D192ED03 ^ ((seed & 0xFFFFFFFF) << 17)) & mask
    m, v = torch.zeros_like(w), torch.zeros_like(w)
    losses = []
    for step in range(1, case["steps"] + 1):
        idx = np.empty(B, np.int64)
        for i in range(B):
            s ^= s >> 12
            s = (s ^ (s << 25)) & mask
            s ^= s >> 27
            idx[i] = (((s * 2685821657736338717) & mask) >> 32) % n
        at = torch.from_numpy(idx).to(dev)
        loss, g = _grad(w, x[at], y[at])
        losses.append(loss)
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        w = w - 1e-3 * (m / (1 - 0.9 ** step)) / ((v / (1 - 0.999 ** step)).sqrt() + 1e-8)
    return {"losses": np.array(losses), "params": w.cpu().numpy()}
