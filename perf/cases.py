"""Performance cases of the reconstruction engine: what its users run, over the sizes they run it at.

Each case is one pass of a path that a program of this package takes: ePIE, difference-map and MLs
iterations on a handle that holds its frames, the batched difference map, the warm-start network's
training and inference, and the simulator that forms its training frames.  The sizes are the
benchmark workloads' (``ptychopy_amd/workloads.py``), the Python surface's defaults and generic
ones between and below them.

``prepare`` builds a seeded synthetic experiment on the GPU (smooth random-field object, defocused
Gaussian or Hermite-Gaussian probe, raster scan with jitter, Poisson counts stored as FP16 with a
power-of-two scale per frame) and a handle that holds it; ``run`` is the pass; ``exact`` restates the
update equations in 64 bits with torch alone.
"""
from __future__ import annotations

import math

import numpy as np
import torch

DEV = "cuda"
C128, F64 = torch.complex128, torch.float64


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # The smallest reconstruction: a 6 x 6 alignment scan of 64^2 frames. Latency is all there is.
        dict(name="epie 64 6x6", kind="epie", m=64, side=6, step=8.0, modes=1, rms=False),
        # The plain ePIE benchmark workload with its Fourier error: 144 dependent positions of 128^2.
        dict(name="epie 128 12x12", kind="epie", m=128, side=12, step=16.0, modes=1, rms=True),
        # Multi-mode ePIE of a partially coherent beam on a 256^2 detector region.
        dict(name="epie 256 7x7 3 modes", kind="epie", m=256, side=7, step=30.7, modes=3, rms=False),
        # ePIE at the Python surface's default frame size, 512^2, on a small field of view.
        dict(name="epie 512 6x6", kind="epie", m=512, side=6, step=41.0, modes=1, rms=False),
        # Difference map on a small detector region: short launches.
        dict(name="dm 128 20x20", kind="dm", m=128, side=20, step=16.0, iters=5, update_probe=True),
        # The difference-map benchmark workload (30 x 30 positions of 512^2), bound by memory.
        dict(name="dm 512 30x30", kind="dm", m=512, side=30, step=17.76, iters=3, update_probe=True),
        # Independent scans of uneven size advanced together, as in a multi-sample queue.
        dict(name="batch of 4 scans", kind="batch", scans="20x128,27x256,13x512,33x128", iters=3),
        # MLs at the Python surface's default 26 x 26 scan on a small region: about 100 groups of 6
        # frames, launch-bound.
        dict(name="mls 128 26x26 3 modes", kind="mls", m=128, side=26, step=9.3, modes=3),
        # The headline workload: 51 x 51 positions of 256^2, five modes, position refinement.
        dict(name="mls 256 51x51 5 modes", kind="mls", m=256, side=51, step=14.0, modes=5),
        # Warm-start network: two Adam steps at the size and batch that the experiment trains with.
        dict(name="net train 256", kind="train", size=256, c=32, batch=16, steps=2),
        # Warm-start inference on a ragged number of raw frames.
        dict(name="net predict 256", kind="predict", size=256, c=32, batch=8, n=60),
        # The simulator forming one object's training frames.
        dict(name="simulate 256 x200", kind="simulate", m=256, n=200, canvas=611),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["epie", "epie", "dm", "dm", "batch", "mls", "mls", "train", "predict", "simulate"])
    if kind == "epie":
        m = rng.choice([64, 128, 256, 512])
        side = rng.randint(3, {64: 13, 128: 12, 256: 7, 512: 5}[m])
        return dict(kind=kind, m=m, side=side, step=round(m * rng.uniform(0.07, 0.14), 2),
                    modes=rng.randint(1, 3) if m < 512 else 1, rms=rng.random() < 0.5)
    if kind == "dm":
        m = rng.choice([64, 128, 256, 512])
        side = _log_int(rng, 5, {64: 51, 128: 51, 256: 41, 512: 27}[m])
        return dict(kind=kind, m=m, side=side, step=round(m * rng.uniform(0.04, 0.13), 2), iters=rng.randint(2, 4),
                    update_probe=rng.random() < 0.8)
    if kind == "batch":
        sizes = [rng.choice([128, 256]) for _ in range(rng.randint(2, 5))]
        return dict(kind=kind, scans=",".join("%dx%d" % (rng.randint(7, 29), m) for m in sizes),
                    iters=rng.randint(2, 4))
    if kind == "mls":
        m = rng.choice([64, 128, 256])
        side = _log_int(rng, 10, 39)
        return dict(kind=kind, m=m, side=side, step=round(m * rng.uniform(0.05, 0.08), 2), modes=rng.randint(1, 5))
    if kind == "train":
        return dict(kind=kind, size=rng.choice([64, 128, 256]), c=rng.choice([16, 32]), batch=rng.randint(2, 12),
                    steps=rng.randint(1, 2))
    if kind == "predict":
        return dict(kind=kind, size=rng.choice([64, 128, 256]), c=rng.choice([16, 32]), batch=rng.randint(3, 16),
                    n=rng.randint(1, 70))
    m = rng.choice([64, 128, 256])
    return dict(kind=kind, m=m, n=_log_int(rng, 10, 300), canvas=m + rng.randint(40, 500))


# ------------------------------------------------------------------ synthetic experiments
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 13)
    return g


def _smooth(x, sigma):
    """Gaussian filter with wrapped edges."""
    fy = torch.fft.fftfreq(x.shape[0], device=DEV, dtype=F64)[:, None]
    fx = torch.fft.fftfreq(x.shape[1], device=DEV, dtype=F64)[None, :]
    return torch.fft.ifft2(torch.fft.fft2(x) * torch.exp(-2 * math.pi ** 2 * sigma ** 2 * (fy ** 2 + fx ** 2))).real


def _object(rows, cols, g):
    amp = _smooth(0.8 + 0.2 * torch.rand(rows, cols, device=DEV, dtype=F64, generator=g), 4.0)
    ph = _smooth(torch.randn(rows, cols, device=DEV, dtype=F64, generator=g), 6.0)
    return torch.polar(amp, 0.5 * (ph - ph.mean()) / ph.std())


def _modes(m, k):
    """k orthogonal Hermite-Gaussian modes with a defocus phase, powers 0.6, 0.2, 0.1, 0.06, 0.04."""
    c = torch.arange(m, device=DEV, dtype=F64) - m / 2
    y, x = c[:, None], c[None, :]
    w = math.sqrt(2.0) * (m * 24.0 / 128.0) / (2 * math.sqrt(2 * math.log(2)))
    r2 = x * x + y * y
    base = torch.polar(torch.exp(-r2 / w ** 2), 2.0 * r2 / (m / 2) ** 2)
    u, v = math.sqrt(2) * x / w, math.sqrt(2) * y / w
    poly = [torch.ones_like(r2), u + 0 * v, v + 0 * u, (u * u - 0.5) + 0 * v, u * v][:k]
    out = []
    for p, power in zip(poly, (0.6, 0.2, 0.1, 0.06, 0.04)):
        f = base * p
        for o in out:
            f = f - o * (torch.sum(o.conj() * f) / torch.sum(o.abs() ** 2))
        out.append(f * torch.sqrt(power * torch.sum(base.abs() ** 2) / torch.sum(f.abs() ** 2)))
    return torch.stack(out)


def _diffuser(m, g):
    """A random phase plate in the beam: it spreads the pattern over the whole detector, as is done to
    keep dark pixels, and the phases that noise would decide there, few."""
    return torch.polar(torch.ones(m, m, device=DEV, dtype=F64),
                       0.6 * torch.randn(m, m, device=DEV, dtype=F64, generator=g))


def _raster(side, step, g, jitter=1.0):
    i = torch.arange(side, device=DEV, dtype=F64) * step
    p = torch.stack(torch.meshgrid(i, i, indexing="ij"), -1).reshape(-1, 2)
    return p + jitter * (2 * torch.rand(p.shape, device=DEV, dtype=F64, generator=g) - 1)


def _patches(obj, origin, m):
    """obj[r + 0..m, c + 0..m] for n integer origins."""
    o = torch.as_tensor(np.asarray(origin), device=DEV, dtype=torch.long)
    k = torch.arange(m, device=DEV)
    return obj[o[:, 0, None, None] + k[None, :, None], o[:, 1, None, None] + k[None, None, :]]


def _counts(obj, modes, origin, m, photons, g):
    """Poisson amplitudes sqrt(N) as FP16 halves and power-of-two scales, from the truth."""
    n = len(origin)
    halves = np.empty((n, m, m), np.float16)
    scales = np.empty(n, np.float32)
    o32, p32 = obj.to(torch.complex64), modes.to(torch.complex64)
    chunk = max(1, (1 << 25) // (m * m))
    for a in range(0, n, chunk):
        patch = _patches(o32, origin[a:a + chunk], m)
        inten = sum(torch.fft.fft2(patch * p).abs() ** 2 for p in p32)
        inten = inten * (photons / inten.sum(dim=(1, 2), keepdim=True))
        amp = torch.poisson(inten, generator=g).sqrt()
        sc = torch.exp2(torch.ceil(torch.log2(amp.amax(dim=(1, 2)).clamp_min(1.0))) - 15)
        halves[a:a + chunk] = (amp / sc[:, None, None]).to(torch.float16).cpu().numpy()
        scales[a:a + chunk] = sc.cpu().numpy()
    return halves, scales


def _scan(m, side, step, modes, seed):
    """A shifted-to-the-canvas scan (ePIE, DM): data, positions and a start a few iterations in: the
    object with weaker phases and no absorption, a probe 10 % off in size. (From a flat
    object the model's spectrum is nothing but rounding over most of the detector, whose phase the
    data then keep.)"""
    g = _gen(seed)
    pos = _raster(side, step, g)
    pos = (pos - pos.amin(dim=0) + 1.0).cpu().numpy().astype(np.float32)
    shape = 2 * (int(math.ceil((side - 1) * step + 3)) + m + 2,)  # the same for every seed
    photons = 100.0 * m * m
    obj, probe = _object(*shape, g), _modes(m, modes) * _diffuser(m, g)
    probe = probe * math.sqrt(photons / float(torch.sum(probe.abs() ** 2)) / (m * m))
    origin = np.floor(pos.astype(np.float64) + 0.5).astype(np.int64)
    halves, scales = _counts(obj, probe, origin, m, photons, g)
    c = torch.arange(m, device=DEV, dtype=F64) - m / 2
    taper = 1.0 + 0.1 * torch.exp(-(c[:, None] ** 2 + c[None, :] ** 2) / (m / 4) ** 2)
    return dict(m=m, n=len(pos), shape=shape, pos=pos, origin=origin, halves=halves, scales=scales,
                obj0=torch.polar(torch.full(shape, 0.9, device=DEV, dtype=F64), 0.7 * obj.angle()).to(
                    torch.complex64).cpu().numpy(),
                probe0=(probe * taper).to(torch.complex64).cpu().numpy())


def _mls_scan(case, seed):
    """An MLs scan: positions centred on the canvas, ROI origins round(pos + centre) - 1."""
    g = _gen(seed)
    m, k = case["m"], case["modes"]
    pos = _raster(case["side"], case["step"], g, 0.7)
    pos = (pos - (case["side"] - 1) / 2 * case["step"]).cpu().numpy().astype(np.float32)
    n = len(pos)
    rows = cols = int(math.ceil(1.2 * ((case["side"] - 1) * case["step"] + 1.4 + m)))
    centre = np.array([math.ceil(rows / 2 - m / 2), math.ceil(cols / 2 - m / 2)], np.float32)
    origin = np.floor(pos + centre + np.float32(0.5)).astype(np.int64) - 1
    obj, probe = _object(rows, cols, g), _modes(m, k) * _diffuser(m, g)
    halves, scales = _counts(obj, probe, origin, m, 100.0 * m * m, g)
    power = (halves.reshape(n, -1).astype(np.float32) ** 2).sum(axis=1, dtype=np.float64) * scales.astype(np.float64) ** 2
    vmode = torch.polar(torch.rand(m, m, device=DEV, dtype=F64, generator=g),
                        2 * math.pi * torch.rand(m, m, device=DEV, dtype=F64, generator=g))
    evo = 1e-6 * torch.randn(n, device=DEV, dtype=F64, generator=g)
    mn, mx = np.minimum(pos.min(axis=0), 0), np.maximum(pos.max(axis=0), 0)
    box = (int(round(rows * 0.5 + mn[0])), int(round(rows * 0.5 + mx[0])) - 1,
           int(round(cols * 0.5 + mn[1])), int(round(cols * 0.5 + mx[1])) - 1)
    rng = np.random.default_rng(seed)
    size = max(1, n // 100)  # the driver's partition: groups of about a hundredth of the scan
    parts = []
    for _ in range(4):
        idx = rng.permutation(n).astype(np.int32)
        parts.append([idx[i:i + size] for i in range(0, n, size)])
    near = _smooth(obj.real, 8.0) + 1j * _smooth(obj.imag, 8.0)  # a start that a few iterations have reached
    return dict(m=m, n=n, k=k, shape=(rows, cols), pos=pos, halves=halves, scales=scales, power=power, box=box,
                vmode=vmode.to(torch.complex64).cpu().numpy(), evo=evo.cpu().numpy(), parts=parts,
                obj0=near.to(torch.complex64).cpu().numpy(), probe0=probe.to(torch.complex64).cpu().numpy())


# the network's layers: (channels in, channels out, taps, resolution level)
def _layers(c):
    return [(1, c, 3), (c, c, 3), (c, 2 * c, 3), (2 * c, 2 * c, 3), (2 * c, 4 * c, 3), (4 * c, 4 * c, 3),
            (4 * c, 8 * c, 3), (8 * c, 8 * c, 3), (12 * c, 4 * c, 3), (4 * c, 4 * c, 3), (6 * c, 2 * c, 3),
            (2 * c, 2 * c, 3), (3 * c, c, 3), (c, c, 3), (c, 2, 1)]


_LEVEL = (0, 0, 1, 1, 2, 2, 3, 3, 2, 2, 1, 1, 0, 0, 0)


def _net_params(c, g):
    """He-normal weights and small biases, in the parameter vector's order (float32)."""
    out = []
    for ci, co, ks in _layers(c):
        out.append(torch.randn(co * ci * ks * ks, device=DEV, generator=g) * math.sqrt(2.0 / (ci * ks * ks)))
        out.append(0.02 * torch.randn(co, device=DEV, generator=g))
    return torch.cat(out)


def _frames_of(m, n, g):
    """n simulated frames' amplitudes and their object patches."""
    side = m + 200
    obj = _object(side, side, g)
    origin = torch.randint(0, side - m, (n, 2), device=DEV, generator=g).cpu().numpy()
    patch = _patches(obj, origin, m).to(torch.complex64)
    inten = torch.fft.fft2(patch * _modes(m, 1)[0].to(torch.complex64)).abs() ** 2
    amp = torch.poisson(inten * (1e5 / inten.sum(dim=(1, 2), keepdim=True)), generator=g).sqrt()
    return amp, patch


def _net_data(case, seed):
    g = _gen(seed)
    if case["kind"] == "predict":
        return dict(params=_net_params(case["c"], g), amp=_frames_of(case["size"], case["n"], g)[0])
    n = case["batch"] * case["steps"]
    params = _net_params(case["c"], g)
    amp, patch = _frames_of(case["size"], n, g)
    x = torch.log1p(amp)
    x = (x / x.amax(dim=(1, 2), keepdim=True)).to(torch.bfloat16).float()
    t = torch.stack([patch.abs(), patch.angle()], 1).to(torch.bfloat16).float()
    return dict(params=params, x=x, t=t)


def _sim_data(case, seed):
    g = _gen(seed)
    m = case["m"]
    obj = _object(case["canvas"], case["canvas"], g).to(torch.complex64)
    pos = torch.rand(case["n"], 2, device=DEV, dtype=F64, generator=g) * (case["canvas"] - m - 2) + 0.5
    return obj.cpu().numpy(), _modes(m, 1)[0].to(torch.complex64).cpu().numpy(), pos.cpu().numpy().astype(np.float32)


# ------------------------------------------------------------------ states
def _engine(d, modes):
    from ptychopy_amd._engine import Engine
    e = Engine(d["n"], d["m"], d["shape"], modes)
    e.set_frames_f16(d["halves"], d["scales"])
    return e


def _dm_engine(d):
    from ptychopy_amd import _engine as E
    e = _engine(d, 1)
    e.set_positions(d["pos"])
    e.set_object(d["obj0"])
    e.set_probe(d["probe0"])
    e.refresh_maxima()
    s = e.get_scalars()
    s[E.SCAL_DM_FACTOR_OBJ], s[E.SCAL_DM_FACTOR_PROBE] = 1.0 / s[E.SCAL_OBJ_MAX], 1.0 / s[E.SCAL_PROBE_MAX]
    return dict(engine=e, obj0=d["obj0"], probe0=d["probe0"], scal=s)


def _batch_scans(case, seed):
    out = []
    for i, t in enumerate(case["scans"].split(",")):
        side, m = (int(v) for v in t.split("x"))
        out.append(_scan(m, side, m / 8.0, 1, seed * 31 + i))
    return out


def prepare(case, seed):
    from ptychopy_amd import _engine as E
    kind = case["kind"]
    if kind == "epie":
        d = _scan(case["m"], case["side"], case["step"], case["modes"], seed)
        e = _engine(d, case["modes"])
        e.set_positions(d["pos"])
        e.set_object(d["obj0"])
        flags = E.FLAG_UPDATE_PROBE | (E.FLAG_RMS if case["rms"] else 0)
        e.set_probe(d["probe0"])
        if case["modes"] > 1:  # a multi-mode reconstruction that goes on from its own modes
            flags |= E.FLAG_UPDATE_MODES
            e.begin_modal()
            e.set_probe(d["probe0"])
        e.refresh_maxima()
        s = e.get_scalars()
        s[E.SCAL_PROBE_MAX] = float((np.abs(d["probe0"].astype(np.complex128)) ** 2).sum(axis=0).max())
        e.set_scalars(s)
        rng = np.random.default_rng(seed)
        return dict(kind=kind, engine=e, flags=flags, step=0, orders=[rng.permutation(d["n"]).astype(np.int32)
                                                                      for _ in range(8)])
    if kind == "dm":
        s = _dm_engine(_scan(case["m"], case["side"], case["step"], 1, seed))
        return dict(s, kind=kind, iters=case["iters"], flags=E.FLAG_UPDATE_PROBE if case["update_probe"] else 0)
    if kind == "batch":
        scans = [_dm_engine(d) for d in _batch_scans(case, seed)]
        return dict(kind=kind, scans=scans, batch=E.Batch([s["engine"] for s in scans]), iters=case["iters"],
                    flags=E.FLAG_UPDATE_PROBE)
    if kind == "mls":
        d = _mls_scan(case, seed)
        e = _engine(d, d["k"])
        e.set_object(d["obj0"])
        e.set_probe(d["probe0"])
        e.mls_begin(E.mls_config(d["box"]), d["pos"], d["vmode"], d["evo"], d["power"])
        # the pass is an iteration of the refinement stage: all updates are on from iteration 20
        return dict(kind=kind, engine=e, parts=d["parts"], it=20)
    if kind == "simulate":
        obj, probe, pos = _sim_data(case, seed)
        return dict(kind=kind, engine=E.Engine(1, case["m"], (case["m"], case["m"])), obj=obj, probe=probe, pos=pos)
    from ptychopy_amd.warmstart import Net
    d = _net_data(case, seed)
    net = Net(size=case["size"], c=case["c"], batch=case["batch"], seed=1)
    net.set_params(d["params"].cpu().numpy())
    if kind == "predict":
        return dict(kind=kind, net=net, amp=d["amp"].cpu().numpy())
    net.set_data(d["x"].cpu().numpy(), d["t"].cpu().numpy())
    return dict(kind=kind, net=net, order=np.arange(case["batch"] * case["steps"]))


# ------------------------------------------------------------------ the passes
def run(state):
    kind = state["kind"]
    if kind == "epie":  # one iteration over all positions, then the object and the probe
        e = state["engine"]
        err = e.epie_iteration(state["orders"][state["step"] % len(state["orders"])], state["flags"])
        state["step"] += 1
        return dict(object=e.get_object(), probe=e.get_probe(), error=np.array([err], np.float32))  # of 32-bit spectra
    if kind == "dm":  # a few iterations from the given object and probe
        e = state["engine"]
        e.set_object(state["obj0"])
        e.set_probe(state["probe0"])
        e.set_scalars(state["scal"])
        for _ in range(state["iters"]):
            e.dm_iteration(state["flags"])
        return dict(object=e.get_object(), probe=e.get_probe())
    if kind == "batch":
        for s in state["scans"]:
            s["engine"].set_object(s["obj0"])
            s["engine"].set_probe(s["probe0"])
            s["engine"].set_scalars(s["scal"])
        for _ in range(state["iters"]):
            state["batch"].dm_iteration(state["flags"])
        state["batch"].synchronize()
        return [dict(object=s["engine"].get_object(), probe=s["engine"].get_probe()) for s in state["scans"]]
    if kind == "mls":  # the next iteration over all groups
        e, it = state["engine"], state["it"]
        state["it"] = it + 1
        e.mls_iteration(it, state["parts"][it % len(state["parts"])])
        return dict(object=e.get_object(), probe=e.get_probe())
    if kind == "train":
        state["net"].train(state["order"], 1e-3)
        return state["net"].get_params()
    if kind == "predict":
        return state["net"].predict_amplitudes(state["amp"])
    return state["engine"].simulate(state["obj"], state["probe"], state["pos"])


def _shape_of(case):
    """Frames and (about) the canvas pixels of a scan."""
    return case["side"] ** 2, (case["side"] * case["step"] + case["m"] + 2) ** 2


def work(case):
    kind = case["kind"]
    if kind in ("epie", "dm", "mls"):
        (n, canvas), m, k = _shape_of(case), case["m"], case.get("modes", 1)
        fft = 10.0 * m * m * math.log2(m)
        if kind == "epie":  # frames and arrays once
            return dict(bytes=2.0 * n * m * m + 16 * canvas + 16 * k * m * m, flops=n * k * (2 * fft + 40 * m * m))
        if kind == "dm":  # per iteration: frames and exit waves in, exit waves out, arrays in and out
            return dict(bytes=case["iters"] * (18.0 * n * m * m + 16 * canvas + 16 * m * m),
                        flops=case["iters"] * n * (2 * fft + 60 * m * m))
        groups = math.ceil(n / max(1, n // 100))
        return dict(bytes=2.0 * n * m * m + 36 * 1.44 * canvas * groups, flops=n * (2 * k + 4) * fft)
    if kind == "batch":
        b = f = 0.0
        for t in case["scans"].split(","):
            side, m = (int(v) for v in t.split("x"))
            w = work(dict(kind="dm", m=m, side=side, step=m / 8.0, iters=case["iters"]))
            b, f = b + w["bytes"], f + w["flops"]
        return dict(bytes=b, flops=f)
    if kind == "simulate":
        m, n = case["m"], case["n"]
        return dict(bytes=4.0 * n * m * m + 8 * case["canvas"] ** 2, flops=n * (10.0 * m * m * math.log2(m) + 30 * m * m))
    s, c = case["size"], case["c"]
    flops = sum(2.0 * ci * co * ks * ks * (s >> lv) ** 2 for (ci, co, ks), lv in zip(_layers(c), _LEVEL))
    par = sum(ci * co * ks * ks + co for ci, co, ks in _layers(c))
    # activations of the 15 layers written once and read once (BF16), the samples and the parameters
    act = sum(4.0 * co * (s >> lv) ** 2 for (ci, co, ks), lv in zip(_layers(c), _LEVEL))
    if kind == "predict":
        return dict(bytes=case["n"] * (12.0 * s * s + act) + 4 * par, flops=case["n"] * flops)
    n = case["batch"] * case["steps"]
    return dict(bytes=n * (6.0 * s * s + 3 * act) + case["steps"] * 28.0 * par, flops=3 * n * flops)


# ------------------------------------------------------------------ the same in 64 bits
def _c(a):
    return torch.as_tensor(a, device=DEV).to(C128)


def _amps(d, frames):
    return torch.as_tensor(d["halves"][frames], device=DEV).to(F64) * torch.as_tensor(d["scales"][frames], device=DEV).to(
        F64)[:, None, None]


def _bilinear(obj, pos, m):
    """obj at (pos.row + i, pos.col + j), linear weights from float32 coordinates, clamped edges."""
    rows, cols = obj.shape
    r = np.arange(m, dtype=np.float32) + np.float32(pos[0]) + np.float32(0.5) - np.float32(0.5)
    q = np.arange(m, dtype=np.float32) + np.float32(pos[1]) + np.float32(0.5) - np.float32(0.5)
    r0, q0 = np.floor(r), np.floor(q)
    be = torch.as_tensor((r - r0).astype(np.float64), device=DEV)[:, None]
    al = torch.as_tensor((q - q0).astype(np.float64), device=DEV)[None, :]
    ix = [torch.as_tensor(np.clip(r0.astype(np.int64) + o, 0, rows - 1), device=DEV) for o in (0, 1)]
    jx = [torch.as_tensor(np.clip(q0.astype(np.int64) + o, 0, cols - 1), device=DEV) for o in (0, 1)]
    t = [[obj[i][:, j] for j in jx] for i in ix]
    return (1 - be) * ((1 - al) * t[0][0] + al * t[0][1]) + be * ((1 - al) * t[1][0] + al * t[1][1])


def _exact_epie(case, seed):
    d = _scan(case["m"], case["side"], case["step"], case["modes"], seed)
    m, k, n = case["m"], case["modes"], d["n"]
    obj, p = _c(d["obj0"]), _c(d["probe0"])
    order = np.random.default_rng(seed).permutation(n)
    pint = p.abs() ** 2
    pmax, omax = pint.sum(dim=0).max(), None
    oint = obj.abs() ** 2
    err = 0.0
    for f in order:
        a = _amps(d, [f])[0]
        old = _bilinear(obj, d["pos"][f], m) * p
        F = torch.fft.fft2(old)
        mod = (F.abs() ** 2).sum(dim=0).sqrt()
        unit = torch.where(mod > 0, F / mod.clamp_min(1e-300), torch.ones_like(F) if k == 1 else torch.zeros_like(F))
        delta = torch.fft.ifft2(a * unit) - old
        r, c = d["origin"][f]
        o = obj[r:r + m, c:c + m] + (p.conj() * delta).sum(dim=0) / pmax
        obj[r:r + m, c:c + m] = o
        oint[r:r + m, c:c + m] = o.abs() ** 2
        omax = oint.max()
        p = p + o.conj() * delta / omax
        pmax = (p.abs() ** 2).sum(dim=0).max()
        if case["rms"]:
            err += float((a - F.sum(dim=0).abs()).abs().sum() / a.sum()) / k
    return dict(object=obj.cpu().numpy(), probe=p.cpu().numpy(), error=np.array([err / n], np.float32))


def _exact_dm(d, iters, update):
    m, n = d["m"], d["n"]
    obj, p = _c(d["obj0"]), _c(d["probe0"])[0]
    fo, fp = np.float32(1.0 / float((obj.abs() ** 2).max())), np.float32(1.0 / float((p.abs() ** 2).max()))
    psi = torch.zeros(n, m, m, device=DEV, dtype=C128)
    chunk = max(1, (1 << 24) // (m * m))
    for _ in range(iters):
        dobj, dp = torch.zeros_like(obj), torch.zeros_like(p)
        for a in range(0, n, chunk):
            fr = np.arange(a, min(n, a + chunk))
            op = _patches(obj, d["origin"][fr], m)
            x = 2 * p * op - psi[a:a + chunk]
            F = torch.fft.fft2(x)
            mod = F.abs()
            F = _amps(d, fr) * torch.where(mod > 0, F / mod.clamp_min(1e-300), torch.ones_like(F))
            psi[a:a + chunk] = torch.fft.ifft2(F) - x
            u = p.conj() * psi[a:a + chunk] * float(fp)
            for j, f in enumerate(fr):
                r, c = d["origin"][f]
                dobj[r:r + m, c:c + m] += u[j]
            if update:
                dp += (op.conj() * psi[a:a + chunk]).sum(dim=0) * float(fo)
        obj, p = obj + dobj, p + dp
        for was, s in ((0, obj), (1, p)):
            new = np.float32(1.0 / float((s.abs() ** 2).sum()))
            if was == 0 and abs(fo - new) > 1e-3:
                fo = new
            if was == 1 and abs(fp - new) > 1e-3:
                fp = new
    return dict(object=obj.cpu().numpy(), probe=p[None].cpu().numpy())


def _exact_mls(case, seed):
    """ptyk_mls_begin's normalisation and iteration 20 over the scan's groups."""
    d = _mls_scan(case, seed)
    m, n, k, (rows, cols) = d["m"], d["n"], d["k"], d["shape"]
    mm = float(m * m)
    kk = torch.arange(m, device=DEV)
    centre = np.array([math.ceil(rows / 2 - m / 2), math.ceil(cols / 2 - m / 2)], np.float32)
    shifted = d["pos"] + centre
    near = np.floor(shifted + np.float32(0.5))
    roi = torch.as_tensor(near.astype(np.int64) - 1, device=DEV)
    sub = torch.as_tensor((shifted - near)[:, ::-1].astype(np.float64).copy(), device=DEV)  # (column, row)

    def at(f):
        r = roi[f]
        return r[:, 0, None, None] + kk[None, :, None], r[:, 1, None, None] + kk[None, None, :]

    def cover(w):
        out = torch.zeros(rows, cols, device=DEV, dtype=F64)
        for r, c in roi.tolist():
            out[r:r + m, c:c + m] += w
        return out

    obj, p, v = _c(d["obj0"]), _c(d["probe0"]), _c(d["vmode"])
    e0 = torch.ones(n, device=DEV, dtype=F64)
    e1 = torch.as_tensor(d["evo"], device=DEV)
    rv = (v.abs() ** 2).mean().sqrt()
    v, e1 = v / rv, e1 * rv
    illum = cover(p[0].abs() ** 2)
    obj = obj / ((illum * obj.abs() ** 2).sum() / illum.sum()).sqrt()
    corr = np.sort(float((p.abs() ** 2).sum()) / mm / (d["power"] / mm))
    med = (corr[n // 2 - 1] + corr[n // 2]) / 2 if n % 2 == 0 else corr[n // 2]
    cr = math.sqrt(med * mm)
    p, v, illum = p / cr, v / cr, illum / cr ** 2
    max_illum = float(illum.max())

    # the iteration's own steps: object norm over the box, the evolution's extra degree, illumination
    b = d["box"]
    w = illum[b[0] - 1:b[1], b[2] - 1:b[3]]
    o = obj[b[0] - 1:b[1], b[2] - 1:b[3]]
    norm = ((o * w).abs() ** 2).mean().sqrt() / (w ** 2).mean().sqrt()
    p, v, obj = p * norm, v * norm, obj / norm
    rv = (v.abs() ** 2).mean().sqrt()
    v, e1 = v / rv, e1 * rv
    h = min(2, n)
    e0[:h] = (e0[:h] - float(np.float32(float(e0[:h].mean())))) * 0.99 + 1
    e1[:h] = e1[:h] - float(np.float32(float(e1[:h].mean())))
    cn = (e0[:h] ** 2).mean().sqrt()
    e0[:h] /= cn
    p[0] = p[0] * cn
    illum = (illum + cover(p[0].abs() ** 2)) / 2

    fr = ((torch.arange(m, device=DEV) + m // 2) % m).to(F64) / m - 0.5

    def ramp(f, sign):
        ph = sub[f, 0][:, None, None] * fr[None, None, :] + sub[f, 1][:, None, None] * fr[None, :, None]
        return torch.polar(torch.ones_like(ph), -2 * math.pi * sign * ph)

    lam = float(np.float32(1.1920928955078125e-07 / mm)) * mm
    for grp in d["parts"][20 % len(d["parts"])]:
        f = torch.as_tensor(grp.astype(np.int64), device=DEV)
        G = len(grp)
        ix = at(f)
        op = obj[ix]
        vp = torch.fft.ifft2(torch.fft.fft2(e0[f][:, None, None] * p[0] + e1[f][:, None, None] * v) * ramp(f, 1))
        psi = [torch.fft.fft2(op * vp)] + [torch.fft.fft2(q * op) for q in p[1:]]
        ap = sum(s.abs() ** 2 for s in psi).sqrt()
        R = _amps(d, grp) / (ap + 1e-9) - 1
        chi = [torch.fft.ifft2(s * R) for s in psi]
        wt = illum[ix] / (illum[ix] + 0.01 * max_illum)
        pu = torch.fft.ifft2(torch.fft.fft2(chi[0] * op.conj()) * ramp(f, -1))
        pum = (wt * pu).mean(dim=0)
        upd = torch.full((rows, cols), complex(0.0, float(np.float32(2.220446049250313e-16))), device=DEV, dtype=C128)
        contrib = chi[0] * vp.conj()
        for j, (r, c) in enumerate(roi[f].tolist()):
            upd[r:r + m, c:c + m] += contrib[j]
        upd = upd / (illum + 0.1 * max_illum)
        dop, dpo = upd[ix] * vp, pum * op
        s = lambda t: t.sum(dim=(1, 2))  # noqa: E731
        a1, a4 = s(dop.abs() ** 2) + lam, s(dpo.abs() ** 2) + lam
        a2 = s(dop * dpo.conj())
        b1, b2 = s((dop.conj() * chi[0]).real), s((dpo.conj() * chi[0]).real)
        A11, A22 = a1 + 0.1 * a1.mean(), a4 + 0.1 * a4.mean()
        det = A11 * A22 - a2 * a2.conj()
        bo = 0.9 * ((b1 * A22 - a2 * b2) / det).mean()
        bp = 0.9 * ((A11 * b2 - a2.conj() * b1) / det).mean()
        obj = obj + upd * bo
        p = p.clone()
        p[0] = p[0] + pum * bp
        # variable probe: the mode, then the two coefficients (the position step moves nothing that
        # this iteration still reads)
        wn = illum[ix] / illum.max()
        img = wn * (pu - pum)
        cj = ((v * img.conj()).real.mean(dim=(1, 2)) + e1[f]) / (e1[f] ** 2).sum()
        U = (img * cj[:, None, None]).sum(dim=0) / mm
        v = v + U * (G / n) / max(1.0, float((U.abs() ** 2).mean().sqrt()))
        v = v / (v.abs() ** 2).mean().sqrt()
        ov = op * v
        den, num = (ov.abs() ** 2).mean(dim=(1, 2)), (chi[0] * ov.conj()).real.mean(dim=(1, 2))
        e1[f] = e1[f] + num / (den + 0.1 * den.mean())
        ov = op * p[0]
        e0[f] = e0[f] + 0.1 * s((chi[0] * ov.conj()).real) / s(ov.abs() ** 2)
        for q in range(1, k):
            p[q] = p[q] + (wt * chi[q] * op.conj()).mean(dim=0) * bp
    if k > 1:
        power = [float((q.abs() ** 2).sum()) for q in p]
        for i in range(k):
            for j in range(i):
                p[i] = p[i] - p[j] * ((p[i] * p[j].conj()).sum() / (p[j].abs() ** 2).sum())
        by = sorted(range(k), key=lambda i: -power[i])
        p = torch.stack([p[0]] + [p[by[i]] for i in range(1, k)])
    return dict(object=obj.cpu().numpy(), probe=p.cpu().numpy())


def _conv(x, wt, bias):
    """3 x 3 (or 1 x 1) correlation with zero edges, one sample: x (C, S, S)."""
    co, ci, ks, _ = wt.shape
    s = x.shape[-1]
    if ks == 1:
        return (wt[:, :, 0, 0] @ x.reshape(ci, -1)).reshape(co, s, s) + bias[:, None, None]
    xp = torch.nn.functional.pad(x, (1, 1, 1, 1))
    out = bias[:, None] + 0 * x[0].reshape(1, -1)
    for dy in range(3):
        for dx in range(3):
            out = out + wt[:, :, dy, dx] @ xp[:, dy:dy + s, dx:dx + s].reshape(ci, -1)
    return out.reshape(co, s, s)


def _net_forward(x, params, c):
    at, layers = 0, []
    for ci, co, ks in _layers(c):
        layers.append((params[at:at + co * ci * ks * ks].reshape(co, ci, ks, ks),
                       params[at + co * ci * ks * ks:at + co * ci * ks * ks + co]))
        at += co * ci * ks * ks + co
    f = lambda i, t: torch.relu(_conv(t, *layers[i]))  # noqa: E731
    pool = lambda t: torch.nn.functional.max_pool2d(t[None], 2)[0]  # noqa: E731
    up = lambda t: t.repeat_interleave(2, 1).repeat_interleave(2, 2)  # noqa: E731
    s0 = f(1, f(0, x[None]))
    s1 = f(3, f(2, pool(s0)))
    s2 = f(5, f(4, pool(s1)))
    t = f(7, f(6, pool(s2)))
    t = f(9, f(8, torch.cat([up(t), s2])))
    t = f(11, f(10, torch.cat([up(t), s1])))
    t = f(13, f(12, torch.cat([up(t), s0])))
    return _conv(t, *layers[14])


def _exact_net(case, seed):
    d = _net_data(case, seed)
    params = d["params"].to(F64)
    if case["kind"] == "predict":
        x = torch.log1p(d["amp"].to(F64))
        x = x / x.amax(dim=(1, 2), keepdim=True)
        with torch.no_grad():
            return np.stack([_net_forward(q, params, case["c"]).cpu().numpy() for q in x])
    x, t, B = d["x"].to(F64), d["t"].to(F64), case["batch"]
    mo, ve = torch.zeros_like(params), torch.zeros_like(params)
    for step in range(case["steps"]):
        g = torch.zeros_like(params)
        for i in range(step * B, step * B + B):
            w = params.clone().requires_grad_(True)
            loss = ((_net_forward(x[i], w, case["c"]) - t[i]) ** 2).sum() / (B * 2 * case["size"] ** 2)
            g += torch.autograd.grad(loss, w)[0]
        mo, ve = 0.9 * mo + 0.1 * g, 0.999 * ve + 0.001 * g * g
        params = params - 1e-3 * (mo / (1 - 0.9 ** (step + 1))) / ((ve / (1 - 0.999 ** (step + 1))).sqrt() + 1e-8)
    return params.cpu().numpy()


def _exact_simulate(case, seed):
    obj, probe, pos = _sim_data(case, seed)
    o, p = _c(obj), _c(probe)
    return np.stack([torch.fft.fft2(_bilinear(o, q, case["m"]) * p).abs().cpu().numpy() for q in pos])


def exact(case, seed):
    kind = case["kind"]
    if kind == "epie":
        return _exact_epie(case, seed)
    if kind == "dm":
        return _exact_dm(_scan(case["m"], case["side"], case["step"], 1, seed), case["iters"], case["update_probe"])
    if kind == "batch":
        return [_exact_dm(d, case["iters"], True) for d in _batch_scans(case, seed)]
    if kind == "mls":
        return _exact_mls(case, seed)
    if kind == "simulate":
        return _exact_simulate(case, seed)
    return _exact_net(case, seed)
