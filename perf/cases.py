"""Performance cases: the work that map-making users have this package do.

A user has boresight pointing, one timestream and one inverse noise spectrum
per detector, and wants I/Q/U maps: a context is created and fed, the samples
are pixelised, the set-up makes the right-hand side and the preconditioner, and
CG iterations apply A = P^T N^-1 P.  The cases cover each of these entry
points, from a few thousand samples (where launches and host calls count) to
the 16-detector NSIDE-512 run, in both precisions, with power-of-two and
3 x 2^l / 5 x 2^l segments, odd segment counts, detectors that share the
boresight's line of sight and detectors at their own focal-plane offsets, one
segment length for all detectors and one for each.

The pointing of a case is fixed by its sizes (so that the seen pixels are);
the seed draws the sky, the detectors' noise levels, knees, slopes and
orientations, the timestreams and the trial maps.
"""
import ctypes
import math

import numpy as np
import torch
import torch.nn.functional as F

import sanepic_amd

FSAMP = 19.0
TWO_PI = 2.0 * math.pi
DEV = "cuda" if torch.cuda.is_available() else "cpu"


# ------------------------------------------------------------------- the cases
def _case(kind, nside, ndet, nseg, ns, **kw):
    c = dict(kind=kind, nside=nside, ndet=ndet, nseg=nseg, ns=ns, mixed=False, precond="diag",
             offsets="none", hwp=False, iters=0, lens="")
    c.update(kw)
    return c


def listed():
    return [
        # one operator application inside a caller's own iteration, at test size: pure latency
        dict(_case("apply", 16, 2, 3, 1024), name="apply small"),
        # the same on a radix-5 length with an odd segment count, four-step passes of moderate size
        dict(_case("apply", 128, 3, 5, 5 * 2 ** 13, offsets="spread"), name="apply radix 5"),
        # a single bolometer's map (1 detector, NSIDE 64, 8 segments of 2^19): the drop-in's default solver
        dict(_case("solve", 64, 1, 8, 2 ** 19, iters=11), name="solve 1 detector"),
        # short segments (single-pass transforms) of a small array: launch-bound iterations
        dict(_case("solve", 64, 4, 24, 2048, precond="block", iters=21), name="solve short segments"),
        # the 16-detector NSIDE-512 run with 2^20-sample segments, a quarter of its length: FP64 block-Jacobi
        dict(_case("solve", 512, 16, 16, 2 ** 20, precond="block", iters=11), name="solve 16 detectors fp64"),
        # the same in mixed precision
        dict(_case("solve", 512, 16, 8, 2 ** 20, precond="block", mixed=True, iters=11),
             name="solve 16 detectors mixed"),
        # a focal plane of detector pairs at their own offsets, odd segment count
        dict(_case("solve", 256, 6, 5, 2 ** 19, offsets="pairs", iters=11), name="solve offset pairs fp64"),
        # single detectors at their own offsets, radix-3 segments, mixed precision
        dict(_case("solve", 256, 5, 9, 3 * 2 ** 16, offsets="spread", mixed=True, iters=11),
             name="solve offsets mixed"),
        # every detector with its own segment length on one timeline
        dict(_case("solve", 256, 12, 0, 2 ** 21, precond="block", iters=11,
                   lens="65536 98304 131072 163840 196608 262144 65536 327680 131072 393216 524288 262144"),
             name="solve per-detector lengths"),
        # a whole run from host buffers to maps, as the drop-in executable makes it, with a half-wave plate
        dict(_case("map", 128, 4, 6, 2 ** 17, hwp=True, iters=5), name="map from host buffers"),
        # one pass of the relative calibration loop: new gains, a warm-started solve, the gain fit
        dict(_case("recal", 64, 4, 12, 2 ** 16, iters=5), name="recalibration pass"),
        # a training step of the preconditioner's network: forward and every parameter's gradient
        dict(_case("unet", 64, 0, 0, 0), name="network gradient"),
    ]


def _fits(c):
    n = _lengths(c)
    tot = sum(L * s for L, s in n)
    return tot <= 2 ** 28 and 12 * c["nside"] ** 2 <= max(3072, max(L * s for L, s in n) // 2)


def draw(rng):
    while True:
        kind = rng.choices(["solve", "apply", "map", "uneven", "leak", "recal", "unet"], [10, 4, 4, 4, 2, 2, 1])[0]
        if kind == "unet":
            return _case("unet", rng.choice([64, 128]), 0, 0, 0, iters=rng.randrange(1000))
        l2 = rng.uniform(10, 20)
        ns = 2 ** int(l2)
        if ns >= 2 ** 14 and rng.random() < 0.4:
            ns = rng.choice([3, 5]) * 2 ** max(13, int(l2) - 2)
        ndet = max(1, round(2 ** rng.uniform(0, 4)))
        nseg = max(1, round(2 ** rng.uniform(0, 4.3)))
        if kind in ("map", "recal"):
            ndet, ns = min(ndet, 6), min(ns, 2 ** 17)
        nside = rng.choice([8, 16, 32, 64, 128, 256, 512, 48, 100, 200])
        offsets = rng.choice(["none", "none", "pairs", "spread"])
        mixed = rng.random() < 0.4
        block = offsets == "none" and ndet >= 3 and rng.random() < 0.6
        c = _case("solve" if kind == "uneven" else kind, nside, ndet, nseg, ns, offsets=offsets, mixed=mixed,
                  precond="block" if block else "diag", iters=rng.choice([6, 11, 16]))
        if kind == "uneven":
            T = 2 ** rng.randint(17, 21)
            lens = []
            for _ in range(max(3, ndet)):
                m, l = rng.choice([1, 3, 5]), rng.randint(13, 18)
                lens.append(min(m * 2 ** l, T))
            c.update(ndet=len(lens), nseg=0, ns=T, lens=" ".join(str(v) for v in lens), offsets="none",
                     precond="diag")
        elif kind == "apply":
            c.update(iters=0, precond="diag")
        elif kind == "map":
            c.update(hwp=rng.random() < 0.5, mixed=False, precond="diag", iters=5)
        elif kind == "leak":
            c.update(mixed=False, precond="diag", ndet=max(3, ndet), iters=6)
        elif kind == "recal":
            c.update(mixed=False, precond="diag", iters=5)
        if _fits(c):
            return c


def _lengths(c):
    """(segment length, segments) of every detector."""
    if c["lens"]:
        return [(int(v), c["ns"] // int(v)) for v in c["lens"].split()]
    return [(c["ns"], c["nseg"])] * c["ndet"]


# ------------------------------------------------------------------ the inputs
def _scan(nsamp):
    """Boresight (ra, dec, psi): a spin about an axis that precesses about the
    anti-solar direction.  Short streams scan faster, so that pixels are
    revisited at several angles as in a long survey."""
    minutes = nsamp / FSAMP / 60.0
    spin, prec = min(20.0, minutes / 40.0), min(192.0, minutes / 5.0)
    t = torch.arange(nsamp, dtype=torch.float64, device=DEV) / FSAMP
    ps, pp = t * (TWO_PI / (spin * 60.0)), t * (TWO_PI / (prec * 60.0))
    lam = t * (TWO_PI / (365.25 * 86400.0))
    sb, cb, sa = math.sin(math.radians(50.0)), math.cos(math.radians(50.0)), math.sin(math.radians(45.0))
    bx, by = sb * torch.cos(ps), sb * torch.sin(ps)
    x1, z1 = sa * bx + sa * cb, -sa * bx + sa * cb  # tilt by 45 degrees: cos = sin
    x2, y2 = torch.cos(pp) * x1 - torch.sin(pp) * by, torch.sin(pp) * x1 + torch.cos(pp) * by
    x4, y4 = torch.cos(lam) * z1 - torch.sin(lam) * y2, torch.sin(lam) * z1 + torch.cos(lam) * y2
    ra = torch.remainder(torch.atan2(y4, x4), TWO_PI)
    ra = torch.where(ra <= 0.0, torch.full_like(ra, TWO_PI), ra)
    dec = 0.5 * math.pi - torch.acos(torch.clamp(-x2, -1.0, 1.0))
    psi = torch.atan2(torch.sin(ps), torch.cos(ps))
    psi = torch.where(psi <= -math.pi, torch.full_like(psi, math.pi), psi)
    return ra, dec, psi


def _offsets(c):
    """Focal-plane offsets in degrees (fixed: they decide the seen pixels)."""
    n = c["ndet"]
    if c["offsets"] == "pairs":  # two detectors behind each horn
        return [(0.35 * math.cos(2.0 * (k // 2) + 0.3), 0.5 * math.sin(2.0 * (k // 2) + 0.3)) for k in range(n)]
    if c["offsets"] == "spread":
        return [(0.4 * math.cos(1.7 * k + 0.2), 0.45 * math.sin(1.1 * k + 0.4)) for k in range(n)]
    return [(0.0, 0.0)] * n


def _detectors(c, seed):
    """Per detector: offsets, orientation, noise level, knee and slope."""
    r = np.random.default_rng([seed, 1])
    out = []
    for k, ((lel, xel), (L, nseg)) in enumerate(zip(_offsets(c), _lengths(c))):
        out.append(dict(lel=lel, xel=xel, angle=22.5 * k + (90.0 * (k % 2) if c["offsets"] == "pairs" else 0.0)
                        + float(r.uniform(-2.0, 2.0)), sigma=50e-6 * float(r.uniform(0.8, 1.25)),
                        fknee=float(r.uniform(0.05, 0.2)), alpha=float(r.uniform(0.8, 1.2)), L=L, nseg=nseg))
    return out


def _ispf(d):
    k = np.arange(d["L"], dtype=np.float64)
    k = np.minimum(k, d["L"] - k)
    k[0] = 1.0
    return 1.0 / (d["sigma"] ** 2 * (1.0 + (d["fknee"] / (k * FSAMP / d["L"])) ** d["alpha"]))


def _generator(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1000003 + stream) & 0x7FFFFFFF)
    return g


def _data(c, seed):
    """Everything a run reads: pointing, detectors and timestreams (numpy),
    each timestream a sky of smooth patches seen along the boresight plus
    white and 1/f noise."""
    dets = _detectors(c, seed)
    T = c["ns"] if c["lens"] else c["nseg"] * c["ns"]
    ra, dec, psi = _scan(T)
    r = np.random.default_rng([seed, 2])
    sky = torch.zeros((3, T), dtype=torch.float64, device=DEV)
    for s, amp in enumerate((1e-4, 1e-5, 1e-5)):
        for _ in range(6):
            m, n, ph = int(r.integers(1, 12)), int(r.integers(1, 12)), float(r.uniform(0, TWO_PI))
            sky[s] += amp * torch.cos(m * ra + ph) * torch.cos(n * dec + 0.7 * ph)
    tods = []
    for k, d in enumerate(dets):
        n = d["L"] * d["nseg"]
        w = torch.randn((d["nseg"], d["L"]), dtype=torch.float64, device=DEV, generator=_generator(seed, k + 10))
        f = torch.arange(d["L"] // 2 + 1, dtype=torch.float64, device=DEV) * (FSAMP / d["L"])
        f[0] = f[1]
        noise = torch.fft.irfft(torch.fft.rfft(w * d["sigma"]) * torch.sqrt(1.0 + (d["fknee"] / f) ** d["alpha"]),
                                d["L"]).reshape(-1)
        a2 = 2.0 * (psi[:n] + math.radians(d["angle"]))
        tod = sky[0, :n] + sky[1, :n] * torch.cos(a2) + sky[2, :n] * torch.sin(a2) + noise
        tods.append(tod.cpu().numpy())
    return dict(dets=dets, ra=ra.cpu().numpy(), dec=dec.cpu().numpy(), psi=psi.cpu().numpy(), tod=tods,
                ispf=[_ispf(d) for d in dets], relf=_relf(c, seed), gains=_gains(c, seed))


def _relf(c, seed):
    """Leakage coefficients, zero mean and unit variance over the detectors."""
    v = np.random.default_rng([seed, 3]).standard_normal(max(2, c["ndet"]))
    return ((v - v.mean()) / v.std())[:c["ndet"]]


def _gains(c, seed):
    return np.random.default_rng([seed, 4]).uniform(0.9, 1.1, (c["ndet"], max(1, c["nseg"])))


OMEGA_HWP = 0.0482


def _context(c):
    prec = sanepic_amd.MIXED if c["mixed"] else sanepic_amd.FP64
    if c["lens"]:
        return sanepic_amd.Context.uneven(c["nside"], [L for L, _ in _lengths(c)], c["ns"], precision=prec)
    return sanepic_amd.Context(c["nside"], c["ndet"], c["nseg"], c["ns"], hwp=1 if c["hwp"] else 0,
                               omega=OMEGA_HWP if c["hwp"] else 0.0, precision=prec)


def _feed(ctx, c, data):
    for k, d in enumerate(data["dets"]):
        ctx.set_detector(k, d["lel"], d["xel"], d["angle"], data["ispf"][k])
    if c["lens"]:
        ctx.set_pointing_range(0, data["ra"], data["dec"], data["psi"])
        for k, t in enumerate(data["tod"]):
            ctx.set_tod_range(k, 0, t)
        return
    ns = c["ns"]
    for s in range(c["nseg"]):
        sl = slice(s * ns, (s + 1) * ns)
        ctx.set_pointing(s, data["ra"][sl], data["dec"][sl], data["psi"][sl])
    for k, t in enumerate(data["tod"]):
        for s in range(c["nseg"]):
            ctx.set_tod(k, s, t[s * ns:(s + 1) * ns])


def _trial_map(c, seed, n):
    """A trial vector of a caller's iteration, block layout."""
    return np.random.default_rng([seed, 5]).standard_normal(n) * 1e-4


def _pinned(a, keep):
    """A copy in pinned host memory, as the drop-in reads its files into."""
    p = ctypes.c_void_p()
    if sanepic_amd.lib().sanepic_host_alloc(a.nbytes, ctypes.byref(p)):
        raise RuntimeError("pinned allocation failed")
    keep.append(p)
    out = np.ctypeslib.as_array((ctypes.c_double * a.size).from_address(p.value))
    out[:] = a
    return out


class _Pins(list):
    def __del__(self):
        for p in self:
            sanepic_amd.lib().sanepic_host_free(p)


def prepare(case, seed):
    c = dict(case)
    if c["kind"] == "unet":
        u = sanepic_amd.UNet(c["nside"])
        p, x, dy = _unet_inputs(c, seed, u.nparams)
        u.set_params(p)
        return dict(case=c, unet=u, x=x, dy=dy)
    data = _data(c, seed)
    if c["kind"] == "map":
        keep = _Pins()
        for key in ("ra", "dec", "psi"):
            data[key] = _pinned(data[key], keep)
        data["tod"] = [_pinned(t, keep) for t in data["tod"]]
        return dict(case=c, data=data, keep=keep)
    ctx = _context(c)
    _feed(ctx, c, data)
    if c["kind"] == "leak":
        ctx.set_leakage(data["relf"])
    npix, _ = ctx.pixelize()
    if c["kind"] == "recal":
        ctx.set_recalib(True)
    ctx.setup()
    state = dict(case=c, ctx=ctx)
    if c["kind"] == "apply":
        state["x"] = _trial_map(c, seed, 3 * npix)
    if c["kind"] == "recal":
        state["gains"] = data["gains"]
        state["x0"] = _trial_map(c, seed, 3 * npix)
    return state


# --------------------------------------------------------------------- a pass
def _precond(c):
    return sanepic_amd.PRECOND_BLOCK3 if c["precond"] == "block" else sanepic_amd.PRECOND_DIAG


def _solve(ctx, c, x0=None):
    ctx.solve_begin(_precond(c), 10, x0)
    hist = [ctx.step() for _ in range(c["iters"])]
    return ctx.map(), np.array([h["crit"] for h in hist]), np.array([h["chi2"] for h in hist])


def _single(a):
    """The mixed-precision operator's results carry single precision."""
    return np.asarray(a, dtype=np.float32)


def run(state):
    c = state["case"]
    if c["kind"] == "unet":
        y, g = state["unet"].backward(state["x"], state["dy"])
        # the network's weights, activations and gradients are BF16
        return dict(y=torch.from_numpy(y).to(torch.bfloat16), grad=torch.from_numpy(g).to(torch.bfloat16))
    if c["kind"] == "apply":
        y = state["ctx"].apply(state["x"])
        return dict(y=_single(y) if c["mixed"] else y)
    if c["kind"] == "recal":
        ctx = state["ctx"]
        ctx.set_gains(state["gains"])
        m, crit, _ = _solve(ctx, c, state["x0"])
        return dict(rhs=ctx.rhs(), map=m, crit=crit, sums=ctx.recal_sums(m))
    if c["kind"] == "map":
        data = state["data"]
        ctx = _context(c)
        _feed(ctx, c, data)
        npix, _ = ctx.pixelize()
        ctx.setup()
        hits, mp, cross = ctx.get_setup()
        m, crit, chi2 = _solve(ctx, c)
        out = dict(npix=npix, indpix=ctx.indpix(), hits=hits, mp=mp, cross=cross, rhs=ctx.rhs(), nvar=ctx.nvar(),
                   map=m, crit=crit, chi2=chi2)
        ctx.close()
        return out
    m, crit, chi2 = _solve(state["ctx"], c)
    if c["mixed"]:
        return dict(map=_single(m), crit=_single(crit))
    return dict(map=m, crit=crit, chi2=chi2)


# --------------------------------------------------------------------- the work
def work(case):
    """One operator application reads each sample's pixel (4 bytes) and
    polarisation angle (8 bytes FP64, 4 FP32) on the way in and on the way out
    and takes two real transforms of each segment (2.5 N log2 N each); a pass
    is its operator applications plus the maps and timestreams it takes."""
    c = dict(case)
    if c["kind"] == "unet":
        S2 = 12 * c["nside"] ** 2
        macs = sum(9 * ci * co / 4 ** lv for ci, co, lv in UNET) * S2
        acts = sum((ci + co) / 4 ** lv for ci, co, lv in UNET) * S2
        return dict(bytes=2.0 * 3 * acts, flops=2.0 * 3 * macs)
    lens = _lengths(c)
    tot = float(sum(L * s for L, s in lens))
    fft = sum(2 * 2.5 * L * math.log2(L) * s for L, s in lens)
    op_bytes = tot * 2 * (4 + (4 if c["mixed"] else 8))
    maps = 12 * c["nside"] ** 2 * 3 * 8.0
    if c["kind"] == "apply":
        napply = 1
    else:
        napply = c["iters"] + (c["iters"] + 9) // 10 + (1 if c["kind"] == "recal" else 0)
    b = napply * (op_bytes + 8 * maps)
    f = napply * (fft + 12 * tot)
    if c["kind"] in ("map", "recal"):
        b += 2 * (tot * 8 + op_bytes)
        f += 2 * fft
    return dict(bytes=b, flops=f)


# ------------------------------------------------------ the same in plain torch
UNET = [(16, 16, 0), (16, 16, 0), (16, 32, 1), (32, 32, 1), (32, 64, 2), (64, 64, 2), (64, 128, 3), (128, 128, 3),
        (192, 64, 2), (64, 64, 2), (96, 32, 1), (32, 32, 1), (48, 16, 0), (16, 16, 0), (16, 16, 0)]


def _unet_inputs(c, seed, nparams):
    """Weights of a trained network's size (He-normal, small biases), the
    features of a residual (M r around zero, hits and noise blocks that vary
    slowly around their mean) and an output gradient."""
    r = np.random.default_rng([seed, 6])
    parts = []
    for ci, co, _ in UNET:
        parts.append(r.standard_normal(9 * ci * co) * math.sqrt(2.0 / (9 * ci)))
        parts.append(r.standard_normal(co) * 0.01)
    p = np.concatenate(parts).astype(np.float32)
    assert p.size == nparams
    S = c["nside"]
    x = r.standard_normal((12, S, S, 10)) * 0.3
    u = np.arange(S) * (TWO_PI / S)
    wave = np.cos(u)[None, :, None, None] * np.sin(u)[None, None, :, None]
    x[..., 3:] += 0.7 + 0.3 * wave
    dy = 1.0 + 0.5 * wave + 0.2 * r.standard_normal((12, S, S, 3))
    x, dy = x.astype(np.float32), dy.astype(np.float32)
    return p, x, dy


def _unet_exact(c, seed):
    p, x, dy = _unet_inputs(c, seed, sum(9 * ci * co + co for ci, co, _ in UNET))
    p = torch.from_numpy(p).double()
    layers, o = [], 0
    for ci, co, _ in UNET:
        w = p[o:o + 9 * ci * co].reshape(co, 3, 3, ci).clone().requires_grad_(True)
        o += 9 * ci * co
        b = p[o:o + co].clone().requires_grad_(True)
        o += co
        layers.append((w, b))

    def conv(i, t, relu=True):
        w, b = layers[i]
        t = F.conv2d(t, w.permute(0, 3, 1, 2), b, padding=1)
        return torch.relu(t) if relu else t

    def up(t):
        return F.interpolate(t, scale_factor=2, mode="nearest")

    t = torch.zeros((12, c["nside"], c["nside"], 16), dtype=torch.float64)
    t[..., :10] = torch.from_numpy(x)
    t = t.permute(0, 3, 1, 2)
    e0 = conv(1, conv(0, t))
    e1 = conv(3, conv(2, F.avg_pool2d(e0, 2)))
    e2 = conv(5, conv(4, F.avg_pool2d(e1, 2)))
    t = conv(7, conv(6, F.avg_pool2d(e2, 2)))
    t = conv(9, conv(8, torch.cat([up(t), e2], 1)))
    t = conv(11, conv(10, torch.cat([up(t), e1], 1)))
    t = conv(13, conv(12, torch.cat([up(t), e0], 1)))
    y = conv(14, t, relu=False).permute(0, 2, 3, 1)[..., :3]
    (y * torch.from_numpy(dy).double()).sum().backward()
    g = torch.cat([torch.cat([w.grad.reshape(-1), b.grad]) for w, b in layers])
    return dict(y=y.detach().contiguous(), grad=g)


def _ring_pixel(nside, theta, phi):
    """HEALPix RING pixel of (theta, phi) (Gorski et al. 2005)."""
    z, tt = torch.cos(theta), phi / (0.5 * math.pi)
    za = z.abs()
    n, ncap = nside, 2 * nside * (nside - 1)
    jp, jm = torch.floor(n * (0.5 + tt - 0.75 * z)).long(), torch.floor(n * (0.5 + tt + 0.75 * z)).long()
    ir = n + 1 + jp - jm
    ip = (jp + jm - n + 1 - (ir & 1) + 1) // 2 + 1
    ip = torch.where(ip > 4 * n, ip - 4 * n, ip)
    belt = ncap + 4 * n * (ir - 1) + ip - 1
    tp, tmp = tt - torch.floor(tt), torch.sqrt(3.0 * (1.0 - za))
    jp, jm = torch.floor(n * tp * tmp).long(), torch.floor(n * (1.0 - tp) * tmp).long()
    ir = jp + jm + 1
    ip = torch.floor(tt * ir).long() + 1
    ip = torch.where(ip > 4 * ir, ip - 4 * ir, ip)
    cap = torch.where(z > 0, 2 * ir * (ir - 1) + ip - 1, 12 * n * n - 2 * ir * (ir + 1) + ip - 1)
    return torch.where(za <= 2.0 / 3.0, belt, cap)


def _lines_of_sight(c, d, ra, dec, psi):
    """Pixel, cos and sin of twice the polarisation angle, and of twice the
    angle without the half-wave plate, of one detector's samples."""
    x, y = math.radians(d["lel"]), math.radians(d["xel"])
    off, ph = math.asin(math.hypot(x, y)), math.atan2(y, x)
    tb, st, ct = 0.5 * math.pi - dec, math.sin(off), math.cos(off)
    a = ph + psi
    theta = torch.acos(torch.sin(tb) * st * torch.cos(a) + torch.cos(tb) * ct)
    dphi = torch.atan2(-st * torch.sin(a), -torch.cos(tb) * st * torch.cos(a) + torch.sin(tb) * ct)
    phi = torch.remainder(ra + dphi, TWO_PI)
    v0, v1, v2 = torch.cos(psi) * ct, torch.sin(psi) * ct, -st * math.cos(ph)
    r0, r1 = -torch.cos(tb) * v0 + torch.sin(tb) * v2, -v1
    r2 = torch.sin(tb) * v0 + torch.cos(tb) * v2
    cosang = (-torch.sin(dphi) * r0 + torch.cos(dphi) * r1) / torch.sqrt(r0 * r0 + r1 * r1 + r2 * r2)
    p = torch.acos(torch.clamp(cosang, -1.0, 1.0))
    p = torch.where(r2 < 0, -p, p)
    fp = torch.remainder(p + 2.5 * math.pi, TWO_PI) - math.pi + math.radians(d["angle"])
    t = torch.arange(ra.numel(), dtype=torch.float64, device=ra.device)
    op = -fp + 2.0 * OMEGA_HWP * t if c["hwp"] else fp
    return (_ring_pixel(c["nside"], theta, phi), torch.cos(2 * op), torch.sin(2 * op), torch.cos(2 * fp),
            torch.sin(2 * fp))


class _Plain:
    """The map-making problem in plain float64 torch."""

    def __init__(self, c, seed):
        self.c, data = c, _data(c, seed)
        self.data, self.nc = data, 4 if c["kind"] == "leak" else 3
        ra, dec, psi = (torch.from_numpy(data[k]).to(DEV) for k in ("ra", "dec", "psi"))
        self.dets, pixels = [], []
        for k, d in enumerate(data["dets"]):
            n = d["L"] * d["nseg"]
            los = _lines_of_sight(c, d, ra[:n], dec[:n], psi[:n])
            i, ispf = np.arange(d["L"] // 2 + 1, dtype=np.float64), data["ispf"][k]
            row = ispf[(i / d["L"] * d["L"]).astype(np.int64)] / float(d["L"]) / float(d["L"])
            row[0] = ispf[1] * 1e-6 / float(d["L"]) / float(d["L"])
            self.dets.append(dict(L=d["L"], nseg=d["nseg"], ring=los[0], c=los[1], s=los[2], cfp=los[3], sfp=los[4],
                                  w=torch.from_numpy(row).to(DEV), relf=float(data["relf"][k]), gain=None,
                                  tod=torch.from_numpy(data["tod"][k]).to(DEV).reshape(d["nseg"], d["L"])))
            pixels.append(torch.unique(los[0]))
        ring = torch.unique(torch.cat(pixels))
        self.npix = ring.numel()
        self.indpix = torch.full((12 * c["nside"] ** 2,), -1, dtype=torch.int64, device=DEV)
        self.indpix[ring] = torch.arange(self.npix, device=DEV)
        self.cnt = torch.zeros(self.npix, dtype=torch.int64, device=DEV)
        for d in self.dets:
            d["pix"] = self.indpix[d.pop("ring")]
            self.cnt += torch.bincount(d["pix"], minlength=self.npix)
        self.masked = self.cnt < 2

    def zeros(self, n=None):
        return torch.zeros((n or self.nc, self.npix), dtype=torch.float64, device=DEV)

    def mask(self, m):
        m = m.clone()
        m[1:3, self.masked] = 0.0
        return m

    def filtered(self, d, v):
        """N^-1 v of one detector's segments, unnormalised transforms."""
        f = torch.fft.rfft(v) * d["w"]
        return torch.fft.irfft(f, d["L"], norm="forward")

    def model(self, d, m, gains=True):
        v = m[0][d["pix"]] + m[1][d["pix"]] * d["c"] + m[2][d["pix"]] * d["s"]
        if self.nc == 4:
            v = v + m[3][d["pix"]] * d["relf"]
        v = v.reshape(d["nseg"], d["L"])
        return v * d["gain"] if gains and d["gain"] is not None else v

    def bin(self, q, d, z):
        if d["gain"] is not None:
            z = z * d["gain"]
        z = z.reshape(-1)
        q[0].index_add_(0, d["pix"], z)
        q[1].index_add_(0, d["pix"], z * d["c"])
        q[2].index_add_(0, d["pix"], z * d["s"])
        if self.nc == 4:
            q[3].index_add_(0, d["pix"], z * d["relf"])

    def apply(self, m):
        q = self.zeros()
        for d in self.dets:
            self.bin(q, d, self.filtered(d, self.model(d, m)))
        return q

    def rhs(self):
        q = self.zeros()
        for d in self.dets:
            self.bin(q, d, self.filtered(d, d["tod"]))
        return q

    def chi2(self, m):
        tot = 0.0
        for d in self.dets:
            r = torch.fft.rfft(d["tod"]) - torch.fft.rfft(self.model(d, m))
            tot = tot + 2.0 * (d["w"] * (r.real ** 2 + r.imag ** 2)).sum()
        return float(tot)

    def crosslinks(self):
        q = self.zeros(3)
        for d in self.dets:
            q[0].index_add_(0, d["pix"], d["cfp"])
            q[1].index_add_(0, d["pix"], d["sfp"])
        return q

    def pair_sums(self):
        """Diagonal blocks of A (b00 b01 b02 b11 b12 b22) and the I sum over
        pairs less than half a segment apart, per pixel: sums over the pairs
        of samples of one pixel, detector and segment."""
        out = self.zeros(7)
        for d in self.dets:
            n = d["L"]
            auto = torch.fft.irfft(d["w"].abs().to(torch.complex128), n, norm="forward")
            t = torch.arange(d["pix"].numel(), device=DEV)
            key = d["pix"] * d["nseg"] + t // n
            key, order = torch.sort(key, stable=True)
            t, c, s = (t % n)[order], d["c"][order], d["s"][order]
            u = torch.zeros((4, key.numel()), dtype=torch.float64, device=DEV)
            live, step = torch.arange(key.numel(), device=DEV), 1
            while True:
                live = live[live + step < key.numel()]
                live = live[key[live + step] == key[live]]
                if not live.numel():
                    break
                j = live + step
                dt = t[j] - t[live]
                w = auto[dt]
                u[0, live] += w
                u[1, live] += w * c[j]
                u[2, live] += w * s[j]
                u[3, live] += torch.where(dt < n // 2, w, torch.zeros_like(w))
                step += 1
            w0 = auto[0]
            terms = (w0 + 2 * u[0], w0 * c + u[1] + c * u[0], w0 * s + u[2] + s * u[0], w0 * c * c + 2 * c * u[1],
                     w0 * c * s + c * u[2] + s * u[1], w0 * s * s + 2 * s * u[2], w0 + 2 * u[3])
            for k, v in enumerate(terms):
                out[k].index_add_(0, d["pix"][order], v)
        return out

    def preconditioner(self, pairs):
        z, ok = torch.zeros_like(pairs[0]), ~self.masked
        m = [[z] * self.nc for _ in range(self.nc)]

        def inv(v, where):
            return torch.where(where & (v != 0), 1.0 / v, z)

        everywhere = torch.ones_like(ok)
        if self.c["precond"] != "block":
            m[0][0] = inv(2 * pairs[6], everywhere)
            m[1][1] = m[2][2] = inv(pairs[6], ok)
            if self.nc == 4:
                m[3][3] = inv(2 * pairs[6] * self.dets[0]["relf"] ** 2, everywhere)
            return m
        b00, b01, b02, b11, b12, b22 = pairs[:6]
        c00, c01, c02 = b11 * b22 - b12 * b12, b02 * b12 - b01 * b22, b01 * b12 - b02 * b11
        c11, c12, c22 = b00 * b22 - b02 * b02, b01 * b02 - b00 * b12, b00 * b11 - b01 * b01
        det = b00 * c00 + b01 * c01 + b02 * c02
        full = ok & (b00 > 0) & (b11 > 0) & (b22 > 0) & (det > 1e-10 * b00 * b11 * b22)
        own = {0: torch.where(b00 > 0, 1.0 / b00, z), 1: torch.where(ok & (b11 > 0), 1.0 / b11, z),
               2: torch.where(ok & (b22 > 0), 1.0 / b22, z)}
        for (i, j), v in {(0, 0): c00, (0, 1): c01, (0, 2): c02, (1, 1): c11, (1, 2): c12, (2, 2): c22}.items():
            m[i][j] = m[j][i] = torch.where(full, v / det, own[i] if i == j else z)
        return m

    def solve(self, pairs, x0=None, chi2=True):
        """The preconditioned CG iterations: map, crit and chi2 of each."""
        c, M, b = self.c, self.preconditioner(pairs), self.mask(self.rhs())
        x, q = self.zeros(), self.zeros()
        if x0 is not None:
            q, x = self.mask(self.apply(x0)), self.mask(x0)

        def step(r):
            z = torch.stack([sum(M[i][j] * r[j] for j in range(self.nc)) for i in range(self.nc)])
            return z, (r * z).sum()

        r = b - q
        d, delta = step(r)
        var00, last, crits, chis = (b * b).sum(), 0.0, [], []
        for it in range(c["iters"]):
            q = self.mask(self.apply(d))
            alpha = delta / (q * d).sum()
            x = x + alpha * d
            if it % 10 == 0:
                r = b - self.mask(self.apply(x))
                last = self.chi2(x) if chi2 else 0.0
            else:
                r = r - alpha * q
            z, new = step(r)
            d, delta = z + (new / delta) * d, new
            crits.append(float((r * r).sum() / var00))
            chis.append(last)
        return x, np.array(crits), np.array(chis)

    def fit_sums(self, m):
        out = []
        for d in self.dets:
            D, C = torch.fft.rfft(d["tod"]), torch.fft.rfft(self.model(d, m, gains=False))
            out.append(torch.stack([(d["w"] * (D * C.conj()).real).sum(1), (d["w"] * C.abs() ** 2).sum(1),
                                    (d["w"] * D.abs() ** 2).sum(1)], 1))
        return torch.stack(out)


def exact(case, seed):
    c = dict(case)
    if c["kind"] == "unet":
        return _unet_exact(c, seed)
    p = _Plain(c, seed)
    flat = lambda m: m.reshape(-1).cpu().numpy()  # noqa: E731
    if c["kind"] == "apply":
        x = torch.from_numpy(_trial_map(c, seed, 3 * p.npix)).to(DEV).reshape(3, -1)
        return dict(y=flat(p.apply(x)))
    pairs = p.pair_sums()
    if c["kind"] == "recal":
        g = torch.from_numpy(p.data["gains"]).to(DEV)
        for k, d in enumerate(p.dets):
            d["gain"] = g[k][:, None]
        x0 = torch.from_numpy(_trial_map(c, seed, 3 * p.npix)).to(DEV).reshape(3, -1)
        m, crit, _ = p.solve(pairs, x0, chi2=False)
        return dict(rhs=flat(p.rhs()), map=flat(m), crit=crit, sums=p.fit_sums(m).cpu().numpy())
    m, crit, chi2 = p.solve(pairs, chi2=not c["mixed"])
    if c["kind"] == "map":
        diag = torch.stack([2 * pairs[6], pairs[6], pairs[6]])
        nv = p.mask(1.0 / diag)
        hits = (2 * p.cnt).repeat(2).cpu().numpy()
        return dict(npix=p.npix, indpix=p.indpix.cpu().numpy(), hits=hits, mp=flat(diag), cross=flat(p.crosslinks()),
                    rhs=flat(p.rhs()), nvar=flat(nv), map=flat(m), crit=crit, chi2=chi2)
    if c["mixed"]:
        return dict(map=flat(m), crit=crit)
    return dict(map=flat(m), crit=crit, chi2=chi2)
