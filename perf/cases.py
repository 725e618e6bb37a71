"""Timing cases of the gridding path: what a user's program has it do, through
the public Python entry points, from the smallest maps to the largest cube.

Every case grids a raster scan (constant-Dec lines, samples evenly spaced in
RA with a uniform jitter) that covers a square SIN map of 0.01 degree cells,
with inputs resident on the GPU.  Four kinds of call:

  plain    PlainGridder.run: the single-channel FP64 path, from coordinates
           and values to the normalised map (pre-sort, records, ring table,
           gridding, normalisation);
  cube     CubeGridder.run: the same for a spectral cube of 16-bit channels;
  batch    Batch.enqueue on resident geometries: several uneven cubes in one
           launch, new channel values on known coordinates;
  request  what a served request with new coordinates costs on the device: a
           Geometry built in the caching allocator's memory and a one-job
           Batch on it.
"""
from __future__ import annotations

import math
import random

import torch

from hcgrid_amd import batch as hbatch
from hcgrid_amd import capi, gridder, synth

CDELT = 0.01  # degrees per cell
RA0 = 180.0
D2R = math.pi / 180.0
KERNELS = {"gauss1d": capi.GAUSS1D, "gauss2d": capi.GAUSS2D, "tapered_sinc": capi.TAPERED_SINC}


def _plain(name, lines, per_line, side, dec=30.0, sigma=0.02, nsigma=3.0, kernel="gauss1d", select="compat",
           values="f32", weights=False, factor=1):
    return dict(name=name, path="plain", lines=lines, per_line=per_line, side=side, dec=dec, sigma=sigma,
                nsigma=nsigma, kernel=kernel, select=select, values=values, weights=weights, factor=factor)


def _cube(name, lines, per_line, side, nchan, dtype="bf16", layout=0, dec=30.0, sigma=0.02, select="compat",
          path="cube"):
    return dict(name=name, path=path, lines=lines, per_line=per_line, side=side, nchan=nchan, dtype=dtype,
                layout=layout, dec=dec, sigma=sigma, nsigma=3.0, kernel="gauss1d", select=select, factor=1)


def listed():
    return [
        # a quick look at a pointing: a few thousand samples, all latency
        _plain("plain_small", 30, 150, 20),
        # one observing session's map (200 lines x 1250 samples onto 400^2)
        _plain("plain_250k", 200, 1250, 400),
        # a survey field (1000 lines x 20000 samples onto 2048^2)
        _plain("plain_20m", 1000, 20000, 2048),
        # the command line's default: a 300 arcsec beam gridded out to 5 sigma, FP64 values, here with
        # per-sample weights and sizes that divide by nothing
        _plain("plain_beam300", 501, 1499, 347, dec=-33.0, sigma=0.0353892, nsigma=5.0, values="f64", weights=True),
        # an elliptical beam
        _plain("plain_gauss2d", 300, 900, 300, dec=12.0, kernel="gauss2d"),
        # a high-declination field with the complete disc of every cell
        _plain("plain_disc_polar", 400, 1500, 333, dec=80.0, select="disc", values="f64"),
        # the reference's 500^2 HDF5 target with three spectral channels
        _cube("cube_3ch", 260, 750, 500, 3, dtype="f16"),
        # a backend that writes spectra sample by sample, odd channel count and side
        _cube("cube_67_samples", 401, 1203, 511, 67, dtype="f16", layout=1, dec=-20.0),
        # few channels on a sparsely sampled large map
        _cube("cube_sparse_16", 548, 548, 2048, 16, dec=45.0),
        # a full spectral cube (2M samples x 1024 channels onto 1024^2)
        _cube("cube_2m_1024", 500, 4000, 1024, 1024),
        # six uneven jobs on resident geometries
        dict(name="batch_6", path="batch", mix=11, njobs=6),
        # a served request on coordinates not seen before
        _cube("request_1m2", 1000, 1200, 512, 64, dec=-40.0, sigma=0.03, path="request"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_raster(rng, nmin, nmax, side):
    """Lines and samples per line of about a log-uniform count, at most 40 samples per cell."""
    n = _log_int(rng, nmin, max(nmin, min(nmax, 40 * side * side)))
    lines = max(2, int(round(math.sqrt(n) * math.exp(rng.uniform(-0.9, 0.2)))))
    return lines, max(2, n // lines)


def _field_dec(rng, side, lo, hi):
    half = side * CDELT / 2.0
    return round(max(-86.0 + half, min(86.0 - half, rng.uniform(lo, hi))), 3)


def draw(rng: random.Random):
    path = rng.choice(["plain"] * 6 + ["cube"] * 4 + ["batch", "request"])
    if path == "batch":
        return dict(path="batch", mix=rng.randrange(1 << 20), njobs=rng.randint(2, 8))
    select = rng.choice(["compat", "compat", "compat", "disc"])
    sigma = rng.choice([0.015, 0.02, 0.03])
    if path == "plain":
        kernel = rng.choice(["gauss1d"] * 5 + ["gauss2d", "tapered_sinc"])
        side = _log_int(rng, 16, 2048 if kernel == "gauss1d" else 600)
        lines, per_line = _draw_raster(rng, 2e3, 2e7 if kernel == "gauss1d" else 1e6, side)
        wide = kernel == "gauss1d" and rng.random() < 0.2 and lines * per_line < 2e6
        c = _plain("", lines, per_line, side, dec=_field_dec(rng, side, -60.0, 85.0),
                   sigma=0.0353892 if wide else sigma, nsigma=5.0 if wide else 3.0, kernel=kernel, select=select,
                   values=rng.choice(["f32", "f64"]), weights=rng.random() < 0.25,
                   factor=rng.choice([1, 1, 1, 2]))
    else:
        side = _log_int(rng, 64, 2048 if path == "cube" else 512)
        nmax = 3e6 if path == "cube" else 1.2e6
        lines, per_line = _draw_raster(rng, 5e4, nmax, side)
        nchan = _log_int(rng, 1, 1024)
        n = lines * per_line
        # samples x channels, and cells x channels, no more than the full cube's
        nchan = max(1, min(nchan, int(1e9 // n), int(5e8 // (side * side))))
        c = _cube("", lines, per_line, side, nchan, dtype=rng.choice(["bf16", "f16"]),
                  layout=rng.randrange(2) if path == "cube" else 0, dec=_field_dec(rng, side, -60.0, 75.0),
                  sigma=sigma, select=select, path=path)
    del c["name"]
    return c


# ---- inputs --------------------------------------------------------------------------------


def _jobs(case):
    """The cube jobs of a batch case: uneven sizes drawn from its mix number."""
    rng = random.Random(case["mix"])
    out = []
    for _ in range(case["njobs"]):
        side = rng.choice([128, 256, 512, 1024])
        lines, per_line = _draw_raster(rng, 5e4, 1.5e6, side)
        nchan = rng.choice([1, 16, 64, 256, 512])
        nchan = max(1, min(nchan, int(1.5e8 // (lines * per_line)), int(1e8 // (side * side))))
        c = _cube("", lines, per_line, side, nchan, dtype=rng.choice(["bf16", "f16"]),
                  dec=_field_dec(rng, side, -60.0, 80.0), sigma=rng.choice([0.015, 0.02, 0.03]))
        out.append(c)
    return out


def _generator(seed, k=0):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + 7919 * k) % (1 << 62))
    return g


def _geometry(case):
    """First line, line spacing, first RA and RA spacing (degrees) of a case's raster over its map's field."""
    field = case["side"] * CDELT
    ddec = field / case["lines"]
    dra = field / case["per_line"] / math.cos(case["dec"] * D2R)
    return (case["dec"] - field / 2.0 + 0.5 * ddec, ddec, RA0 - dra * case["per_line"] / 2.0 + 0.5 * dra, dra)


def _coords(case, gen):
    lat0, ddec, lon0, dra = _geometry(case)
    lines, per = case["lines"], case["per_line"]
    k = torch.arange(lines, dtype=torch.float64, device="cuda")
    j = torch.arange(per, dtype=torch.float64, device="cuda")
    jit = torch.rand(lines * per, generator=gen, dtype=torch.float64, device="cuda") * 2.0 - 1.0
    lon = (lon0 + dra * j).repeat(lines) + jit * (dra / 6.4)
    lat = (lat0 + ddec * k).repeat_interleave(per)
    return lon, lat


def _target(case):
    """Cell coordinates (degrees) of the SIN map centred on the field."""
    side = case["side"]
    p = (torch.arange(1, side + 1, dtype=torch.float64, device="cuda") - side / 2.0) * (CDELT * D2R)
    x, y = -p[None, :], p[:, None]
    d0 = case["dec"] * D2R
    z = torch.sqrt(1.0 - x * x - y * y)
    lat = torch.asin(z * math.sin(d0) + y * math.cos(d0))
    lon = RA0 + torch.atan2(x.expand(side, side), z * math.cos(d0) - y * math.sin(d0)) / D2R
    return lon.reshape(-1).contiguous(), (lat / D2R).reshape(-1).contiguous()


def _sources(case, lon, lat, gen):
    """Three Gaussian sources' summed brightness at every sample."""
    half = 0.4 * case["side"] * CDELT
    r = torch.rand(3, 3, generator=gen, dtype=torch.float64, device="cuda").tolist()
    out = torch.zeros_like(lon)
    for a, u, v in r:
        dx = (lon - RA0) * math.cos(case["dec"] * D2R) - half * (2 * u - 1)
        dy = lat - case["dec"] - half * (2 * v - 1)
        out += (1 + 9 * a) * torch.exp(-(dx * dx + dy * dy) / (2 * 0.05 ** 2))
    return out


def _plain_inputs(case, seed):
    gen = _generator(seed)
    lon, lat = _coords(case, gen)
    v = torch.randn(lon.numel(), generator=gen, dtype=torch.float64, device="cuda") + _sources(case, lon, lat, gen)
    w = torch.rand(lon.numel(), generator=gen, dtype=torch.float64, device="cuda") + 0.5 if case["weights"] else None
    return lon, lat, (v if case["values"] == "f64" else v.float()), w


def _cube_inputs(case, seed, k=0):
    gen = _generator(seed, k)
    lon, lat = _coords(case, gen)
    n, c = lon.numel(), case["nchan"]
    src = _sources(case, lon, lat, gen).float()
    line = torch.exp(-((torch.arange(c, device="cuda") - 0.5 * c) / (0.1 * c + 1.0)) ** 2)
    dt = torch.bfloat16 if case["dtype"] == "bf16" else torch.float16
    vals = torch.empty((c, n), dtype=dt, device="cuda")
    step = max(1, (1 << 26) // n)
    for c0 in range(0, c, step):
        c1 = min(c, c0 + step)
        vals[c0:c1] = 0.5 * torch.randn((c1 - c0, n), generator=gen, device="cuda") + line[c0:c1, None] * src
    return lon, lat, (vals.t().contiguous() if case["layout"] else vals)


def _kernel(case):
    """Kernel type, its parameters and the radius (degrees)."""
    s = case["sigma"]
    params = {"gauss1d": [s], "gauss2d": [s, 0.75 * s, 0.3], "tapered_sinc": [s, 1.55, 2.52]}[case["kernel"]]
    return KERNELS[case["kernel"]], params, case["nsigma"] * s


def prepare(case, seed):
    if case["path"] == "batch":
        jobs, keep = [], []
        for k, job in enumerate(_jobs(case)):
            lon, lat, vals = _cube_inputs(job, seed, k)
            kt, params, radius = _kernel(job)
            kern, hp = gridder.prepare_grid_kernel(kt, params, radius, job["sigma"] / 2, 1, job["select"])
            g = hbatch.Geometry(kern, hp, lon.numel(), job["side"], in_torch=True)
            g.build(lon, lat, *_target(job))
            m = job["side"] ** 2
            jobs.append(dict(geometry=g, values=vals, dtype=job["dtype"],
                             cube=torch.empty((job["nchan"], m), dtype=torch.float32, device="cuda"),
                             wsum=torch.empty(m, dtype=torch.float32, device="cuda")))
            keep.append((lon, lat))
        return dict(case=case, jobs=jobs, keep=keep, batch=hbatch.Batch(jobs, stream=torch.cuda.current_stream()))
    kt, params, radius = _kernel(case)
    kern, hp = gridder.prepare_grid_kernel(kt, params, radius, case["sigma"] / 2, case["factor"], case["select"])
    if case["path"] == "plain":
        lon, lat, v, w = _plain_inputs(case, seed)
        g = gridder.PlainGridder(lon.numel(), case["side"], kern, hp, with_weights=w is not None)
        return dict(case=case, grid=g, inputs=(lon, lat, v) + _target(case), weights=w)
    lon, lat, vals = _cube_inputs(case, seed)
    if case["path"] == "request":
        tgt = synth.Target(case["side"], CDELT, RA0, case["dec"], case["side"] / 2.0)
        return dict(case=case, kern=kern, hp=hp, lon=lon, lat=lat, vals=vals, target=tgt, held=[])
    g = gridder.CubeGridder(lon.numel(), case["side"], case["nchan"], kern, hp, dtype=case["dtype"])
    return dict(case=case, grid=g, inputs=(lon, lat, vals) + _target(case))


def run(state):
    case = state["case"]
    if case["path"] == "plain":
        g = state["grid"]
        g.run(*state["inputs"], weights=state["weights"])
        b = g.buf
        return dict(map=b.map, datacube=b.datacube, weightscube=b.weightscube, keys=b.keys, perm=b.perm)
    if case["path"] == "cube":
        g = state["grid"]
        g.run(*state["inputs"], layout=case["layout"])
        return dict(cube=g.cube, wsum=g.wsum)
    if case["path"] == "batch":
        state["batch"].enqueue()
        return [dict(cube=j["cube"], wsum=j["wsum"]) for j in state["jobs"]]
    # request: everything is made anew, as for coordinates that no earlier request had; what earlier passes
    # made is dropped once the GPU is done with it
    held = state["held"]
    while held and held[0][0].query():
        held.pop(0)
    s = torch.cuda.current_stream()
    m = case["side"] ** 2
    g = hbatch.Geometry(state["kern"], state["hp"], state["lon"].numel(), case["side"], in_torch=True)
    g.set_target(state["target"])
    g.build(state["lon"], state["lat"])
    job = dict(geometry=g, values=state["vals"], dtype=case["dtype"],
               cube=torch.empty((case["nchan"], m), dtype=torch.float32, device="cuda"),
               wsum=torch.empty(m, dtype=torch.float32, device="cuda"))
    b = hbatch.Batch([job], stream=s)
    b.enqueue()
    done = torch.cuda.Event()
    done.record(s)
    held.append((done, b, g))
    return dict(cube=job["cube"], wsum=job["wsum"])


# ---- the work of one pass --------------------------------------------------------------------


def _pairs(case):
    """(cell, sample) pairs within the radius: every sample meets pi R^2 / cell area cells."""
    r = _kernel(case)[2] / CDELT
    return case["lines"] * case["per_line"] * math.pi * min(r * r, case["side"] ** 2 / math.pi)


def work(case):
    if case["path"] == "batch":
        # known coordinates: sorted positions, permutation and values in, cubes out
        b = f = 0.0
        for j in _jobs(case):
            n, m, c = j["lines"] * j["per_line"], j["side"] ** 2, j["nchan"]
            b += n * (2.0 * c + 28.0) + m * (16.0 + 4.0 + 4.0 * c)
            f += _pairs(j) * (2.0 * c + 20.0)
        return {"bytes": b, "flops": f}
    n, m, pairs = case["lines"] * case["per_line"], case["side"] ** 2, _pairs(case)
    if case["path"] == "plain":
        size = 8.0 if case["values"] == "f64" else 4.0
        # coordinates, values and weights in; keys, permutation, two sums and the map out
        return {"bytes": n * (16.0 + size + (8.0 if case["weights"] else 0.0) + 8.0) + m * (16.0 + 24.0),
                "flops": pairs * 20.0}
    c = case["nchan"]
    return {"bytes": n * (16.0 + 2.0 * c) + m * (16.0 + 4.0 + 4.0 * c), "flops": pairs * (2.0 * c + 20.0)}


# ---- 64-bit results in plain torch -------------------------------------------------------------


def _ring_start(ns, r):
    """First pixel and length of HEALPix ring r (RING ordering)."""
    npix, ncap = 12 * ns * ns, 2 * ns * (ns - 1)
    q = 4 * ns - r
    start = torch.where(r < ns, 2 * r * (r - 1), torch.where(r < 3 * ns, ncap + (r - ns) * 4 * ns,
                                                             npix - 2 * q * (q + 1)))
    return start, torch.where(r < ns, 4 * r, torch.where(r < 3 * ns, torch.full_like(r, 4 * ns), 4 * q))


def _ring_pix(ns, z, phi):
    """HEALPix ring and RING pixel of (cos theta, phi), |z| < 0.99997."""
    za = z.abs()
    tt = torch.remainder(phi * (2.0 / math.pi), 4.0)
    t1, t2 = ns * (0.5 + tt), ns * z * 0.75
    jp, jm = (t1 - t2).to(torch.int64), (t1 + t2).to(torch.int64)
    ir = ns + 1 + jp - jm
    ip = ((jp + jm + (1 - (ir & 1)) + 1 + 7 * ns) >> 1) & (4 * ns - 1)
    tp = tt - torch.floor(tt)
    s = ns * torch.sqrt(3.0 * (1.0 - za))
    irc = (tp * s).to(torch.int64) + ((1.0 - tp) * s).to(torch.int64) + 1
    ipc = (tt * irc).to(torch.int64)
    ring = torch.where(za <= 2.0 / 3.0, ns - 1 + ir, torch.where(z > 0, irc, 4 * ns - irc))
    return ring, _ring_start(ns, ring)[0] + torch.where(za <= 2.0 / 3.0, ip, ipc)


def _ring_z(ns, r):
    """cos of ring r's centre colatitude, by way of the angle."""
    n, q = r.double(), (4 * ns - r).double()
    cap = 4.0 / (12 * ns * ns)
    z = torch.where(r < ns, 1.0 - n * n * cap, torch.where(r < 3 * ns, (2.0 * ns - n) * (2 * ns * cap), q * q * cap - 1.0))
    return torch.cos(torch.acos(z))


def _pair_terms(case, lon, lat, xw, yw):
    """Yields (sample index, weight) for every cell at once, sample offset by sample offset: the kernel's weight
    where the pair is selected, 0 elsewhere.  The raster's layout gives the samples that can lie within a cell's
    radius; the selection is great-circle distance < R, and with the compat selection also the reference's windows
    (ring range and per-ring pixel range around the window anchor, first used ring left out)."""
    lat0, ddec, lon0, dra = _geometry(case)
    lines, per, side = case["lines"], case["per_line"], case["side"]
    kt, params, radius = _kernel(case)
    rr = radius * D2R
    b1, l1 = yw * D2R, xw * D2R
    half = torch.asin((math.sin(rr) / torch.cos(b1)).clamp(max=1.0)) / D2R  # longitude reach of the disc
    k0 = torch.ceil((yw - radius - lat0) / ddec - 1e-6).to(torch.int64)
    j0 = torch.ceil((xw - half - lon0) / dra - 0.2).to(torch.int64)
    nk = int(math.floor(2 * radius / ddec)) + 2
    nj = int(float((2 * half / dra).max())) + 3
    compat = case["select"] == "compat"
    if compat:
        ns = 1
        while ns <= math.sqrt(math.pi / 3) / (case["sigma"] / 2 * D2R) + 0.5:
            ns *= 2
        disc = rr + math.sqrt(4.0 * math.pi / (12 * ns * ns))
        ring_s, key_s = _ring_pix(ns, torch.cos(math.pi / 2 - lat * D2R), lon * D2R)
        first, last = int(ring_s.min()), int(ring_s.max())
        cell = torch.arange(side * side, device="cuda")
        f = 1 if "factor" not in case else case["factor"]
        anchor = cell - cell % side + (cell % side) // f * f
        ta, pa = math.pi / 2 - b1[anchor], l1[anchor]
        ur = _ring_pix(ns, torch.cos((ta - disc).clamp(min=0.0)), pa)[0].clamp(min=first)
        dr = _ring_pix(ns, torch.cos(ta + disc), pa)[0].clamp(max=last)
        whole = (ta / D2R <= 20) | (ta / D2R >= 160)
    cb1 = torch.cos(b1)
    sb1 = torch.sin(b1)
    for a in range(nk):
        k = k0 + a
        okk = (k >= 0) & (k < lines)
        if not bool(okk.any()):
            continue
        for c in range(nj):
            j = j0 + c
            i = k.clamp(0, lines - 1) * per + j.clamp(0, per - 1)
            b2, l2 = lat[i] * D2R, lon[i] * D2R
            hav = torch.sin((b1 - b2) / 2) ** 2 + cb1 * torch.cos(b2) * torch.sin((l1 - l2) / 2) ** 2
            d = 2 * torch.asin(torch.sqrt(hav)) / D2R
            ok = okk & (j >= 0) & (j < per) & (d < radius)
            if compat:
                r = ring_s[i]
                z = _ring_z(ns, r)
                rl, pl = _ring_pix(ns, z, pa - disc)
                rh, ph = _ring_pix(ns, z, pa + disc)
                key = key_s[i]
                ok &= (r >= ur) & (r <= dr) & (r != first)
                ok &= whole | ((rl == r) & (rh == r) & (key >= pl) & (key <= ph))
            if kt == capi.GAUSS1D:
                w = torch.exp(-0.5 / params[0] ** 2 * d * d)
            elif kt == capi.GAUSS2D:
                dl, cb2 = l2 - l1, torch.cos(b2)
                bear = torch.atan2(cb2 * torch.sin(dl), cb1 * torch.sin(b2) - sb1 * cb2 * torch.cos(dl)) - params[2]
                ell = params[0] ** 2 * torch.sin(bear) ** 2 + params[1] ** 2 * torch.cos(bear) ** 2
                w = torch.exp(-((d / params[0] / params[1]) ** 2 / 2 * ell))
            else:
                arg = math.pi * d / params[0]
                w = torch.sinc(arg / params[2] / math.pi) * torch.exp((arg / params[1]) ** 2)
            yield i, torch.where(ok, w, torch.zeros_like(w))


def _exact_cube(case, lon, lat, vals, xw, yw):
    c, m = case["nchan"], case["side"] ** 2
    acc = torch.zeros((c, m), dtype=torch.float64, device="cuda")
    wsum = torch.zeros(m, dtype=torch.float64, device="cuda")
    v = vals.t() if case["layout"] else vals
    step = max(1, (1 << 28) // m)
    for i, w in _pair_terms(case, lon, lat, xw, yw):
        wsum += w
        for c0 in range(0, c, step):
            acc[c0:c0 + step].addcmul_(v[c0:c0 + step].index_select(1, i).double(), w[None, :])
    acc /= wsum
    return dict(cube=acc, wsum=wsum)


def exact(case, seed):
    if case["path"] == "batch":
        jobs = _jobs(case)
        if sum(_cost(j) for j in jobs) > 4e11:
            return None
        return [_exact_cube(j, *_cube_inputs(j, seed, k), *_target(j)) for k, j in enumerate(jobs)]
    if case["path"] == "plain":
        lon, lat, v, weights = _plain_inputs(case, seed)
        v = v.double()
        xw, yw = _target(case)
        data, wsum = torch.zeros_like(xw), torch.zeros_like(xw)
        for i, w in _pair_terms(case, lon, lat, xw, yw):
            if weights is not None:
                w = w * weights[i]
            data += v[i] * w
            wsum += w
        return dict(map=data / wsum, datacube=data, weightscube=wsum, keys=None, perm=None)
    if _cost(case) > 4e11:
        return None
    lon, lat, vals = _cube_inputs(case, seed)
    return _exact_cube(case, lon, lat, vals, *_target(case))


def _cost(case):
    """Sample offsets x cells x channels that the 64-bit sums of a cube visit."""
    r = _kernel(case)[2]
    _, ddec, _, dra = _geometry(case)
    return (2 * r / ddec + 2) * (2 * r / (dra * math.cos(case["dec"] * D2R)) + 3) * case["side"] ** 2 * case["nchan"]
