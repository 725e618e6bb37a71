"""The belt-ring form of the compat window against the pixels themselves.

In a belt ring (nside < r < 3 nside) the kernels take a window from tl to tr
(longitudes in units of pi/2) as the samples with hl <= g <= hr + 1, h =
floor(2 nside t), g = 2 p + 1 - (r odd) for pixel p of the ring, instead of
evaluating the pixels lpix and rpix of its two edges in every ring.  Here both
are evaluated on the host, lpix and rpix by hcg_host_ang2pix at the ring's
centre (the reference's own formulas, HCGrid/healpix.cu:126-224), for every
pixel near the edges, except where the kernels do the same: an edge within
1e-6 half pixels of a boundary, or a window that meets longitude 0.
"""
import ctypes as C
import math

import numpy as np
import pytest

from hcgrid_amd import capi


@pytest.mark.parametrize("nside", [2, 4, 64, 1024, 4096, 8192])
def test_belt_window_selects_the_same_pixels(nside):
    lib = capi.load()
    hp = capi.Healpix()
    capi.call("hcg_healpix_init", nside, C.byref(hp))
    rng = np.random.default_rng(nside)
    checked = 0
    for _ in range(4000):
        ring = int(rng.integers(nside + 1, 3 * nside))
        tl = float(rng.uniform(0.0, 4.0))
        tr = tl + float(rng.uniform(0.0, 12.0 / nside))
        if rng.integers(4) == 0:  # on and next to pixel boundaries too
            tl = (math.floor(2 * nside * tl) + float(rng.choice([1e-5, 0.5, 1 - 1e-5]))) / (2 * nside)
        xl, xr = 2.0 * nside * tl, 2.0 * nside * tr
        near = any(abs(x - round(x)) <= 1e-6 for x in (xl, xr))
        if near or not xl < xr < 8.0 * nside - 2.0:
            continue  # the kernels evaluate these windows ring by ring
        sp, npr = C.c_uint64(), C.c_uint64()
        lib.hcg_host_ring_info(C.byref(hp), ring, C.byref(sp), C.byref(npr))
        th = lib.hcg_host_pix2theta(C.byref(hp), sp.value)
        lpix = lib.hcg_host_ang2pix(C.byref(hp), th, tl * math.pi / 2) - sp.value
        rpix = lib.hcg_host_ang2pix(C.byref(hp), th, tr * math.pi / 2) - sp.value
        assert 0 <= lpix < npr.value and 0 <= rpix < npr.value
        hl, hr = math.floor(xl), math.floor(xr)
        for p in {q for e in (lpix, rpix) for q in range(e - 3, e + 4) if 0 <= q < npr.value}:
            g = 2 * p + 1 - (ring & 1)
            assert (hl <= g <= hr + 1) == (lpix <= p <= rpix), (nside, ring, tl, tr, p, lpix, rpix)
            checked += 1
    assert checked > 1000
