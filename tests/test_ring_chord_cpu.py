"""What the kernels' ring chord rests on: a pixel's points lie between the
centre latitudes of the neighbouring rings, at longitudes whose pixel is
floor(tt npr / 4) or the next one; and the chord bound holds every pair within
the radius (evaluated here in double precision, without the kernels' margins)."""
import numpy as np
import pytest

import oracle


@pytest.mark.parametrize("nside", [4, 64, 1024, 8192])
def test_band_and_position(nside):
    h = oracle.hpx(nside)
    rng = np.random.default_rng(nside)
    n = 200000
    z = np.concatenate([rng.uniform(-1, 1, n), np.sign(rng.uniform(-1, 1, n)) * (2 / 3 + rng.normal(0, 2 / nside, n))])
    z = np.clip(z, -0.9999, 0.9999)
    phi = rng.uniform(0, 2 * np.pi, z.size)
    theta = np.arccos(z)
    pix = oracle.ang2pix(h, theta, phi)
    ring = oracle.pix2ring(h, pix).astype(np.int64)
    keep = (ring > 1) & (ring < 4 * nside - 1)
    theta, phi, pix, ring = theta[keep], phi[keep], pix[keep].astype(np.int64), ring[keep]

    def ring_theta(r):
        sp, _ = oracle.ring_info(h, r)
        return oracle.pix2ang(h, sp)[0]

    up, dn = ring_theta((ring - 1).astype(np.uint64)), ring_theta((ring + 1).astype(np.uint64))
    assert np.all(theta >= up - 1e-12) and np.all(theta <= dn + 1e-12)
    sp, npr = oracle.ring_info(h, ring.astype(np.uint64))
    p, npr = pix - sp.astype(np.int64), npr.astype(np.int64)
    f = np.floor(phi / (np.pi / 2) * npr / 4).astype(np.int64)
    edge = np.abs(phi / (np.pi / 2) * npr / 4 - np.round(phi / (np.pi / 2) * npr / 4)) < 1e-9
    assert np.all((p == f) | (p == (f + 1) % npr) | edge)


@pytest.mark.parametrize("radius", [0.03, 0.3, 3.0])
def test_bound_holds_every_pair(radius):
    rng = np.random.default_rng(3)
    n = 400000
    bc = np.radians(rng.uniform(-86, 86, n))
    R = np.radians(radius)
    bs = np.clip(bc + rng.uniform(-1, 1, n) * R, -1.55, 1.55)
    dl = rng.uniform(0, 1, n) * np.minimum(3 * R / np.cos(bs), 3.0)
    hav = np.sin((bs - bc) / 2) ** 2 + np.cos(bs) * np.cos(bc) * np.sin(dl / 2) ** 2
    inside = hav < np.sin(R / 2) ** 2
    # the band and the cells reduced to single latitudes: dz their gap
    dz = np.abs(np.sin(bs) - np.sin(bc))
    straddle = np.sign(bs) != np.sign(bc)
    cmax = np.where(straddle, 1.0, np.maximum(np.cos(bs), np.cos(bc)))
    num = np.sin(R / 2) ** 2 - (dz / (2 * cmax)) ** 2
    s2 = num / (np.cos(bs) * np.cos(bc))
    lim = np.where(s2 < 0.25, 2 * np.sqrt(np.maximum(s2, 0) / (1 - np.minimum(s2, 0.25))), np.inf)
    assert inside.sum() > 50000
    assert np.all(num[inside] > 0)
    assert np.all(dl[inside] <= lim[inside] * (1 + 1e-12))
