"""GAUSS2D and TAPERED_SINC weights near the largest radius of the tangent-frame
and series forms, cell by cell against extended precision: one sample per cell,
so that a cell's weight sum is one weight.

Tolerance: a unit vector's components are good to 1.2e-16 and |p - q|^2 to
8e-16 / |p - q| relative (4e-14 at 1.1 deg); an exponent of up to 7 carries
seven times that, 3e-13, and 1e-12 is allowed."""
import numpy as np
import pytest

from hcgrid_amd import GAUSS2D, TAPERED_SINC, gridder

pytestmark = pytest.mark.gpu

L = np.longdouble


def _weights(kt, params, lon_c, lat_c, lon_s, lat_s):
    d2r = L(np.pi) / L(180)  # the framework's PI is the double one
    l1, b1, l2, b2 = (L(v) * d2r for v in (lon_c, lat_c, lon_s, lat_s))
    h = np.sin((b1 - b2) / 2) ** 2 + np.cos(b1) * np.cos(b2) * np.sin((l1 - l2) / 2) ** 2
    dist = 2 * np.arcsin(np.sqrt(h)) / d2r
    if kt == GAUSS2D:
        dl = l2 - l1
        bear = np.arctan2(np.cos(b2) * np.sin(dl), np.cos(b1) * np.sin(b2) - np.sin(b1) * np.cos(b2) * np.cos(dl))
        p0, p1, pa = (L(p) for p in params)
        ell = (p0 * np.sin(bear - pa)) ** 2 + (p1 * np.cos(bear - pa)) ** 2
        return dist, np.exp(-((dist / p0 / p1) ** 2) / 2 * ell)
    a = L(np.pi) * dist / L(params[0])
    x = a / L(params[2])
    return dist, np.sin(x) / x * np.exp((a / L(params[1])) ** 2)


@pytest.mark.parametrize("kt,params", [(GAUSS2D, [0.3, 0.35, 0.7]), (GAUSS2D, [0.45, 0.3, -1.2]),
                                       (TAPERED_SINC, [1.0, 3.0, 1.2])])
@pytest.mark.parametrize("dec", [3.0, -47.0])
def test_weight_near_the_largest_radius(gpu, kt, params, dec):
    side, radius = 24, 1.1
    rng = np.random.default_rng(8)
    # cells 3 deg apart, one sample near each
    rows, cols = np.divmod(np.arange(side * side), side)
    lat_c = dec + (rows - side / 2) * 3.0
    lat_c = np.clip(lat_c, -84.0, 84.0) + rng.uniform(-0.1, 0.1, side * side)
    lon_c = 180.0 + (cols - side / 2) * 3.0 / np.cos(np.radians(lat_c))
    keep = np.abs(lon_c - 180.0) < 170.0
    lon_c = np.where(keep, lon_c, 180.0)
    r, az = np.radians(rng.uniform(0.9, 1.09, side * side)), rng.uniform(0, 2 * np.pi, side * side)
    b = np.radians(lat_c)
    lat_s = np.degrees(np.arcsin(np.sin(b) * np.cos(r) + np.cos(b) * np.sin(r) * np.cos(az)))
    lon_s = lon_c + np.degrees(np.arctan2(np.sin(az) * np.sin(r) * np.cos(b),
                                          np.cos(r) - np.sin(b) * np.sin(np.radians(lat_s))))
    idx = np.flatnonzero(keep)
    print(f"case: kt={kt} params={params} dec={dec}", flush=True)
    dev = gridder.grid_plain(lon_s[idx], lat_s[idx], np.ones(idx.size), lon_c, lat_c, side, 0.0, radius, 0.2,
                             kernel_type=kt, kernel_params=params, selection="disc")
    # cells that meet exactly one sample
    d2r = np.pi / 180
    cosd = (np.sin(b)[:, None] * np.sin(lat_s[idx] * d2r)[None, :] + np.cos(b)[:, None] *
            np.cos(lat_s[idx] * d2r)[None, :] * np.cos((lon_c[:, None] - lon_s[idx][None, :]) * d2r))
    near = np.degrees(np.arccos(np.clip(cosd, -1, 1))) < radius + 0.01
    one = np.flatnonzero(near.sum(1) == 1)
    s = idx[np.argmax(near[one], axis=1)]
    dist, want = _weights(kt, params, lon_c[one], lat_c[one], lon_s[s], lat_s[s])
    sel = (dist < radius - 1e-6) & (np.abs(want) > 1e-3)
    got = dev["weightscube"][one][sel]
    rel = np.abs(got.astype(L) - want[sel]) / np.abs(want[sel])
    print(f"  {sel.sum()} weights, largest error {float(rel.max()):.2e}", flush=True)
    assert sel.sum() > 100
    assert rel.max() <= 1e-12
