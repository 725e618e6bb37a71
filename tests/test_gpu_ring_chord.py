"""The chord that narrows rings and windows, against the oracle where it could
cut too much: fields over the equator, at the caps' edge, next to the poles and
to longitude 0, anchors of factors 2 and 3, wide radii, scattered samples."""
import numpy as np
import pytest

from hcgrid_amd import gridder, synth

from test_gpu_cube import _run_case
from helpers import map_errors, normalise
from test_gpu_plain import _compare, _target_coords

pytestmark = pytest.mark.gpu


def _scattered(side, dec, ra, cdelt, n, seed):
    """Uniform samples over a little more than the field, unordered."""
    t = synth.Target(side, cdelt, ra, dec, side / 2.0)
    xw, yw = _target_coords(t)
    rng = np.random.default_rng(seed)
    half = 0.55 * side * cdelt
    lat = rng.uniform(max(dec - half, -89.9), min(dec + half, 89.9), n)
    wide = min(half / max(np.cos(np.radians(min(abs(dec) + half, 89.0))), 0.02), 179.0)
    lon = np.mod(ra + rng.uniform(-wide, wide, n), 360.0)
    return lon, lat, rng.normal(size=n).astype(np.float32), xw, yw


@pytest.mark.parametrize("dec,ra,cdelt,sigma,factor", [
    (0.0, 180.0, 0.01, 0.02, 1), (0.003, 90.0, 0.01, 0.02, 3), (41.81, 200.0, 0.01, 0.02, 2),
    (-41.81, 10.0, 0.01, 0.02, 1), (-84.0, 45.0, 0.01, 0.02, 1), (30.0, 0.02, 0.01, 0.02, 1),
    (0.1, 120.0, 0.2, 0.4, 1), (55.0, 250.0, 0.3, 1.0, 1),
])
def test_compat(gpu, dec, ra, cdelt, sigma, factor):
    lon, lat, v, xw, yw = _scattered(41, dec, ra, cdelt, 6000, 51)
    _compare(lon, lat, v, xw, yw, 41, sigma=sigma, radius=3 * sigma, res=sigma / 2, factor=factor)


@pytest.mark.parametrize("dec,ra,cdelt,sigma", [
    (0.0, 180.0, 0.01, 0.02), (41.81, 200.0, 0.01, 0.02), (88.8, 45.0, 0.01, 0.02), (20.0, 0.01, 0.01, 0.02),
    (-60.0, 250.0, 0.2, 0.5),
])
def test_disc(gpu, dec, ra, cdelt, sigma):
    lon, lat, v, xw, yw = _scattered(41, dec, ra, cdelt, 6000, 52)
    print(f"case: disc dec={dec} ra={ra} sigma={sigma}", flush=True)
    import oracle
    dev = gridder.grid_plain(lon, lat, v, xw, yw, 41, sigma, 3 * sigma, sigma / 2, selection="disc")
    dc, wc = oracle.grid_disc_textbook(lon, lat, v.astype(np.float64), xw, yw, 3 * sigma, 1.0 / (2 * sigma * sigma))
    e, ew = map_errors(dev["map"], normalise(dc, wc)), map_errors(dev["weightscube"], wc)
    print(f"  map={e} weights={ew}", flush=True)
    assert e["nan_match"] and e["cells"] > 0
    assert e["max_rel"] <= 1e-6 and ew["max_rel"] <= 1e-6


@pytest.mark.parametrize("dec", [0.0, 41.8, -84.0])
def test_cube(gpu, dec):
    _run_case(40, 200, 27, 20, "f16", 0, seed=53, dec=dec)
