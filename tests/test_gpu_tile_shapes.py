"""The tile loop at the sizes where its launch or a ring's handling changes,
against the oracle (the bar of test_gpu_plain: maps and weights within 1e-6).

* sides on both sides of the rules that choose a tile's rows and waves
  (16 x 4 tiles: 138, 552, 2093 and 4096 of them), none a multiple of 16;
* fields across the longitude where windows wrap, and across the declination
  (41.8 deg) where belt rings meet the polar caps' and a cell's window stops
  being one pair of numbers for every ring;
* rings longer than a staged chunk, and rings of a few samples.
"""
import numpy as np
import pytest

from hcgrid_amd import synth

from test_gpu_plain import _compare, _target_coords

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side,lines,per,dec,ra,weighted", [
    (90, 60, 150, 30.0, 180.0, False),
    (90, 50, 120, 41.8, 0.05, True),
    (182, 90, 150, 41.8, 180.0, False),
    (182, 80, 160, -20.0, 0.3, False),
    (182, 60, 90, -41.9, 180.0, True),
    (364, 120, 160, 10.0, 180.0, False),
    (509, 100, 120, 41.8, 180.0, False),
    (20, 8, 6000, 30.0, 180.0, True),  # rings of hundreds of samples per chunk
    (37, 6000, 4, 0.0, 180.0, False),  # every line its own short rings
])
def test_tile_shapes(gpu, side, lines, per, dec, ra, weighted):
    field = side * 0.01
    wl = synth.raster_small(lines, per, side, dec_c=dec, ra_c=ra, spacing_dec=field / lines,
                            spacing_ra=field / per / np.cos(np.radians(dec)), seed=side + lines)
    wl.lon[:] = np.mod(wl.lon, 360.0)
    xw, yw = _target_coords(wl.target)
    w = np.random.default_rng(side).uniform(0.5, 1.5, wl.n) if weighted else None
    _compare(wl.lon, wl.lat, wl.values, xw, yw, side, weights=w)
