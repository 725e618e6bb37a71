"""The GAUSS2D and TAPERED_SINC weights from tangent-frame offsets and series,
on both sides of the rules that choose them, against the oracle.

Tolerance 1e-9: |p - q|^2 from FP64 unit vectors is good to 1e-12 relative at
these radii, an exponent is at most 40 times that, and a map cell is a
quotient of two such sums.
"""
import numpy as np
import pytest

from hcgrid_amd import GAUSS2D, TAPERED_SINC, synth

from test_gpu_plain import _compare, _target_coords

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kt,params,radius,dec,cdelt", [
    (GAUSS2D, [0.02, 0.012, 0.4], 0.06, 30.0, 0.01),
    (GAUSS2D, [0.02, 0.02, -2.0], 0.06, -62.0, 0.01),
    (GAUSS2D, [0.02, 0.015, 0.3], 0.06, 88.5, 0.01),
    (GAUSS2D, [0.3, 0.35, 1.0], 1.1, 10.0, 0.2),      # below the radius limit (~1.146 deg)
    (GAUSS2D, [0.4, 0.35, 1.0], 1.2, 10.0, 0.2),      # above it: the general form
    (GAUSS2D, [0.02, 0.0015, 0.3], 0.06, 20.0, 0.01),  # exponents down to -800: general
    (TAPERED_SINC, [0.02, 1.55, 2.52], 0.06, 30.0, 0.01),
    (TAPERED_SINC, [0.02, 1.55, 2.357], 0.06, 30.0, 0.01),  # x^2 to 15.99: the series
    (TAPERED_SINC, [0.02, 1.55, 2.355], 0.06, 30.0, 0.01),  # 16.02: the general form
    (TAPERED_SINC, [0.4, 1.55, 2.52], 1.1, -35.0, 0.2),
])
def test_frame_weights(gpu, kt, params, radius, dec, cdelt):
    f = cdelt / 0.01
    wl = synth.raster_small(30, 150, 20, dec_c=dec, cdelt=cdelt, spacing_dec=0.02 * f,
                            spacing_ra=0.0032 * f / np.cos(np.radians(dec)), seed=21)
    xw, yw = _target_coords(wl.target)
    _compare(wl.lon, wl.lat, wl.values, xw, yw, wl.target.side, radius=radius, res=radius / 6, kernel_type=kt,
             kernel_params=params, tol=1e-9)
