"""The contraction kernel's instances at their edges, against the FP64 oracle:
channel counts on both sides of every instance, the many-channel kernel with
and without its plan and over more than 64 rings per block, general weights,
and pairs within rounding of the radius.  Bounds as in test_gpu_cube (weights
carried to ~2^-17, FP32 sums)."""
import numpy as np
import pytest

import oracle
from hcgrid_amd import GAUSS1D, GAUSS2D, gridder, synth

from helpers import map_errors
from test_gpu_cube import _run_case, _values

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nchan", [2, 3, 16, 17, 33, 65, 96, 97, 129, 192, 193, 256, 257, 513])
def test_instance_edges(gpu, nchan):
    _run_case(40, 200, 27, nchan, "bf16" if nchan % 2 else "f16", 0, seed=300 + nchan)


@pytest.mark.parametrize("dec", [-78.0, -41.8, 41.5, 88.5])
def test_many_channels_declinations(gpu, dec):
    # both sides of the polar caps' edge (rings of general windows), a map over the pole
    _run_case(40, 200, 24, 260, "bf16", 0, seed=41, dec=dec)


def _grid(wl, side, nchan, kt, params, radius, res, plan=True, shape=None, extra=None):
    import torch
    t = wl.target
    xw, yw = gridder.wcs_sin(side, side, t.crpix, t.crpix, -t.cdelt, t.cdelt, t.crval1, t.crval2)
    lon, lat = wl.lon, wl.lat
    V = _values(wl, nchan, 9)
    if extra is not None:
        xe, ye = extra(xw, yw)
        lon, lat = np.concatenate([lon, xe]), np.concatenate([lat, ye])
        V = np.concatenate([V, np.ones((nchan, len(xe)), np.float32)], axis=1)
    Vt = torch.tensor(V).to(torch.bfloat16).cuda()
    kern, hp = gridder.prepare_grid_kernel(kt, params, radius, res)
    g = gridder.CubeGridder(len(lon), side, nchan, kern, hp)
    d = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda")  # noqa: E731
    g.run(d(lon), d(lat), Vt, d(xw), d(yw), shape=shape)
    torch.cuda.synchronize()
    cube, wsum = g.cube.cpu().numpy().copy(), g.wsum.cpu().numpy().copy()
    if plan:
        g.grid(d(xw), d(yw), shape=shape, plan=False)
        torch.cuda.synchronize()
        assert np.array_equal(cube, g.cube.cpu().numpy(), equal_nan=True)
        assert np.array_equal(wsum, g.wsum.cpu().numpy())
    Vr = Vt.float().cpu().numpy()
    ref = oracle.pipeline(lon, lat, Vr[0], xw, yw, side, 0.0, radius, res, kernel_type=kt, kernel_params=params)
    out, ws = oracle.grid_compat_multi(ref["h"], ref["g"], ref["lon_s"], ref["lat_s"], Vr[:, ref["perm"]], None,
                                       ref["keys_sorted"], ref["firstring"], ref["usedrings"], ref["lut"], xw, yw,
                                       0, side)
    with np.errstate(invalid="ignore", divide="ignore"):
        e = map_errors(cube.reshape(-1), (out / ws[None, :]).reshape(-1))
    wrel = np.abs(wsum - ws)[ws > 0] / ws[ws > 0]
    print(f"  errors {e} wsum_rel_max {wrel.max():.2e}", flush=True)
    assert e["nan_match"] and e["max_rel"] <= 1e-4 and e["rms_rel"] <= 1e-4
    assert wrel.max() <= 2.0 ** -14


@pytest.mark.parametrize("sigma,radius,shape", [(0.02, 0.06, None), (0.08, 0.24, None), (0.08, 0.24, (64, 0, 0)),
                                                (0.1, 0.3, (8, 0, 0))])
def test_plan_and_set_up_agree(gpu, sigma, radius, shape):
    # at nside 8192 the wider beams span 70 rings and more per block, which no
    # plan holds; the last one is past the lean weight's radius
    wl = synth.raster_small(40, 200, 24, seed=31)
    print(f"case: sigma={sigma} shape={shape}", flush=True)
    _grid(wl, 24, 280, GAUSS1D, [sigma], radius, 0.01, shape=shape)


@pytest.mark.parametrize("nchan", [1, 3, 70])
def test_general_weights(gpu, nchan):
    wl = synth.raster_small(30, 150, 20, seed=33)
    print(f"case: general weights nchan={nchan}", flush=True)
    _grid(wl, 20, nchan, GAUSS2D, [0.02, 0.015, 0.3], 0.06, 0.01)


@pytest.mark.parametrize("nchan", [5, 40, 300])
def test_pairs_at_the_radius(gpu, nchan):
    # samples at a cell's longitude and its latitude +- the radius: rounding
    # decides each, and the reference's formula has to
    wl = synth.raster_small(12, 60, 20, spacing_dec=0.05, spacing_ra=0.02, seed=35)
    print(f"case: pairs at the radius nchan={nchan}", flush=True)
    pick = np.arange(7, 400, 3)
    _grid(wl, 20, nchan, GAUSS1D, [0.02], 0.06, 0.01,
          extra=lambda x, y: (np.concatenate([x[pick], x[pick]]), np.concatenate([y[pick] + 0.06, y[pick] - 0.06])))
