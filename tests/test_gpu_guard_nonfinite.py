"""Samples just outside a cell's radius that carry a non-finite weight or
value: the radius test decides such a pair exactly, and a rejected one adds
nothing to the cell.  The oracle has the same sums and the same NaN cells."""
import numpy as np
import pytest

import oracle
from hcgrid_amd import GAUSS1D, GAUSS2D, gridder, synth

from test_gpu_plain import _target_coords

pytestmark = pytest.mark.gpu

RADIUS, RES = 0.06, 0.01


def _with_edge_samples(wl, xw, yw, cells):
    """The workload's samples and, north of each of the cells, one within
    rounding of the radius and two less than 1e-6 of it outside."""
    north = RADIUS * np.array([1.0, 1.0 + 2e-7, 1.0 + 7e-7])
    lon = np.concatenate([wl.lon, np.repeat(xw[cells], 3)])
    lat = np.concatenate([wl.lat, (yw[cells][:, None] + north[None, :]).ravel()])
    return lon, lat


def _same(dev, ref, what):
    bad_d, bad_r = ~np.isfinite(dev), ~np.isfinite(ref)
    assert np.array_equal(bad_d, bad_r), f"{what}: {bad_d.sum()} non-finite cells, the oracle {bad_r.sum()}"
    assert bad_r.any() and not bad_r.all()
    ok = ~bad_r
    assert np.max(np.abs(dev[ok] - ref[ok])) <= 1e-6 * np.max(np.abs(ref[ok]))


@pytest.mark.parametrize("side", [20, 70, 200])
@pytest.mark.parametrize("kt,params", [(GAUSS1D, [0.02]), (GAUSS2D, [0.02, 0.012, 0.4])])
@pytest.mark.parametrize("weight", [np.nan, np.inf])
def test_plain_weights(gpu, side, kt, params, weight):
    wl = synth.raster_small(30, 150, side, seed=51)
    xw, yw = _target_coords(wl.target)
    cells = np.arange(side * side // 2 + side // 2, side * side, max(side * side // 9, 7 * side))[:5]
    cells = cells[:1] if side < 64 else cells
    lon, lat = _with_edge_samples(wl, xw, yw, cells)
    rng = np.random.default_rng(5)
    data = np.concatenate([wl.values, np.ones(3 * len(cells))])
    w = np.concatenate([rng.uniform(0.5, 2.0, wl.n), np.full(3 * len(cells), weight)])
    print(f"case: plain side={side} kt={kt} weight={weight} n={len(lon)}", flush=True)
    dev = gridder.grid_plain(lon, lat, data, xw, yw, side, 0.02, RADIUS, RES, weights=w, kernel_type=kt,
                             kernel_params=params)
    ref = oracle.pipeline(lon, lat, data, xw, yw, side, 0.02, RADIUS, RES, weights=w, kernel_type=kt,
                          kernel_params=params)
    _same(dev["weightscube"], ref["weightscube"], "weights")
    _same(dev["datacube"], ref["datacube"], "data")


@pytest.mark.parametrize("nchan", [2, 7])
def test_few_channels_values(gpu, nchan):
    import torch
    side = 512
    wl = synth.raster_small(30, 150, side, seed=52)
    xw, yw = _target_coords(wl.target)
    cells = (np.arange(40, 480, 20)[:, None] * side + np.arange(40, 480, 20)[None, :]).ravel()
    lon, lat = _with_edge_samples(wl, xw, yw, cells)
    rng = np.random.default_rng(6)
    V = rng.uniform(0.5, 2.0, (nchan, len(lon))).astype(np.float32)
    V[:, wl.n:] = np.inf
    Vt = torch.tensor(V).to(torch.bfloat16).cuda()
    assert len(lon) * 10 <= side * side
    print(f"case: few nchan={nchan} n={len(lon)}", flush=True)
    kern, hp = gridder.prepare_grid_kernel(GAUSS1D, [0.02], RADIUS, RES)
    g = gridder.CubeGridder(len(lon), side, nchan, kern, hp)
    d = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda")  # noqa: E731
    g.run(d(lon), d(lat), Vt, d(xw), d(yw), normalize=False)
    torch.cuda.synchronize()
    Vr = Vt.float().cpu().numpy()
    ref = oracle.pipeline(lon, lat, np.ones(len(lon)), xw, yw, side, 0.02, RADIUS, RES)
    out, _ = oracle.grid_compat_multi(ref["h"], ref["g"], ref["lon_s"], ref["lat_s"], Vr[:, ref["perm"]], None,
                                      ref["keys_sorted"], ref["firstring"], ref["usedrings"], ref["lut"], xw, yw,
                                      0, side)
    cube = g.cube.cpu().numpy().reshape(nchan, -1)
    for ch in (0, nchan - 1):
        _same(cube[ch], out[ch].astype(np.float32), f"channel {ch}")


@pytest.mark.parametrize("nchan", [3, 40, 100])
@pytest.mark.parametrize("weight", [np.nan, np.inf])
def test_contraction_weights(gpu, nchan, weight):
    import ctypes as C

    import torch
    from hcgrid_amd import capi
    side = 70
    wl = synth.raster_small(30, 150, side, seed=53)
    xw, yw = _target_coords(wl.target)
    cells = np.arange(side * side // 2 + side // 2, side * side, 7 * side)[:4]
    lon, lat = _with_edge_samples(wl, xw, yw, cells)
    n, rng = len(lon), np.random.default_rng(7)
    w = np.concatenate([rng.uniform(0.5, 2.0, wl.n), np.full(3 * len(cells), weight)])
    Vt = torch.tensor(rng.uniform(0.5, 2.0, (nchan, n)).astype(np.float32)).to(torch.bfloat16).cuda()
    print(f"case: contraction nchan={nchan} weight={weight} n={n}", flush=True)
    kern, hp = gridder.prepare_grid_kernel(GAUSS1D, [0.02], RADIUS, RES)
    g = gridder.CubeGridder(n, side, nchan, kern, hp)
    d = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda")  # noqa: E731
    x, y, lo, la, p = d(xw), d(yw), d(lon), d(lat), gridder._ptr
    g.plain.presort(lo, la)
    g.gather_records(lo, la)
    g.plain.ring_lut()
    g.gather_channels(Vt)
    perm = g.plain.perm()
    ws, b = d(w[perm]), g.plain.buf
    capi.call("hcg_grid_mfma", C.byref(hp), C.byref(kern), side, n, nchan, g.dcode, p(b.records), p(b.keys),
              p(b.lon_s), p(b.lat_s), p(ws), p(g.values_sorted), p(b.lut), p(b.ring_z), p(b.ring_s), p(b.meta),
              p(x), p(y), p(g.cube), p(g.wsum), 0, gridder._stream_handle(None))
    torch.cuda.synchronize()
    Vr = Vt.float().cpu().numpy()
    ref = oracle.pipeline(lon, lat, Vr[0], xw, yw, side, 0.02, RADIUS, RES, weights=w)
    wsum, cube = g.wsum.cpu().numpy(), g.cube.cpu().numpy().reshape(nchan, -1)[0]
    for dev, r in ((wsum, ref["weightscube"]), (cube, ref["datacube"])):
        bad = ~np.isfinite(r)
        assert np.array_equal(~np.isfinite(dev), bad) and bad.any() and not bad.all()
        ok = ~bad
        # weights carried to ~2^-17, FP32 sums
        assert np.max(np.abs(dev[ok] - r[ok])) <= 1e-4 * np.max(np.abs(r[ok]))
