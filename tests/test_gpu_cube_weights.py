"""The contraction's weights from series, kind by kind, on both sides of the
rules that choose them, against the FP64 oracle: bounds as in test_gpu_cube
(weights carried to ~2^-17, FP32 sums) with bf16, and with fp16, which carries
them to ~2^-22, 2^-19 on the weight sums."""
import ctypes as C

import numpy as np
import pytest

import oracle
from hcgrid_amd import GAUSS1D, GAUSS2D, TAPERED_SINC, capi, gridder, synth

from helpers import map_errors
from test_gpu_plain import _target_coords

pytestmark = pytest.mark.gpu

CASES = [
    (GAUSS1D, [0.02], 0.06, 1.0, False), (GAUSS1D, [0.02], 0.06, 1.0, True),   # lean; with sample weights
    (GAUSS1D, [0.15], 0.45, 8.0, True),                                          # small radius
    (GAUSS1D, [0.35], 1.13, 20.0, False), (GAUSS1D, [0.35], 1.16, 20.0, True),  # the series' ends (1.146 deg)
    (GAUSS1D, [3.2], 9.7, 150.0, False), (GAUSS1D, [3.2], 10.1, 150.0, True),   # series, calls (9.93 deg)
    (GAUSS2D, [0.02, 0.012, 0.4], 0.06, 1.0, False), (GAUSS2D, [0.9, 0.6, -2.0], 2.6, 40.0, True),
    (GAUSS2D, [3.2, 2.5, 0.4], 9.7, 150.0, False), (GAUSS2D, [3.2, 2.5, 0.4], 10.1, 150.0, False),
    (GAUSS2D, [0.02, 0.0008, 0.3], 0.06, 1.0, True),                             # exponents down to -2800
    (TAPERED_SINC, [0.02, 1.55, 2.52], 0.06, 1.0, False), (TAPERED_SINC, [0.9, 1.55, 2.52], 2.6, 40.0, True),
    (TAPERED_SINC, [0.02, 3.0, 0.79], 0.06, 1.0, False),   # x to 11.93: the series
    (TAPERED_SINC, [0.02, 3.0, 0.78], 0.06, 1.0, False),   # 12.08: calls
]


@pytest.mark.parametrize("kt,params,radius,scale,weighted", CASES)
@pytest.mark.parametrize("nchan,dtype,dec", [(3, "bf16", -25.0), (40, "f16", 12.0), (100, "bf16", 30.0),
                                             (200, "f16", 30.0), (300, "bf16", -5.0)])
def test_weights(gpu, kt, params, radius, scale, weighted, nchan, dtype, dec):
    import torch
    if kt == TAPERED_SINC and dtype == "f16" and (np.pi * radius / params[0] / params[1]) ** 2 > np.log(65504.0):
        pytest.skip("FP16 does not hold this kernel's weights (it grows to exp(t^2), far above 65504)")
    side = 21
    wl = synth.raster_small(26, 130, side, dec_c=dec, cdelt=0.01 * scale, spacing_dec=0.02 * scale,
                            spacing_ra=0.0032 * scale / np.cos(np.radians(dec)), seed=71)
    xw, yw = _target_coords(wl.target)
    rng = np.random.default_rng(nchan)
    n, V = wl.n, rng.uniform(0.5, 2.0, (nchan, wl.n)).astype(np.float32)
    w = rng.uniform(0.5, 2.0, n) if weighted else None
    Vt = torch.tensor(V).to(torch.bfloat16 if dtype == "bf16" else torch.float16).cuda()
    print(f"case: kt={kt} params={params} radius={radius} w={weighted} nchan={nchan} {dtype} dec={dec}", flush=True)
    kern, hp = gridder.prepare_grid_kernel(kt, params, radius, max(radius / 6, 0.0075))
    g = gridder.CubeGridder(n, side, nchan, kern, hp, dtype=dtype)
    d = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda")  # noqa: E731
    x, y, lo, la, p = d(xw), d(yw), d(wl.lon), d(wl.lat), gridder._ptr
    g.plain.presort(lo, la)
    g.gather_records(lo, la)
    g.plain.ring_lut()
    g.gather_channels(Vt)
    ws, b = None if w is None else d(w[g.plain.perm()]), g.plain.buf
    nb = int(capi.load().hcg_grid_mfma_workspace_size(side, None))
    work = torch.empty(nb, dtype=torch.uint8, device="cuda")
    capi.call("hcg_grid_mfma_ex", C.byref(hp), C.byref(kern), side, n, nchan, g.dcode, p(b.records), p(b.keys),
              p(b.lon_s), p(b.lat_s), p(ws), p(g.values_sorted), p(b.lut), p(b.ring_z), p(b.ring_s), p(b.meta),
              p(x), p(y), p(g.cube), p(g.wsum), 0, None, p(work), nb, gridder._stream_handle(None))
    torch.cuda.synchronize()
    Vr = Vt.float().cpu().numpy()
    res = max(radius / 6, 0.0075)
    ref = oracle.pipeline(wl.lon, wl.lat, Vr[0], xw, yw, side, 0.0, radius, res, weights=w, kernel_type=kt,
                          kernel_params=params)
    wsr = None if w is None else w[ref["perm"]]
    out, wref = oracle.grid_compat_multi(ref["h"], ref["g"], ref["lon_s"], ref["lat_s"], Vr[:, ref["perm"]], wsr,
                                         ref["keys_sorted"], ref["firstring"], ref["usedrings"], ref["lut"], xw, yw,
                                         0, side)
    e = map_errors(g.cube.cpu().numpy().reshape(-1), out.reshape(-1))
    werr = np.max(np.abs(g.wsum.cpu().numpy() - wref)) / np.max(np.abs(wref))
    print(f"  errors {e} wsum {werr:.2e}", flush=True)
    assert e["nan_match"] and e["max_rel"] <= 1e-4 and e["rms_rel"] <= 1e-4
    assert werr <= (2.0 ** -14 if dtype == "bf16" else 2.0 ** -19)
