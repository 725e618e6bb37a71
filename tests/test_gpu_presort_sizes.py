"""The pre-sort at the sizes where its tiles, passes or digits change: sorted
keys and permutation equal numpy's stable order of the oracle's keys, with
runs of equal keys, invalid samples and the npix sentinel."""
import numpy as np
import pytest

import oracle
from hcgrid_amd import gridder

pytestmark = pytest.mark.gpu

SMALL, MID = 1024 * 512, 2048 * 768  # the last n with small and with middle tiles


@pytest.mark.parametrize("n,res,spread", [
    (1, 0.01, 1.0), (63, 0.01, 1.0), (1024, 0.01, 1.0), (1025, 0.01, 1e-6), (9000, 0.01, 180.0),
    (5000, 0.3, 180.0),    # nside 256: two passes of ten bits
    (5000, 0.25, 180.0),   # nside 512: three passes
    (7000, 30.0, 180.0),   # nside 2: two passes of a few bits
    (SMALL, 0.01, 5.0), (SMALL + 1, 0.02, 5.0), (MID, 0.01, 5.0), (MID + 1, 0.01, 5.0),
])
def test_presort_sizes(gpu, n, res, spread):
    import torch
    rng = np.random.default_rng(n)
    lon = np.mod(180.0 + rng.uniform(-spread, spread, n), 360.0)
    lat = np.clip(rng.uniform(-spread, spread, n), -90.0, 90.0)
    if n > 100:
        lon[::7], lat[::7] = lon[3], lat[3]  # many equal keys
        lat[5::101] = 91.0                   # invalid: MAX_Y, sorted last
        lat[6::103] = np.nan
    print(f"case: presort n={n} res={res} spread={spread}", flush=True)
    kern, hp = gridder.prepare_grid_kernel(1, [2 * res], 6 * res, res)
    g = gridder.PlainGridder(n, 8, kern, hp)
    d = lambda a: torch.as_tensor(a, device="cuda")  # noqa: E731
    g.presort(d(lon), d(lat))
    torch.cuda.synchronize()
    keys = oracle.sample_keys(oracle.hpx(int(hp.nside)), lon, lat)
    order = np.argsort(keys, kind="stable")
    assert np.array_equal(g.keys_sorted()[:n].astype(np.uint64), keys[order])
    assert int(g.keys_sorted()[n]) == int(hp.npix)
    assert np.array_equal(g.perm(), order.astype(np.uint32))
