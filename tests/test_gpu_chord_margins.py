"""Tiles far larger than the radius: each cell's only sample sits in the corner
of its pixel, the cell beyond that corner and just within the radius, so the
ring chord's single-precision margins decide whether the pair is met at all.
Selection against the oracle, all routes of the tile loop and the contraction."""
import ctypes as C
import math

import numpy as np
import pytest

import oracle
from hcgrid_amd import GAUSS1D, capi, gridder

pytestmark = pytest.mark.gpu


def _corner_pairs(hp, side, radius, seed):
    lib = capi.load()
    rng = np.random.default_rng(seed)
    ns, R, cells, samples = int(hp.nside), math.radians(radius), [], []
    sp, npr = C.c_uint64(), C.c_uint64()

    def ring_z(r):
        lib.hcg_host_ring_info(C.byref(hp), r, C.byref(sp), C.byref(npr))
        return math.cos(lib.hcg_host_pix2theta(C.byref(hp), sp.value))

    while len(cells) < side * side:
        r = 2 * ns + int(rng.integers(-ns // 20, ns // 20))
        away = 1 if rng.integers(2) else -1
        za, z0 = ring_z(r + away), ring_z(r)
        p = int(rng.integers(int(0.42 * npr.value), int(0.55 * npr.value)))
        shift = 0.5 if (r - ns) % 2 == 0 else 0.0
        lon = 360.0 * (p + shift) / npr.value
        lat = math.asin(za + (z0 - za) * 10.0 ** rng.uniform(-8, -4))
        if lib.hcg_host_pix2ring(C.byref(hp), lib.hcg_host_ang2pix(C.byref(hp), math.pi / 2 - lat,
                                                                   math.radians(lon))) != r:
            continue
        samples.append((lon, math.degrees(lat)))
        cells.append((lon, math.degrees(lat - away * R * (1 - 10.0 ** rng.uniform(-7, -4)))))
    return np.array(cells), np.array(samples)


@pytest.mark.parametrize("side", [16, 48, 130])
@pytest.mark.parametrize("radius", [0.0005, 0.02])
def test_far_larger_tiles(gpu, side, radius):
    import torch
    kern, hp = gridder.prepare_grid_kernel(GAUSS1D, [radius / 3], radius, 0.01)
    cells, samples = _corner_pairs(hp, side, radius, seed=side)
    lon, lat = samples[:, 0], samples[:, 1]
    xw, yw = np.ascontiguousarray(cells[:, 0]), np.ascontiguousarray(cells[:, 1])
    print(f"case: side={side} radius={radius} n={len(lon)}", flush=True)
    data = np.random.default_rng(1).uniform(1.0, 2.0, len(lon))
    ref = oracle.pipeline(lon, lat, data, xw, yw, side, radius / 3, radius, 0.01)
    met = ref["weightscube"] > 0
    assert met.mean() > 0.9
    dev = gridder.grid_plain(lon, lat, data, xw, yw, side, radius / 3, radius, 0.01)
    assert np.array_equal(dev["weightscube"] > 0, met)
    for nchan in (1, 3, 300):
        V = torch.tensor(np.repeat(data[None, :], nchan, 0)).to(torch.bfloat16).cuda()
        cube = gridder.grid_cube(lon, lat, V, xw, yw, side, radius / 3, radius, 0.01)
        assert np.array_equal(cube["wsum"] > 0, met), nchan
