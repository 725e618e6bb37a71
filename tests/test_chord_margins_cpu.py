"""The ring chord as the kernels evaluate it (their own functions, compiled for
the host): a sample within the radius of a cell is in the range of keys and
half-pixel positions that the chord leaves, also for tiles that are far larger
than the radius, near the poles, and where the single-precision margins are all
that separates a pair from the bound: a sample in the corner of its pixel, the
cell beyond that corner and just within the radius."""
import ctypes as C
import math

import numpy as np
import pytest

from hcgrid_amd import capi
from hostlib import host_lib

CODE = """
#include "mfma_job.hpp"
using namespace hcg;
// cells: (z = sin lat, cos lat, tt = lon in units of pi/2), as tile_span takes them
extern "C" int chord(int ncells, const double* z, const double* coslat, const double* tt, int cell, double half2,
                     unsigned sp, unsigned npr, unsigned kr, unsigned used, const double* ring_z, unsigned key,
                     unsigned odd) {
  TileSpan T{};
  T.zref = z[0];
  for (int i = 1; i < ncells; ++i) T.zref = fmin(T.zref, z[i]);
  float zm = 0.f, cm = 2.f, t0 = 8.f, t1 = -8.f;
  for (int i = 0; i < ncells; ++i) {
    zm = fmaxf(zm, (float)(z[i] - T.zref));
    cm = fminf(cm, (float)coslat[i]);
    t0 = fminf(t0, (float)tt[i]);
    t1 = fmaxf(t1, (float)tt[i]);
  }
  T.zmin = 0.f;
  T.zmax = zm * (1.f + 1e-6f);
  T.cmin = cm * (1.f - 1e-6f);
  T.tmin = t0 - 1e-6f;
  T.tmax = t1 + 1e-6f;
  const RingChord c = ring_chord(half2, T, npr, kr, used, ring_z);
  uint32_t lp = sp, rp = sp + npr - 1;
  if (!chord_pixels(T, c, sp, npr, lp, rp) || key < lp || key > rp) return 1;
  const CellReach reach = chord_cell([&](float RingChord::*m) { return c.*m; }, (float)(z[cell] - T.zref), (float)tt[cell]);
  if (!reach.any) return 2;
  const uint32_t g = 2 * (key - sp) + 1 - odd;
  return reach.narrow && (g < (uint32_t)reach.xl || g > (uint32_t)reach.xh) ? 3 : 0;
}
"""


@pytest.mark.parametrize("nside", [64, 1024, 8192])
@pytest.mark.parametrize("radius", [1e-5, 1e-3, 0.06, 1.0])
def test_pairs_within_the_radius_are_kept(tmp_path, nside, radius):
    lib = capi.load()
    chord = host_lib(tmp_path, CODE).chord
    hp = capi.Healpix()
    capi.call("hcg_healpix_init", nside, C.byref(hp))
    rng = np.random.default_rng(nside)
    R = math.radians(radius)
    half2 = math.sin(0.5 * R * (1 + 1e-6)) ** 2
    checked = 0
    for trial in range(6000):
        # the sample in the corner of a pixel of ring r that points away from or to the pole
        r = int(rng.choice([rng.integers(3, 4 * nside - 2), rng.integers(3, max(5, nside // 20)),
                            2 * nside + rng.integers(-3, 4)]))
        away = 1 if rng.integers(2) else -1
        zs = [math.cos(lib.hcg_host_pix2theta(C.byref(hp), _start(lib, hp, r + d))) for d in (-1, 0, 1)]
        sp, npr = _info(lib, hp, r)
        ring_z = (C.c_double * 3)(*zs)
        p = int(rng.integers(npr // 8, npr // 2))
        # a pixel's corners lie on its own centre's longitude
        shift = 0.5 if r < nside or r > 3 * nside or (r - nside) % 2 == 0 else 0.0
        tt_s = 4.0 * (p + shift) / npr
        z_s = zs[1 + away] + (zs[1] - zs[1 + away]) * 10.0 ** rng.uniform(-9, -3)
        lat_s = math.asin(z_s)
        key = lib.hcg_host_ang2pix(C.byref(hp), math.pi / 2 - lat_s, tt_s * math.pi / 2)
        if lib.hcg_host_pix2ring(C.byref(hp), key) != r:
            continue
        # the cell beyond that corner, or in any direction
        d, az = R * (1 - 10.0 ** rng.uniform(-9, -3)), rng.uniform(0, 2 * math.pi)
        lat_c, tt_c = lat_s - away * d, tt_s
        if trial % 2:
            lat_c = math.asin(math.sin(lat_s) * math.cos(d) + math.cos(lat_s) * math.sin(d) * math.cos(az))
            dl = math.atan2(math.sin(az) * math.sin(d) * math.cos(lat_s),
                            math.cos(d) - math.sin(lat_s) * math.sin(lat_c))
            tt_c = (tt_s + dl / (math.pi / 2)) % 4.0
        if abs(lat_c) > math.pi / 2 - 1e-9:
            continue
        # the tile: this cell and others up to many radii away
        ext = min(R * 10.0 ** rng.uniform(-1, 5), 0.3)
        lats = [lat_c] + [min(max(lat_c + ext * u, -1.57), 1.57) for u in rng.uniform(-1, 1, 3)]
        tts = [tt_c] + [min(max(tt_c + 0.3 * ext * u, 0.0), 3.99) for u in rng.uniform(-1, 1, 3)]
        arr = lambda v: (C.c_double * 4)(*v)  # noqa: E731
        got = chord(4, arr([math.sin(b) for b in lats]), arr([math.cos(b) for b in lats]), arr(tts), 0,
                    C.c_double(half2), sp, npr, 1, 3, ring_z, key, r & 1)
        assert got == 0, (nside, radius, r, math.degrees(lat_s), math.degrees(lat_c), ext / R, got)
        checked += 1
    assert checked > 1500


def _info(lib, hp, r):
    sp, npr = C.c_uint64(), C.c_uint64()
    lib.hcg_host_ring_info(C.byref(hp), r, C.byref(sp), C.byref(npr))
    return sp.value, npr.value


def _start(lib, hp, r):
    return _info(lib, hp, r)[0]
