"""A workspace (or a geometry's memory) sized for the largest input serves
every smaller one: the sizes never fall as n grows, across the sample counts
where the sort changes its tile too."""
import ctypes as C

import pytest

from hcgrid_amd import capi

EDGES = (1024, 524288, 1572864, 8388608)


def _counts():
    near = {e + d for e in EDGES for d in (-4097, -1025, -257, -2, -1, 0, 1, 2, 257, 1025, 4097)}
    return sorted({1, 2, 63, 64, 65} | {n for n in near if n > 0} | {int(1.07 ** k) for k in range(1, 320)})


def test_workspace_size_never_falls():
    size = capi.load().hcg_presort_workspace_size
    counts = _counts()
    sizes = [size(n) for n in counts]
    for a, b, sa, sb in zip(counts, counts[1:], sizes, sizes[1:]):
        assert sa <= sb, (a, b, sa, sb)


@pytest.mark.parametrize("nside", [256, 8192])
def test_geometry_bytes_never_fall(nside):
    lib = capi.load()
    hp = capi.Healpix()
    capi.call("hcg_healpix_init", nside, C.byref(hp))
    counts = _counts()
    sizes = [lib.hcg_geometry_bytes(n, 64, C.byref(hp)) for n in counts]
    for a, b, sa, sb in zip(counts, counts[1:], sizes, sizes[1:]):
        assert sa <= sb, (a, b, sa, sb)
