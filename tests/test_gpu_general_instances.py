"""The general weights' contraction instances (GAUSS2D, sample weights) at the
edges of their channel counts, against the FP64 oracle; bounds as in
test_gpu_mfma_instances."""
import pytest

from hcgrid_amd import GAUSS2D, synth

from test_gpu_mfma_instances import _grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nchan", [1, 2, 7, 8, 16, 17, 64, 65])
def test_general_instance_edges(gpu, nchan):
    wl = synth.raster_small(30, 150, 20, seed=200 + nchan)
    print(f"case: general instance nchan={nchan} n={wl.n}", flush=True)
    _grid(wl, 20, nchan, GAUSS2D, [0.02, 0.015, 0.3], 0.06, 0.01)
