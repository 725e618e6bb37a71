"""A map of 32768^2 cells: 2^24 workgroups of 256 threads, more threads than
one launch takes.  One sample each at places of the first, the last and the
runs' last tiles; the weight sums and values around them, and nothing elsewhere."""
import numpy as np
import pytest

from hcgrid_amd import GAUSS2D, batch, gridder

pytestmark = pytest.mark.gpu

SIDE, CDELT, RADIUS = 32768, 0.004, 0.014


@pytest.mark.parametrize("how", ["gridder", "batch"])
def test_contraction_over_several_launches(gpu, how):
    import torch
    if torch.cuda.mem_get_info()[0] < 80 << 30:
        pytest.skip("needs 80 GB of device memory")
    rows = [0, 2] + [SIDE // 8 * (x + 1) - 2 for x in range(8)]
    cols = [0, 20000] + [SIDE - 7] * 8
    axis = (torch.arange(SIDE, dtype=torch.float64, device="cuda") - SIDE // 2) * CDELT
    xw = (180.0 + axis)[None, :].expand(SIDE, SIDE).reshape(-1).contiguous()
    yw = axis[:, None].expand(SIDE, SIDE).reshape(-1).contiguous()
    lat = np.array([(r - SIDE // 2 + 0.1) * CDELT for r in rows])
    lon = np.array([180.0 + (c - SIDE // 2 + 0.1) * CDELT for c in cols])
    n = len(lat)
    d = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda")  # noqa: E731
    V = torch.arange(1, n + 1, device="cuda").to(torch.bfloat16)[None, :].contiguous()
    kern, hp = gridder.prepare_grid_kernel(GAUSS2D, [0.006, 0.006, 0.0], RADIUS, 0.01, 1, "disc")
    print(f"case: {how} side={SIDE} n={n}", flush=True)
    if how == "gridder":
        g = gridder.CubeGridder(n, SIDE, 1, kern, hp)
        g.plain.presort(d(lon), d(lat))
        g.gather_records(d(lon), d(lat))
        g.plain.ring_lut()
        g.gather_channels(V)
        g.grid(xw, yw, plan=False)
        cube, wsum = g.cube[0], g.wsum
    else:
        geo = batch.Geometry(kern, hp, n, SIDE, in_torch=True)
        geo.build(d(lon), d(lat), xw, yw)
        cube = torch.empty(SIDE * SIDE, dtype=torch.float32, device="cuda")
        wsum = torch.empty(SIDE * SIDE, dtype=torch.float32, device="cuda")
        b = batch.Batch([dict(geometry=geo, values=V, cube=cube.view(1, -1), wsum=wsum)])
        b.enqueue()
    torch.cuda.synchronize()
    total = 0
    for k, (r, c) in enumerate(zip(rows, cols)):
        rr = np.arange(max(r - 6, 0), min(r + 7, SIDE))
        cc = np.arange(max(c - 40, 0), min(c + 41, SIDE))
        y, x = np.radians((rr - SIDE // 2) * CDELT)[:, None], np.radians(180.0 + (cc - SIDE // 2) * CDELT)[None, :]
        b0, l0 = np.radians(lat[k]), np.radians(lon[k])
        h = np.sin((y - b0) / 2) ** 2 + np.cos(y) * np.cos(b0) * np.sin((x - l0) / 2) ** 2
        dist = np.degrees(2 * np.arcsin(np.sqrt(h)))
        want = np.where(dist < RADIUS, np.exp(-0.5 * (dist / 0.006) ** 2), 0.0)
        idx = torch.as_tensor(rr[:, None] * SIDE + cc[None, :], device="cuda")
        got, val = wsum[idx].double().cpu().numpy(), cube[idx].cpu().numpy()
        assert want.any() and np.max(np.abs(got - want)) <= 2.0 ** -14
        assert np.array_equal(got > 0, want > 0)
        assert np.all(np.abs(val[want > 0] - (k + 1)) <= 1e-4 * (k + 1)) and np.isnan(val[want == 0]).all()
        total += int((want > 0).sum())
    assert int(torch.count_nonzero(wsum)) == total
