"""The rebin's scan over cell grids on both sides of the size at which it takes
a pass of its own for the tiles' offsets."""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("cells", [(1279, 1280), (1300, 1310)])
def test_rebin_over_a_wide_grid(pkg, cases, cells):
    c = cases.dam_break(dx=0.02)
    nx, ny = cells
    c.params.update(cellx=nx, celly=ny)
    cs = 4.0 * c.params["h"]
    c.parts["x"] = c.parts["x"] + cs * (nx - 60)
    c.parts["y"] = c.parts["y"] + cs * (ny // 2)
    c.parts["u"][c.parts["tid"] == 3] = 100.0
    print(f"rebin: {nx} x {ny} cells, n={c.n}", flush=True)
    s = pkg.Scenario(c)
    s.init_state()
    moved = 0
    for _ in range(3):
        before, _ = s.cells()
        s.projection()
        s.cellshift()
        cell, start = s.cells()
        assert np.all(np.diff(cell) >= 0)
        assert np.array_equal(start, np.searchsorted(cell, np.arange(nx * ny + 1)))
        d = s.download()
        cj, ci = cell // ny, cell % ny
        assert np.all(np.abs(d["x"] - (cj - 0.5) * cs) <= 0.5 * cs + 1e-9)
        assert np.all(np.abs(d["y"] - (ny - 1.5 - ci) * cs) <= 0.5 * cs + 1e-9)
        moved += int((before != cell).sum())
    s.close()
    assert moved > 0
