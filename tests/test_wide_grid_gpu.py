"""Domains with many more cells than their particles fill: the rebin's scan on
both sides of the size at which it takes a pass of its own for the tiles'
offsets, the cell maxima on both sides of the size to which four lanes share a
cell, and the precision solve on both sides of the cells that its resident form
takes on."""
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


@pytest.mark.gpu
@pytest.mark.parametrize("dx,cells,resident", [
    (0.0025, (290, 320), True), (0.0025, (300, 320), False),  # of 94,208 in all
    (0.02, (80, 100), True), (0.02, (84, 100), False),        # of 4 per thread, 2,048 threads
])
def test_cells_of_a_resident_solve(pkg, cases, dx, cells, resident):
    out = []
    for timed in (True, False):
        c = cases.dam_break(dx=dx)
        c.params.update(cellx=cells[0], celly=cells[1], precision=1, tol=1e-9, max_iter=30,
                        max_outer=1)
        off = 4.0 * c.params["h"] * 5
        c.parts["x"], c.parts["y"] = c.parts["x"] + off, c.parts["y"] + off
        print(f"cells: {cells}, n={c.n}, timed {timed}", flush=True)
        s = pkg.Scenario(c)
        s.init_state()
        s.prof_enable(timed)
        rc, st = s.step(1, check=False)
        out.append((rc, st.iterations, st.rel_residual, s.solution(), s.resident_counts()))
        s.close()
    assert out[1][4]["launches"] == int(resident) and out[1][4]["too_wide"] == 0
    assert out[0][:3] == out[1][:3] and out[0][1] > 3
    assert np.array_equal(out[0][3], out[1][3])


@pytest.mark.gpu
@pytest.mark.parametrize("cells", [(512, 512), (513, 512)])
def test_cell_maxima(pkg, cases, cells):
    """umax is the largest pore velocity of the fluid whatever the grid."""
    c = cases.dam_break(dx=0.005)
    c.params.update(cellx=cells[0], celly=cells[1], tol=1e-6, max_iter=50, max_outer=0)
    fl = c.parts["tid"] == 3
    rng = np.random.default_rng(5)
    c.parts["u"][fl] = rng.uniform(-0.3, 0.3, fl.sum())
    off = 4.0 * c.params["h"] * 200
    c.parts["x"], c.parts["y"] = c.parts["x"] + off, c.parts["y"] + off
    print(f"cell maxima: {cells}", flush=True)
    s = pkg.Scenario(c)
    s.init_state()
    for ph in ("projection", "cellshift", "neighbour", "effpor", "eddyvis", "int_vel"):
        getattr(s, ph)()
    s.ppe_assemble()
    s.ppe_solve(check=False)
    s.comp_vel()
    d, p = s.download(), s.props()
    s.timestep()
    um = s.scalars().umax
    fl = (d["tid"] == 3) & ((d["flags"] & 1) == 0)
    want = np.sqrt(d["u"] * d["u"] + d["v"] * d["v"]) / p["porosity"]
    assert um == want[fl].max() == p["vel"][fl].max() and um > 0.0
    s.close()
