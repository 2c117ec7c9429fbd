"""The resident solves against the launch-per-phase forms, bit for bit: the
same products, sums and scalars in another arrangement.  Kernel timing
(prof_enable) keeps the launch-per-phase form, so the same solve runs in both.
The sizes cover each launch shape of the resident form and its edges: a few
row blocks, one block per workgroup up to the last and first size of the next
shape, several rows per thread; several scenarios in one launch; and a system
whose columns are spread too far for the windows, which both calls then solve
launch by launch."""
import numpy as np
import pytest


def _both(pkg, c, run):
    out = []
    for timed in (True, False):
        s = pkg.Scenario(c)
        s.init_state()
        s.prof_enable(timed)
        out.append(run(s))
        s.close()
    return out


def _stats(st):
    return (st.iterations, st.outer, st.converged, st.breakdown, st.rel_residual, st.bnorm)


def _tank(cases, nx, ny):
    if nx == 12:
        c = cases.tiny_box(nx=nx, ny=ny)
    else:
        c = cases.porous_flume(dx=0.005, length=nx * 0.005, depth=ny * 0.005, toe=1e3,
                               tank_h=ny * 0.005 + 0.05, wavemaker=False)
        fl = c.parts["tid"] == 3
        rng = np.random.default_rng(nx)
        c.parts["x"][fl] += rng.uniform(-5e-5, 5e-5, fl.sum())
        c.parts["u"][fl] = 0.02 * np.sin(c.parts["x"][fl] * 9.0)
    return c


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nx,ny,iters", [
    (12, 10, 20000),     # one to a few row blocks, to convergence
    (200, 40, 20000),    # ~36 blocks, to convergence
    (640, 100, 60),      # ~256 blocks: either side of one block per workgroup
    (660, 100, 60),
    (1280, 100, 40),     # ~512 blocks: either side of two per workgroup
    (1320, 100, 40),
    (1500, 170, 30),     # ~1020 blocks: the last of one row per thread
    (1640, 160, 30),     # two rows per thread
    (3400, 160, 20),     # three rows per thread
])
def test_resident_solve_equals_launches(pkg, cases, nx, ny, iters, precision):
    c = _tank(cases, nx, ny)
    c.params.update(precision=precision, tol=1e-10, max_iter=iters, max_outer=2)
    print(f"resident: n={c.n}, {(c.n + 255) // 256} row blocks, precision {precision}", flush=True)

    def run(s):
        rc, st = s.step(1, check=False)
        return rc, _stats(st), s.solution(), s.download()

    a, b = _both(pkg, c, run)
    assert a[0] == b[0] and a[1] == b[1], (a[:2], b[:2])
    assert np.array_equal(a[2], b[2])
    for k in a[3]:
        assert np.array_equal(a[3][k], b[3][k]), k


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nx,ny", [(200, 40), (1400, 100), (2200, 160)])
def test_rows_longer_than_those_kept_on_the_chip(pkg, cases, nx, ny, precision):
    """Fluid pressed together by a quarter: rows of more than 24 entries, whose
    ends the solves read from memory."""
    c = _tank(cases, nx, ny)
    fl = c.parts["tid"] == 3
    x0 = c.parts["x"][fl].min()
    c.parts["x"][fl] = x0 + 0.75 * (c.parts["x"][fl] - x0)
    c.params.update(precision=precision, tol=1e-10, max_iter=60, max_outer=2)

    def run(s):
        rc, st = s.step(1, check=False)
        longest = int(s.ppe()[0].max())
        return rc, _stats(st), s.solution(), s.download(), longest

    a, b = _both(pkg, c, run)
    print(f"resident: n={c.n}, longest row {b[4]}", flush=True)
    assert b[4] > 24
    assert a[0] == b[0] and a[1] == b[1], (a[:2], b[:2])
    assert np.array_equal(a[2], b[2])
    for k in a[3]:
        assert np.array_equal(a[3][k], b[3][k]), k


@pytest.mark.gpu
def test_far_columns_solve_launch_by_launch(pkg, cases):
    """Each row couples to rows all over the system: no window holds them."""
    c = cases.dam_break(dx=0.0025)
    c.params.update(precision=0, tol=1e-10, max_iter=400)
    n, W = 20000, pkg.ROW_CAP
    rng = np.random.default_rng(5)
    col = np.sort(rng.choice(n, (n, 12)), axis=1)
    col[:, 0] = np.arange(n)
    val = np.full(col.shape, -0.04)
    val[:, 0] = 1.0
    C, V = np.zeros((n, W), np.int32), np.zeros((n, W))
    C[:, :12], V[:, :12] = col, val
    rhs = np.linspace(1.0, 2.0, n)
    print("resident: columns spread over the whole system", flush=True)

    def run(s):
        s.load_system(np.full(n, 12), C, V, rhs, np.zeros(n))
        st = s.ppe_solve(check=False)
        x = np.empty(c.n)
        pkg.lib().isph_ppe_get_solution(s.handle, x.ctypes.data)
        return _stats(st), x[:n]

    a, b = _both(pkg, c, run)
    assert a[0] == b[0] and a[0][2] == 1
    assert np.array_equal(a[1], b[1])
    r = rhs - (val * a[1][col]).sum(1)
    assert np.linalg.norm(r) <= 1e-9 * np.linalg.norm(rhs)


@pytest.mark.gpu
def test_resident_batch_equals_launches(pkg, cases):
    """Scenarios of uneven size in one resident launch, one of them finishing
    at once (a tank at rest without gravity), against the timed (launch by
    launch) batch."""
    sizes = [(12, 10), (200, 40), (330, 61), (660, 100), (900, 130)]
    out = []
    for timed in (True, False):
        scen = []
        for q, (nx, ny) in enumerate(sizes):
            c = _tank(cases, nx, ny)
            c.params.update(precision=1, tol=1e-9, max_iter=200)
            if q == 1:
                c.params.update(g=0.0)
                c.parts["u"][:] = 0.0
            s = pkg.Scenario(c)
            s.init_state()
            s.prof_enable(timed)
            scen.append(s)
        print("resident batch: n =", [s.n for s in scen], "timed", timed, flush=True)
        b = pkg.Batch(scen)
        b.step(2, check=False)
        stats = [_stats(b.stats(q)) for q in range(len(scen))]
        b.close()
        out.append((stats, [s.download() for s in scen]))
        for s in scen:
            s.close()
    assert out[0][0] == out[1][0]
    for a, b in zip(out[0][1], out[1][1]):
        for k in a:
            assert np.array_equal(a[k], b[k], equal_nan=True), k
