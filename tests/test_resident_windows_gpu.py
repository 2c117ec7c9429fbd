"""Systems whose rows couple over more rows than a resident workgroup's window
holds, one for each limit that the set-up tests.  They are solved launch by
launch, which in the precision form reads column offsets where the set-up had
written window positions: the solutions are those of the launch-per-phase form
(kernel timing on), bit for bit."""
import numpy as np
import pytest

from test_resident_gpu import _stats, _tank

PHASES = ("projection", "cellshift", "neighbour", "effpor", "eddyvis", "int_vel",
          "ppe_assemble")


def _basin(cases):
    """Cell columns of some 3,800 rows, and up to 3,072 rows per workgroup."""
    return _tank(cases, 760, 760)


def _splash(cases):
    """Fluid scattered so thinly that a window of two cells per thread (one row
    per thread) has more cells than that."""
    dx, side = 0.005, 6.7
    c = cases.porous_flume(dx=dx, length=side, depth=75 * dx, toe=1e3, tank_h=side + 0.05,
                           wavemaker=False)
    fl = c.parts["tid"] == 3
    rng = np.random.default_rng(11)
    for f in ("x", "y"):
        lo = c.parts[f][fl].min()
        c.parts[f][fl] = rng.uniform(lo, lo + side - 0.1, fl.sum())
    return c


def _crowd(cases):
    """A cell with more rows beyond its workgroup than a workgroup takes from the
    next ones."""
    c = _tank(cases, 200, 40)
    fl = np.flatnonzero(c.parts["tid"] == 3)
    x, y, cs = c.parts["x"], c.parts["y"], 4.0 * c.params["h"]
    rng = np.random.default_rng(3)
    some = rng.choice(fl, 1500, replace=False)
    ox, oy = (np.floor(v[fl].mean() / cs) * cs for v in (x, y))
    x[some] = ox + cs * rng.uniform(0.05, 0.95, some.size)
    y[some] = oy + cs * rng.uniform(0.05, 0.95, some.size)
    return c


def _assembled(pkg, c):
    s = pkg.Scenario(c)
    for ph in ("init_state",) + PHASES:
        try:
            getattr(s, ph)()
        except pkg.IsphError as e:
            assert e.code == -3  # the crowded cell: more neighbours than the list holds
    return s


def _solve(s):
    st = s.ppe_solve(check=False)
    return _stats(st), s.solution()


@pytest.mark.gpu
@pytest.mark.parametrize("case,precision", [(_basin, 0), (_basin, 1), (_splash, 1), (_crowd, 1)])
def test_windows_that_do_not_fit(pkg, cases, case, precision):
    c = case(cases)
    c.params.update(precision=precision, tol=1e-10, max_iter=12, max_outer=1)
    print(f"windows: {case.__name__}, n={c.n}, precision {precision}", flush=True)
    out = []
    for timed in (True, False):
        s = _assembled(pkg, c)
        s.prof_enable(timed)
        out.append(_solve(s))
        k = s.resident_counts()
        s.close()
    assert k == dict(launches=0, too_wide=1, refused=0, ran_out=0)
    assert out[0][0] == out[1][0] and out[0][0][0] > 3
    assert np.array_equal(out[0][1], out[1][1])


@pytest.mark.gpu
@pytest.mark.parametrize("case,precision", [(_basin, 0), (_splash, 1)])
def test_windows_that_did_not_fit_are_not_tried_at_once(pkg, cases, case, precision):
    """The next 32 solves of the context leave the set-up out; a new state is
    tried at once."""
    c = case(cases)
    c.params.update(precision=precision, tol=1e-10, max_iter=3, max_outer=0)
    print(f"windows: {case.__name__}, n={c.n}, 34 solves", flush=True)
    s = _assembled(pkg, c)
    wide = []
    for _ in range(34):
        _solve(s)
        wide.append(s.resident_counts()["too_wide"])
    assert wide == 33 * [1] + [2]
    f = [s._keep[k].ctypes.data for k in pkg.PART_FIELDS + ("tid", "flags")]
    assert pkg.lib().isph_upload(s.handle, c.n, *f) == 0
    for ph in ("init_state",) + PHASES:
        getattr(s, ph)()
    _solve(s)
    assert s.resident_counts() == dict(launches=0, too_wide=3, refused=0, ran_out=0)
    s.close()


@pytest.mark.gpu
def test_batch_with_windows_that_do_not_fit(pkg, cases):
    """One such scenario sends its whole batch launch by launch."""
    out = []
    for timed in (True, False):
        scen = []
        for c in (_tank(cases, 200, 40), _splash(cases), _tank(cases, 12, 10)):
            c.params.update(precision=1, tol=1e-9, max_iter=12, max_outer=1)
            s = pkg.Scenario(c)
            s.init_state()
            s.prof_enable(timed)
            scen.append(s)
        print("windows: batch of n =", [s.n for s in scen], "timed", timed, flush=True)
        b = pkg.Batch(scen)
        b.step(1, check=False)
        out.append(([_stats(b.stats(q)) for q in range(3)], [s.download() for s in scen]))
        counts = [s.resident_counts() for s in scen]
        b.close()
        for s in scen:
            s.close()
    assert [k["too_wide"] for k in counts] == [0, 1, 0]
    assert not any(k["launches"] for k in counts)
    assert out[0][0] == out[1][0]
    for a, b in zip(out[0][1], out[1][1]):
        for k in a:
            assert np.array_equal(a[k], b[k], equal_nan=True), k
