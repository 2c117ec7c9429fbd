"""A resident solve that has to go on, or start over, launch by launch: the
results are those of the launch-per-phase form (kernel timing on), bit for bit,
whatever the iteration at which the resident form ends."""
import threading

import numpy as np
import pytest

from test_resident_gpu import _stats, _tank

# row blocks per workgroup: one, two, four, eight and twelve at most
SIZES = [(200, 40), (1280, 100), (1500, 170), (1640, 160), (3400, 160)]


def _step(pkg, c, before):
    s = pkg.Scenario(c)
    s.init_state()
    before(s)
    rc, st = s.step(1, check=False)
    out = rc, _stats(st), s.solution(), s.download(), s.resident_counts()
    s.close()
    return out


def _same(a, b):
    assert a[0] == b[0] and a[1] == b[1], (a[:2], b[:2])
    assert np.array_equal(a[2], b[2])
    for k in a[3]:
        assert np.array_equal(a[3][k], b[3][k]), k


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nx,ny", SIZES)
@pytest.mark.parametrize("launches", [0, 1, 3])
def test_launch_refused_in_the_middle_of_a_solve(pkg, cases, nx, ny, launches, precision):
    """The resident launches end after 0, 3 and 9 iterations; the state they
    leave is the one the next phase of the other form reads."""
    c = _tank(cases, nx, ny)
    c.params.update(precision=precision, tol=1e-10, max_iter=25, max_outer=2)
    print(f"resident: n={c.n}, precision {precision}, {launches} launches", flush=True)
    a = _step(pkg, c, lambda s: s.prof_enable(True))
    b = _step(pkg, c, lambda s: s.set_resident(launches, 3))
    assert b[4] == dict(launches=launches, too_wide=0, refused=1, ran_out=0)
    assert a[1][0] > 3 * launches
    _same(a, b)


def _over(pkg, cases, nx, ny, ended, precision):
    c = _tank(cases, nx, ny)
    c.params.update(precision=precision, tol=1e-10, max_iter=25, max_outer=2)
    c.parts["p"] = 100.0 * np.cos(7.0 * c.parts["x"])
    print(f"resident: n={c.n}, precision {precision}, {ended} workgroups give up", flush=True)
    a = _step(pkg, c, lambda s: s.prof_enable(True))
    b = _step(pkg, c, lambda s: s.set_resident(-1, 0, ended))
    assert b[4] == dict(launches=1, too_wide=0, refused=0, ran_out=1)
    _same(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nx,ny", SIZES)
def test_wait_that_runs_out_starts_the_solve_over(pkg, cases, nx, ny, precision):
    _over(pkg, cases, nx, ny, 1000, precision)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nx,ny,ended", [(200, 40, 1), (1500, 170, 3), (3400, 160, 100)])
def test_waits_for_workgroups_that_gave_up(pkg, cases, nx, ny, ended, precision):
    """The other workgroups wait for them to the end of their waits."""
    _over(pkg, cases, nx, ny, ended, precision)


@pytest.mark.gpu
@pytest.mark.parametrize("limits", [(1, 3, 0), (2, 8, 0), (-1, 0, 1000)])
def test_batch_leaves_the_resident_form(pkg, cases, limits):
    """Scenarios that have finished, that have not, and one at rest (finished
    before the first iteration), when the batch's launch is refused or a wait of
    one of them runs out."""
    sizes = [(12, 10), (200, 40), (330, 61), (660, 100), (900, 130)]
    out = []
    for timed in (True, False):
        scen = []
        for q, (nx, ny) in enumerate(sizes):
            c = _tank(cases, nx, ny)
            c.params.update(precision=1, tol=1e-9, max_iter=60)
            if q == 1:
                c.params.update(g=0.0)
                c.parts["u"][:] = 0.0
            s = pkg.Scenario(c)
            s.init_state()
            if timed:
                s.prof_enable(True)
            elif q == 3:
                s.set_resident(*limits)
            scen.append(s)
        print("resident batch: n =", [s.n for s in scen], "timed", timed, limits, flush=True)
        b = pkg.Batch(scen)
        b.step(1, check=False)
        stats = [_stats(b.stats(q)) for q in range(len(scen))]
        counts = [s.resident_counts() for s in scen]
        b.close()
        out.append((stats, [s.download() for s in scen]))
        for s in scen:
            s.close()
    if limits[2]:
        assert [k["ran_out"] for k in counts] == [0, 0, 0, 1, 0]
        assert all(k["launches"] == 1 for k in counts)
    else:
        assert all((k["launches"], k["refused"]) == (limits[0], 1) for k in counts)
    assert out[0][0] == out[1][0]
    for a, b in zip(out[0][1], out[1][1]):
        for k in a:
            assert np.array_equal(a[k], b[k], equal_nan=True), k


@pytest.mark.gpu
def test_contexts_stepped_by_several_threads(pkg, cases):
    """Resident launches of three threads' contexts, in either form and of
    different shapes, at once: each gets the results that it has alone."""
    shapes = [(200, 40, 1), (330, 61, 0), (1280, 100, 1)]

    def make(nx, ny, precision):
        c = _tank(cases, nx, ny)
        c.params.update(precision=precision, tol=1e-9, max_iter=80, max_outer=2)
        s = pkg.Scenario(c)
        s.init_state()
        return s

    def run(s, out):
        st = [_stats(s.step(1, check=False)[1]) for _ in range(6)]
        out.append((st, s.solution(), s.resident_counts()))
        s.close()

    alone = []
    for q in shapes:
        run(make(*q), alone)
    print("resident: three threads", flush=True)
    scen, together = [make(*q) for q in shapes], [[] for _ in shapes]
    th = [threading.Thread(target=run, args=a) for a in zip(scen, together)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for a, (b,) in zip(alone, together):
        assert a[0] == b[0] and np.array_equal(a[1], b[1])
        assert b[2]["launches"] + b[2]["refused"] >= 1
