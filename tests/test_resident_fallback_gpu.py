"""A resident solve that has to go on, or start over, launch by launch: the
results are those of the launch-per-phase form (kernel timing on), bit for bit,
whatever the iteration at which the resident form ends."""
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
    assert b[4] == dict(launches=launches, too_wide=0, refused=1)
    assert a[1][0] > 3 * launches
    _same(a, b)
