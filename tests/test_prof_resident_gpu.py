"""The timer of the resident launches leaves the solves as they are."""
import numpy as np
import pytest

from test_resident_gpu import _stats, _tank


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
def test_resident_timer(pkg, cases, precision):
    c = _tank(cases, 200, 40)
    c.params.update(precision=precision, tol=1e-8, max_iter=60, max_outer=2)
    out = []
    for on in (0, 2):
        s = pkg.Scenario(c)
        s.init_state()
        s.prof_enable(on)
        st = [_stats(s.step(1, check=False)[1]) for _ in range(2)]
        ms, launches = s.prof_read("resident")
        assert launches == (s.resident_counts()["launches"] if on else 0)
        assert s.resident_counts()["launches"] >= 2 and (ms > 0.0) == (on == 2)
        out.append((st, s.solution()))
        s.close()
    assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])
