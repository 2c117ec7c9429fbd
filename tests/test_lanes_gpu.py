"""Eight lanes per particle against one lane, bit for bit: a scenario stepped
alone chooses the form of each neighbour sum by its size, the batched phases
run one lane always.  The sizes leave the last group, wavefront and workgroup
of eight-lane particles in every state of filling, and lie on both sides of the
sizes up to which the kernels take eight lanes."""
import numpy as np
import pytest

FIELDS = ("x", "y", "u", "v", "p", "c", "rho", "rho0", "m", "vol0", "tid", "flags")


def _flume(cases, n):
    d = (6.0 * 0.3 / n) ** 0.5
    c = cases.porous_flume(dx=d, length=6.0, depth=0.3, tank_h=0.45, toe=3.0, slope=0.1,
                           porosity=0.4, d50=0.01, dt=0.02 * d)
    rng = np.random.default_rng(n)
    fl = c.parts["tid"] == 3
    for f in ("x", "y"):
        c.parts[f][fl] += rng.uniform(-0.05 * d, 0.05 * d, fl.sum())
    c.parts["u"][fl] = 0.02 * np.sin(c.parts["x"][fl] * 9.0)
    return c


@pytest.mark.gpu
@pytest.mark.parametrize("n", [700, 1511, 2900, 3333, 5000, 7777, 97000, 99000, 107000, 253000,
                               256000])
def test_alone_equals_batch(pkg, cases, n):
    steps = 2
    make = [lambda: _flume(cases, n), lambda: cases.tiny_box(nx=9, ny=7)]
    got = []
    for batched in (False, True):
        scen = []
        for k in make:
            c = k()
            c.params.update(precision=1, tol=1e-8, max_iter=40, max_outer=1)
            s = pkg.Scenario(c)
            s.init_state()
            scen.append(s)
        if not batched:
            print(f"lanes: n={scen[0].n}, {scen[1].n}", flush=True)
        b = pkg.Batch(scen) if batched else None
        its = []
        for _ in range(steps):
            if batched:
                b.step(1, check=False)
                its.append([b.stats(q).iterations for q in range(len(scen))])
            else:
                its.append([s.step(1, check=False)[1].iterations for s in scen])
        if batched:
            b.close()
        got.append((its, [s.download() for s in scen]))
        for s in scen:
            s.close()
    (ia, alone), (ib, batch) = got
    assert ia == ib
    for q in range(len(make)):
        for f in FIELDS:
            assert np.array_equal(alone[q][f], batch[q][f]), (q, f)
