"""The resident form of the allocation-free FP64 solve against its
launch-per-phase form (no resident launches allowed), bit for bit: at the edges
of its launch shapes and of its scratch block, where its launches are refused
half way, and where its waits run out."""
import ctypes

import numpy as np
import pytest

from test_zz_no_alloc import DeviceArrays

# (rows, whether the scratch block has room for the resident form): the last
# and first size of each launch shape, then both sides of the block's limit
SIZES = [(300, True), (65536, True), (65537, True), (131072, True), (131073, True),
         (262144, True), (262145, True), (266240, True), (266752, False), (900, True)]


def _system(pkg, n):
    """Rows of 3 to 13 entries within 700 rows of the diagonal, not symmetric."""
    rng = np.random.default_rng(n)
    off = np.array([0, -1, 1, -2, 2, -3, -5, 9, -64, 130, -350, 700, -699])
    i = np.arange(n)
    ln = rng.integers(3, len(off) + 1, n).astype(np.int32)
    ln = np.maximum.reduceat(ln, np.arange(0, n, 3)).repeat(3)[:n]  # some alike in a row
    cs = np.zeros((pkg.ROW_CAP, n + 3), np.int32)
    vs = np.zeros((pkg.ROW_CAP, n + 3))
    for k, o in enumerate(off):
        j = np.clip(i + o, 0, n - 1)
        cs[k, :n] = j
        vs[k, :n] = 1.0 if o == 0 else rng.uniform(-0.11, 0.02, n)
    rhs = np.sin(0.01 * i) + rng.uniform(-0.1, 0.1, n)
    return ln, cs, vs, rhs, 0.3 * np.cos(0.02 * i)


@pytest.mark.gpu
def test_noalloc_forms_agree(pkg):
    for n, fits in SIZES:  # in one test: each call finds what the one before left
        ln, cs, vs, rhs, x0 = _system(pkg, n)
        dv = DeviceArrays()
        arrays = [dv.put(a) for a in (ln, cs, vs, rhs)]
        out = {}
        for name, limits in (("launches", (0, 0, 0)), ("resident", (-1, 0, 0)),
                             ("refused", (2, 2, 0)), ("waits", (-1, 0, 1000))):
            print(f"noalloc: n={n}, {name}", flush=True)
            d_x = dv.put(x0)
            counts = {}
            rc, st = pkg.ppe_solve_noalloc(n, n + 3, *arrays, d_x, 1e-12, 30, 2, check=False,
                                           limits=limits, counts=counts)
            out[name] = (rc, st.iterations, st.outer, st.converged, st.breakdown,
                         st.rel_residual, st.bnorm), dv.get(d_x, x0), counts
        dv.free()
        assert out["launches"][0][0] in (0, -5) and out["launches"][0][1] > 4
        want = dict(resident=(1, 0, 0), refused=(2, 1, 0), waits=(1, 0, 1))
        for name, k in want.items():
            c = out[name][2]
            got = c["launches"], c["refused"], c["ran_out"]
            assert got == (k if fits else (0, 0, 0)), (n, name, c)
            assert out[name][0] == out["launches"][0], (n, name)
            assert np.array_equal(out[name][1], out["launches"][1]), (n, name)


@pytest.mark.gpu
def test_noalloc_takes_no_device_memory(pkg):
    """Each launch shape's first resident launch apart, at which the runtime sets
    up what it keeps; without resident launches, the first call apart."""
    dv = DeviceArrays()

    def free():
        f, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert dv.hip.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value

    for limits in ((0, 0, 0), (-1, 0, 0)):
        for n in (3000, 65537, 131073, 262145):
            ln, cs, vs, rhs, x0 = _system(pkg, n)
            args = [dv.put(a) for a in (ln, cs, vs, rhs)]
            xs = [dv.put(x0) for _ in range(3)]
            taken = []
            for d_x in xs:
                before = free()
                counts = {}
                print(f"noalloc: n={n}, limits {limits}", flush=True)
                pkg.ppe_solve_noalloc(n, n + 3, *args, d_x, 1e-12, 30, 2, check=False,
                                      limits=limits, counts=counts)
                taken.append(before - free())
                assert counts["launches"] == (1 if limits[0] else 0)
            assert taken[1:] == [0, 0], (n, limits, taken)
            assert limits[0] or n == 3000 or taken[0] == 0, (n, taken)
    dv.free()
