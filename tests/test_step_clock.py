"""The run clock and the dt over single steps, runs bounded by steps and runs
bounded by time, in any order: the same states and dts as single steps, one
count of steps, and a step that a non-finite dt forbids leaves everything as
it was."""
import ctypes

import numpy as np
import pytest

import cases
from test_kernel_emulation import emu_lib  # noqa: F401

BCS = [cases.PERIODIC, cases.PERIODIC, cases.WALL, cases.OUTFLOW, cases.OUTFLOW, cases.WALL]


def solver(lib, interior, precision, **kw):
    import deepgreen
    w, ds = cases.smooth_random(interior, seed=8)
    s = deepgreen.Solver(deepgreen.Simulation(*interior, ds, BCS, gamma=1.4, cfl=0.3, g=0.0, precision=precision, **kw),
                         lib=lib)
    s.set_primitives(w)
    return s


def check(lib, interior, precision, math):
    with solver(lib, interior, precision, math=math) as a, solver(lib, interior, precision, math=math) as b:
        dts = [a.compute_step() for _ in range(25)]
        assert b.compute_step() == dts[0]
        assert b.next_dt() == dts[1]
        t, n = b.run(18)                      # a captured stretch and the rest
        assert n == 19 and b.next_dt() == dts[19]
        assert b.run(0)[1] == 19
        assert b.compute_step() == dts[19]    # a finished run does not hold the step back
        t, n = b.run(2 ** 63 - 1, t_end=t)    # nothing to do: the clock is past the end
        assert n == 20
        t, n = b.run(2 ** 63 - 1, t_end=float(np.sum(dts[:23])))
        assert n in (23, 24) and t >= np.sum(dts[:23]) * (1 - 1e-5)
        for k in range(n, 25):
            assert b.compute_step() == dts[k]
        for f, g in zip(a.get_state(), b.get_state()):
            np.testing.assert_array_equal(a.interior(f), b.interior(g))
        b.reset_clock()
        assert b.run(1)[1] == 1


def check_nonfinite(lib, precision):
    with solver(lib, (4, 3, 5), precision, dt_nan_fallback=False) as s:
        U = s.get_state()
        U[4][3, 3, 3] = np.nan
        s.set_conserved(U)
        before = [np.array(s.interior(a)) for a in s.get_state()]
        dt = ctypes.c_double(-3.0)
        assert s._L.dg_step(s._h, ctypes.byref(dt)) == -4
        assert dt.value == -3.0
        for f, g in zip(before, s.get_state()):
            np.testing.assert_array_equal(f, s.interior(g))


@pytest.mark.parametrize("precision,math", [("fp32", "exact"), ("fp64", "fast")])
def test_emulated_clock(emu_lib, precision, math):  # noqa: F811
    check(emu_lib, (4, 5, 3), precision, math)


def test_emulated_nonfinite_dt_forbids_the_step(emu_lib):  # noqa: F811
    check_nonfinite(emu_lib, "fp32")


@pytest.mark.gpu
@pytest.mark.parametrize("precision,math", [("fp32", "exact"), ("fp32", "fast"), ("fp32_bulk", "exact"),
                                            ("fp64", "exact"), ("fp64", "fast")])
@pytest.mark.parametrize("interior", [(4, 5, 3), (40, 33, 70)])
def test_clock(interior, precision, math):
    print(f"  clock {interior} {precision} {math}", flush=True)
    check(None, interior, precision, math)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_nonfinite_dt_forbids_the_step(precision):
    check_nonfinite(None, precision)
