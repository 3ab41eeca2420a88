"""Exact math at the edges of its shared divisions and skipped wave speeds:
states that span the number range (signed zeros, denormal and huge
velocities, densities and pressures many binades apart, negative face states)
must give the oracle's values exactly, NaN for NaN, with cell sizes that are
powers of two (products) and that are not (quotients by constants)."""
import numpy as np
import pytest

import cases
from test_kernel_emulation import emu_lib, run_both  # noqa: F401

# (precision, largest binade of densities, of pressures, of velocities): FP32 stays in range
# through the squares; FP64 passes both ends of the short division's ranges (2^+-100, 2^+-300)
SPANS = [("fp32", 20, 30, 30), ("fp32", 55, 60, 30), ("fp64", 20, 30, 30), ("fp64", 130, 340, 330)]


def wild_state(interior, seed, span_r, span_p, span_v, dtype):
    rng = np.random.default_rng(seed)
    shape = tuple(n + 4 for n in interior)

    def binades(span):
        return rng.uniform(1.0, 2.0, shape) * np.exp2(rng.integers(-span, span + 1, shape))

    # slabs of calm gas between the wild cells, so that short and plain divisions meet in one wave
    calm = (np.arange(shape[2]) // 3 % 2 == 0)[None, None, :]
    rho = np.where(calm, rng.uniform(0.9, 1.1, shape), binades(span_r))
    p = np.where(calm, rng.uniform(0.9, 1.1, shape), binades(span_p))
    v = []
    for _ in range(3):
        a = binades(span_v) * rng.choice([-1.0, 1.0], shape)
        tiny = np.finfo(dtype).tiny * rng.uniform(-1.0, 1.0, shape)   # denormals
        pick = rng.integers(0, 5, shape)
        a = np.choose(pick, [a, np.zeros(shape), -np.zeros(shape), tiny, rng.uniform(-0.1, 0.1, shape)])
        v.append(np.where(calm & (pick == 0), 0.05, a))
    return [a.astype(dtype) for a in (rho, *v, p)]


def check(lib, precision, spans, ds, limiter, seed, interior, tile_y):
    dtype = np.float64 if precision == "fp64" else np.float32
    w = wild_state(interior, seed, *spans, dtype)
    bcs = [cases.PERIODIC, cases.PERIODIC, cases.WALL, cases.OUTFLOW, cases.PERIODIC, cases.PERIODIC]
    with np.errstate(all="ignore"):
        U, dts, Uo, dto = run_both(lib, interior, w, ds, bcs, 2, precision, limiter=limiter, tile_y=tile_y)
    np.testing.assert_array_equal(dts, dto.astype(np.float64))
    np.testing.assert_array_equal(U, Uo)


@pytest.mark.parametrize("ds", [1.0 / 64, 0.005])
@pytest.mark.parametrize("precision,span_r,span_p,span_v", SPANS)
def test_emulated_wild_states(emu_lib, precision, span_r, span_p, span_v, ds):  # noqa: F811
    check(emu_lib, precision, (span_r, span_p, span_v), ds, "none", 3, (5, 6, 20), 4)


@pytest.mark.gpu
@pytest.mark.parametrize("ds,limiter,tile_y", [(1.0 / 64, "none", 4), (0.005, "minmod", 8), (3.0, "none", 0),
                                               (0.1, "vanleer", 0)])
@pytest.mark.parametrize("precision,span_r,span_p,span_v", SPANS)
def test_wild_states(precision, span_r, span_p, span_v, ds, limiter, tile_y):
    print(f"  wild states {precision} {span_r} {span_p} {span_v} ds {ds} {limiter} tile {tile_y}", flush=True)
    check(None, precision, (span_r, span_p, span_v), ds, limiter, 11, (12, 21, 70), tile_y)
