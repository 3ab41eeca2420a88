"""The automatic tiling of a grid (rows and x-planes per workgroup) and of an
ensemble only moves work between workgroups: the states and dts of the
automatic choice equal those of fixed tilings bit for bit, on grids with one
plane, one row, ragged edges and more workgroups than the device holds; a grid
keeps its place on either side of dg_step_noalloc's limit."""
import ctypes

import numpy as np
import pytest

import cases
from test_kernel_emulation import emu_lib  # noqa: F401

BCS = [cases.OUTFLOW, cases.WALL, cases.PERIODIC, cases.PERIODIC, cases.WALL, cases.OUTFLOW]


def run(lib, interior, precision, math, tile_y=0, chunk_x=0, steps=2):
    import deepgreen
    w, ds = cases.smooth_random(interior, seed=6)
    sim = deepgreen.Simulation(*interior, ds, BCS, gamma=1.4, cfl=0.3, g=0.0, precision=precision, math=math,
                               tile_y=tile_y, chunk_x=chunk_x)
    with deepgreen.Solver(sim, lib=lib) as s:
        s.set_primitives(w)
        dts = [s.compute_step() for _ in range(steps)]
        return dts, np.stack([np.array(s.interior(a)) for a in s.get_state()])


def check(lib, interior, precision, math):
    dts, U = run(lib, interior, precision, math)
    for tile_y, chunk_x in ((4, interior[0]), (8, 3), (0, 2), (8, 0)):
        d, V = run(lib, interior, precision, math, tile_y, chunk_x)
        assert d == dts
        np.testing.assert_array_equal(V, U)


@pytest.mark.parametrize("interior,precision,math", [((5, 3, 6), "fp32", "exact"), ((3, 9, 65), "fp32", "fast"),
                                                     ((7, 2, 5), "fp64", "exact"), ((4, 5, 3), "fp64", "fast")])
def test_emulated_tiling_keeps_bits(emu_lib, interior, precision, math):  # noqa: F811
    check(emu_lib, interior, precision, math)


@pytest.mark.gpu
@pytest.mark.parametrize("precision,math", [("fp32", "exact"), ("fp32", "fast"), ("fp32_bulk", "exact"),
                                            ("fp64", "exact"), ("fp64", "fast")])
@pytest.mark.parametrize("interior", [(2, 2, 130), (30, 31, 63), (257, 2, 128), (2, 300, 257), (64, 64, 64),
                                      (97, 65, 129)])
def test_tiling_keeps_bits(interior, precision, math):
    print(f"  tiling {interior} {precision} {math}", flush=True)
    check(None, interior, precision, math)


def test_emulated_ensemble_chunks_keep_bits(emu_lib):  # noqa: F811
    """Chosen chunks, given ones and a mixture, over few and many slots."""
    import deepgreen
    edges = (19, 5, 9)
    states = [cases.smooth_random((n, n, n), seed=n) for n in edges]

    def advance(chunks, grid):
        sims = [deepgreen.Simulation(n, n, n, ds, BCS, gamma=1.4, cfl=0.3, g=0.0, math="fast", tile_y=4, chunk_x=c)
                for n, (_, ds), c in zip(edges, states, chunks)]
        with deepgreen.Ensemble(sims, lib=emu_lib, grid=grid) as e:
            for i, (w, _) in enumerate(states):
                e.set_state(i, w)
            e.run(2)
            return [e.get_state(i) for i in range(len(edges))]

    ref = advance((19, 5, 9), 2)
    for chunks, grid in (((0, 0, 0), 2), ((0, 0, 0), 40), ((0, 2, 0), 3)):
        for a, b in zip(advance(chunks, grid), ref):
            for f, g in zip(a, b):
                np.testing.assert_array_equal(f, g)


def test_noalloc_limit_is_where_it_was(emu_lib):  # noqa: F811
    """Refused from the configuration alone: 8-row tiles of these grids are
    more than the scratch array holds, although 16-row ones would fit."""
    import deepgreen
    p = (ctypes.c_void_p * 5)(*[1 << 20] * 5)
    q = (ctypes.c_void_p * 5)(*[1 << 21] * 5)
    for precision, math in (("fp32_bulk", "exact"), ("fp32", "fast"), ("fp64", "exact")):
        cfg = deepgreen.Simulation(2, 2080, 2048, 1.0 / 2048, [0] * 6, precision=precision, math=math).config(emu_lib)
        assert emu_lib.dg_step_noalloc(ctypes.byref(cfg), p, q, None, None) == -1
