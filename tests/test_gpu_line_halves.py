"""Vertical-line solve at the edges of its two eliminations: from both ends of a column (up to
512 tiles of 64 columns) and from the bottom up (more), with columns of one, two, even and odd
numbers of levels, windows that end inside a half, and partial tiles; every window and with
and without LDS staging, against the oracle's line solve."""
import numpy as np
import pytest

from asam_amd import workload as W
from test_gpu_parity import OP_TOL, live, rel, small

pytestmark = pytest.mark.gpu

GRIDS = [(1, 1, 1), (3, 2, 2), (65, 3, 3), (64, 4, 9), (70, 5, 17), (33, 2, 64),
         (64, 512, 7), (64, 513, 7)]


@pytest.mark.parametrize("np1", [1, 2])
@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: "x".join(map(str, g)))
def test_line_solve_edges(grid, np1, oracle_mod, sound_mod):
    nx, ny, nz = grid
    p = small(np1=np1, nx=nx, ny=ny, nz=nz)
    orc = oracle_mod.Oracle(p)
    s = sound_mod.SoundSolver.from_problem(p)
    x = live(p, W.normal(p.n, 7))
    want = {"PSolve1": orc.psolve1(x), "PSolve1_T": orc.psolve1_T(x)}
    t0 = s.get_tuning()
    for kw in ({}, {"line_window": 1}, {"line_window": 4, "line_lds": 0}, {"line_window": 8},
               {"line_tiled": 0}):
        s.set_tuning(**{**t0, **kw})
        for name, o in want.items():
            g = getattr(s, name)(x)
            assert rel(g, o) < OP_TOL, (name, kw, rel(g, o))
