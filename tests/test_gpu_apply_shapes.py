"""Stencil apply with the tile its size rule chooses: widths around the edges of 32, 64, 128 and
256 columns, row counts that leave a tile's last rows empty, and level counts that the planes
per tile do not divide, against the oracle's operator; and, for the shapes of the FP32 applies,
a mixed solve checked with the oracle's operator."""
import numpy as np
import pytest

from asam_amd import workload as W
from test_gpu_parity import OP_TOL, live, rel, small

pytestmark = pytest.mark.gpu

GRIDS = [(33, 17, 5), (64, 8, 3), (65, 31, 13), (130, 97, 6), (201, 33, 11), (257, 18, 4),
         (300, 7, 50)]


@pytest.mark.parametrize("np1", [1, 2])
@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: "x".join(map(str, g)))
def test_apply_edges(grid, np1, oracle_mod, sound_mod):
    nx, ny, nz = grid
    p = small(np1=np1, nx=nx, ny=ny, nz=nz)
    orc = oracle_mod.Oracle(p)
    s = sound_mod.SoundSolver.from_problem(p)
    x = live(p, W.normal(p.n, 5))
    for name, o in (("MatVec1", orc.matvec1(x)), ("MatVec1_T", orc.matvec1_T(x))):
        g = getattr(s, name)(x)
        assert rel(g, o) < OP_TOL, (name, rel(g, o))
    s.set_control(method="BICGSTAB", precision="MIXED")
    b = live(p, p.b)
    x, mi, tl, info = s.SolveSound(np.zeros(p.n), b, 300, 1e-8)
    rr = rel(orc.matvec1(x), b)
    print(f"{grid} np1 {np1}: status {info.status}, relative residual {rr:.2e}")
    assert info.status == 0 and rr <= 1.0001e-8
