"""Modified Gram-Schmidt taken several basis vectors a pass: restart lengths that end a step's
passes in blocks of one, two and three vectors, on vectors whose length is not a multiple of a
16-byte pack (so some of them are not aligned to one either), against the oracle's method:
the same number of iterations (+-1) and the solution to the FP64 solve bar."""
import numpy as np
import pytest

from test_gpu_parity import SOL_TOL, rel, small

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method", ["FGMRES", "GMRES"])
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 6, 7, 11])
def test_restart_lengths_odd_vectors(method, m, oracle_mod, sound_mod):
    p = small(np1=1, nx=33, ny=7, nz=9)
    assert p.n % 2 == 1
    orc = oracle_mod.Oracle(p)
    f = {"FGMRES": orc.fgmres, "GMRES": orc.gmres}[method]
    s = sound_mod.SoundSolver.from_problem(p)
    s.set_control(method=method, step_gmres=m)
    xo = f(p.b, 400, 1e-12, m)[0]
    x, mi, tl, info = s.SolveSound(np.zeros(p.n), p.b, 400, 1e-12)
    print(f"{method} m={m}: iterations {info.iterations}, error {rel(x, xo):.2e}")
    assert info.status == 0
    assert rel(x, xo) < SOL_TOL
