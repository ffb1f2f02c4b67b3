"""Modified Gram-Schmidt several basis vectors a pass: it takes the steps of the reference's
vector-at-a-time form (an error that the solve would make up for with more of them shows), with
the remainders that 16-byte packs leave (2 doubles, 4 floats), and with vectors of less than one
and of several turns of the passes' loops."""
import numpy as np
import pytest

from test_gpu_parity import SOL_TOL, rel, small

pytestmark = pytest.mark.gpu

# 2079, 1617, 1386 and 538059 cells: 3, 1, 2 and 3 modulo 4
SHAPES = [(33, 7, 9), (33, 7, 7), (33, 7, 6), (129, 97, 43)]


@pytest.mark.parametrize("method", ["FGMRES", "GMRES"])
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 6, 7, 11])
@pytest.mark.parametrize("shape", SHAPES[:2])
def test_fp64_steps(shape, m, method, oracle_mod, sound_mod):
    p = small(np1=1, nx=shape[0], ny=shape[1], nz=shape[2])
    orc = oracle_mod.Oracle(p)
    xo, ito, _ = (orc.fgmres if method == "FGMRES" else orc.gmres)(p.b, 400, 1e-8, m)
    s = sound_mod.SoundSolver.from_problem(p)
    s.set_control(method=method, step_gmres=m)
    x, _, _, info = s.SolveSound(np.zeros(p.n), p.b, 400, 1e-8)
    print(f"{shape} {method} m={m}: steps {info.iterations} (oracle {ito}), {rel(x, xo):.2e}")
    assert info.status == 0 and abs(info.iterations - ito) <= 1
    assert rel(x, xo) < SOL_TOL


# cycles of 6 and of 7 or 8 steps: the passes end with two vectors, with three and with one
@pytest.mark.parametrize("m,inner", [(7, 1e-5), (10, 1e-5), (11, 1e-6)])
@pytest.mark.parametrize("shape", SHAPES)
def test_mixed_steps(shape, m, inner, oracle_mod, sound_mod):
    """The same refinement with the oracle's FP64 cycles in place of the FP32 ones takes as many
    steps, but for one a cycle where a residual lies close to its tolerance."""
    p = small(np1=1, nx=shape[0], ny=shape[1], nz=shape[2])
    orc = oracle_mod.Oracle(p)
    tol = 1e-8
    x, r0, steps, cycles = np.zeros(p.n), None, 0, 0
    while cycles < 12:
        r = p.b - orc.matvec1(x)
        rn = np.linalg.norm(r)
        r0 = rn if r0 is None else r0
        if rn <= tol * r0:
            break
        d, it, _ = orc.fgmres(r, 1, min(max(inner, 0.5 * tol * r0 / rn), 0.5), m)
        x, steps, cycles = x + d, steps + it, cycles + 1
    s = sound_mod.SoundSolver.from_problem(p)
    s.set_control(method="FGMRES", step_gmres=m, precision="MIXED", inner_tol=inner)
    xg, _, _, info = s.SolveSound(np.zeros(p.n), p.b, 20, tol)
    rr = rel(orc.matvec1(xg), p.b)
    print(f"{shape} m={m}: steps {info.iterations} in {info.restarts} cycles (FP64 cycles: {steps} "
          f"in {cycles}), relative residual {rr:.2e}")
    assert info.status == 0 and rr <= 1.0001 * tol
    assert abs(info.iterations - steps) <= cycles
