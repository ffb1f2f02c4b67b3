"""The pipelined Gauss-Seidel sweeps of the transport preconditioner at the sizes where their
blocking can go wrong, against the oracle (oracle/transport.c).  Both do the same products,
sums and correctly rounded quotients in the same order, so the values are equal:
  - y-extents on either side of a tile edge (a tile holds 53 columns, the sweeps shift by one
    column each), x shorter than a tile, single cells, remainders of the level blocks;
  - more sweeps than one launch runs;
  - components in pairs (chosen above 256 blocks), a component left over, and the three
    operator kinds among them;
  - diagonals that rule out the reciprocal form of the quotient, and quotients that leave the
    normal range."""
import numpy as np
import pytest

from asam_amd import workload as W

pytestmark = pytest.mark.gpu


def problem(nx, ny, nz, **kw):
    p = W.make_problem(nx, ny, nz, 500.0, 500.0, 100.0, H=700.0, a=1200.0,
                       ridge_xc=0.5 * nx * 500.0, np1=1, seed=5)
    return W.transport_problem(p, chem=False, **kw)


def check(tp, x, **tune):
    from asam_amd import transport
    from oracle import pytransport
    s = transport.TransportSolver.from_problem(tp)
    if tune:
        s.set_tuning(**tune)
    y, yo = s.PSolve(x), pytransport.TransportOracle(tp).psolve(x)
    bad = ~((y == yo) | (np.isnan(y) & np.isnan(yo)))
    print(f"{(tp.nx, tp.ny, tp.nz)} {tune}: {int(bad.sum())} of {bad.size} differ")
    assert not bad.any()
    assert np.array_equal(s.PSolve(x), y, equal_nan=True)  # nothing is left from a call


def vector(tp, seed=61):
    return W.normal(tp.ncomp * tp.m, seed).reshape(tp.ncomp, tp.m)


# Y = ny + 2 columns and five shifts: 53 and 54, 106 and 107 columns are one tile or two
@pytest.mark.parametrize("shape", [(7, 46, 5), (7, 47, 5), (3, 99, 4), (3, 100, 4), (1, 1, 1),
                                   (70, 1, 3), (1, 60, 126), (66, 5, 1)])
@pytest.mark.parametrize("rows", [1, 2, 3, 8])
def test_tile_edges(shape, rows, oracle_mod, sound_mod):
    tp = problem(*shape, ncomp=2, fall_comp=1)
    check(tp, vector(tp), gs_rows=rows)


@pytest.mark.parametrize("iterg", [4, 6, 11, 13])
def test_more_sweeps_than_a_launch(iterg, oracle_mod, sound_mod):
    tp = problem(9, 50, 8, ncomp=2, mom_comps=(1,), iterg=iterg)
    check(tp, vector(tp))


# 126 levels and 60 columns: 2 tiles x 44 or 66 level blocks per component
@pytest.mark.parametrize("kinds", [dict(ncomp=4), dict(ncomp=5), dict(ncomp=5, mom_comps=(0, 3)),
                                   dict(ncomp=6, mom_comps=(1,), fall_comp=4)])
@pytest.mark.parametrize("rows", [1, 2, 8])
@pytest.mark.parametrize("iterg", [5, 7])
def test_paired_components(kinds, rows, iterg, oracle_mod, sound_mod):
    tp = problem(4, 60, 126, iterg=iterg, **kinds)
    check(tp, vector(tp), gs_rows=rows)


@pytest.mark.parametrize("ncomp", [1, 4])
@pytest.mark.parametrize("scale", [2.0 ** 600, 2.0 ** -600])
def test_unusual_diagonals(ncomp, scale, oracle_mod, sound_mod):
    tp = problem(6, 50, 126, ncomp=ncomp)
    tp.tpot[:, ::3] *= scale  # whole columns of the matrix: the couplings stay below the diagonal
    check(tp, vector(tp))


@pytest.mark.parametrize("ncomp", [1, 4])
@pytest.mark.parametrize("value", [1e-310, 1e308, np.inf, np.nan])
def test_unusual_values(ncomp, value, oracle_mod, sound_mod):
    tp = problem(6, 50, 126, ncomp=ncomp)
    x = vector(tp)
    tp.interior(x)[:, ::5, 3, 2] = value
    tp.interior(x)[:, :, 20, :] = -0.0
    check(tp, x)
