"""The quotients of the Gauss-Seidel sweeps where a product of quotient and diagonal, or its
remainder, leaves the normal range, against the oracle: both round every quotient correctly, so
the values are equal.  Diagonals far below one beside right-hand sides near the smallest normal
number, and right-hand sides on both sides of where the sweeps change to dividing."""
import pytest

from test_gpu_transport_sweeps import check, problem, vector

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncomp", [1, 6])  # one component, and pairs, per group
@pytest.mark.parametrize("scale,value", [
    (2.0 ** -100, 1e-307), (2.0 ** -61, 1e-305), (2.0 ** -57, 1e-306), (2.0 ** -57, 2.0 ** -957),
    (1.0, 1e-307), (1.0, 2.0 ** -900), (1.0, 2.0 ** -960), (2.0 ** 400, 2.0 ** -500),
    (2.0 ** 400, 1e-300)])
def test_small_quotients(ncomp, scale, value, oracle_mod, sound_mod):
    tp = problem(9, 40, 126, ncomp=ncomp)
    tp.tpot *= scale
    check(tp, vector(tp) * value)
