"""Device memory of a transport context on x-z and y-z slices, and the sweeps on the row widths of
the layout that bounds it, bit for bit against the oracle.  Words per cell by the layout, for X
much larger than Y, which is one tile: natural arrays 16 + nc^2 + 9 nc, skewed arrays 18 + 2 nc
with the places that groups of two add, and the boundary records 2 per component with blocks of
three levels; together 1.6 to 1.8 times the natural arrays as counted here (ten vectors)."""
import ctypes as C

import numpy as np
import pytest

from asam_amd import workload as W
from test_gpu_transport_sweeps import check, problem, vector

pytestmark = pytest.mark.gpu


def free_bytes():
    hip = C.CDLL("libamdhip64.so")
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


# (3, 30000, 20): 6.4 GB of skewed arrays with tiles of 53 columns, so tiles of X + Z = 27, rows of
# 32 entries: 31 rows for 5 cells make 7 times the natural arrays
# (40000, 48, 100): 84 GB with rows of 64 entries for 28 columns, so rows of 32: 1.9 times
@pytest.mark.parametrize("shape,ncomp,times", [((20000, 1, 100), 1, 2.0), ((20000, 1, 60), 4, 2.0),
                                               ((15000, 3, 100), 2, 2.0), ((3, 30000, 20), 1, 9.0),
                                               ((40000, 48, 100), 1, 2.2)])
def test_context_memory(shape, ncomp, times, sound_mod):
    from asam_amd import transport
    warm = transport.TransportSolver(3, 3, 3, 1)
    nx, ny, nz = shape
    m = (nx + 2) * (ny + 2) * (nz + 2)
    natural = 8 * ((16 + 10 * ncomp) * m + ncomp ** 2 * nx * ny * nz)
    before = free_bytes()
    s = transport.TransportSolver(nx, ny, nz, ncomp)
    used = before - free_bytes()
    print(f"{shape} {ncomp} components: {used / 1e6:.0f} MB, natural arrays {natural / 1e6:.0f} MB")
    assert used < times * natural


# rows of 3 to 20 entries and of 64, one tile and two
@pytest.mark.parametrize("ny", [1, 2, 5, 6, 7, 8, 18, 24, 25, 46, 47])
@pytest.mark.parametrize("ncomp,iterg", [(2, 5), (6, 7)])
def test_row_widths(ny, ncomp, iterg, oracle_mod, sound_mod):
    # 6 components of 126 levels go in pairs (more than 256 blocks)
    tp = problem(31, ny, 126 if ncomp == 6 else 9, ncomp=ncomp, mom_comps=(1,), iterg=iterg)
    check(tp, vector(tp))


def test_few_cells_in_x(oracle_mod, sound_mod):
    tp = problem(3, 30000, 20, ncomp=1)
    check(tp, vector(tp))
