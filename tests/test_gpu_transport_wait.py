"""A solve whose sweeps give up waiting (forced from the host: no block publishes its boundary, 64
polls) says so, at the first sum after the sweeps, on host arrays and on device vectors; the same
context then solves as before."""
import numpy as np
import pytest

from test_gpu_transport_sweeps import problem

pytestmark = pytest.mark.gpu


def test_solve_reports_a_wait(oracle_mod, sound_mod):
    from asam_amd import sound, transport
    tp = problem(20, 30, 9, ncomp=2)
    s = transport.TransportSolver.from_problem(tp)
    want, mi, tol, _ = s.BiCGStab(np.zeros_like(tp.b), tp.b, 30, 1e-8)
    db, dx = s.device_vector().upload(tp.b), s.device_vector().upload(np.zeros_like(tp.b))
    s.set_tuning(gs_spin_limit=64)
    s.test_hold_boundary(True)
    with pytest.raises(sound.AsamError, match="waited past its limit"):
        s.BiCGStab(np.zeros_like(tp.b), tp.b, 30, 1e-8)
    with pytest.raises(sound.AsamError, match="waited past its limit"):
        s.solve_device(dx, db, 30, 1e-8)
    s.test_hold_boundary(False)
    s.set_tuning(gs_spin_limit=0)
    x, mi2, tol2, info = s.BiCGStab(np.zeros_like(tp.b), tp.b, 30, 1e-8)
    assert info.status == 0 and (mi2, tol2) == (mi, tol) and np.array_equal(x, want)
    dx.upload(np.zeros_like(tp.b))
    s.solve_device(dx, db, 30, 1e-8)
    assert np.array_equal(dx.download(), want.ravel())
    for v in (dx, db):
        v.free()
