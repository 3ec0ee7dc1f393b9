"""A negative local tolerance: no local solve ends before its bound, so every row
counts as diverged, as in the oracle; the solve is aborted (EXIT) or goes on from the
last iterates (CALLBACK)."""
import numpy as np
import pytest

import oracle
import solfec
from test_gpu_local_newton import _rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["stick", "slide"])
@pytest.mark.parametrize("diageps", [-1e-9, -1.0, -1e-200])
@pytest.mark.parametrize("failure", [1, 2])
def test_negative_tolerance_never_ends(kind, diageps, failure):
    print(f"[local] {kind} diagepsilon={diageps} failure={failure}", flush=True)
    O, R0, U0 = _rows(kind, 70, 3)
    kw = dict(diagepsilon=diageps, diagmaxiter=15, failure=failure)
    dev = solfec.Device(0)
    try:
        dev.system(O["rowptr"], O["col"], O["W"], O["Wd"], O["A"], O["B"], O["V"], O["rho"], O["mu"], O["rest"],
                   O["coh"], O["gap"], O["free_energy"], O["step"], R0, U0)
        rep, _, _ = dev.solve(solfec.make_param(1e-6, 5, **kw))
        R, _ = dev.get_RU()
    finally:
        dev.close()
    _, orep, Ro, _, _, _ = oracle.gs_solve(oracle.System(O), oracle.gs_param(1e-6, 5, **kw),
                                           np.arange(O["n"], dtype=np.int32), R0, U0)
    assert orep.error == 2   # a local solve reached its bound
    assert rep.error == orep.error and rep.aborted == (failure == 1)
    if failure == 2:
        # decoupled rows, 15 iterations of a solve that converges in about five: both are at
        # the solution to the rounding of a 3x3 system, and the second sweep changes nothing
        assert rep.iters == orep.iters
        assert np.abs(R - Ro).max() <= 1e-9 * np.abs(Ro).max()
