"""The flexible GMRES cycles of the Newton solver against the oracle: one Arnoldi
step a cycle, fewer than a cycle holds, all 20 of one and a restart after it (the
residual rebuilt from the Krylov vectors), from systems of a few rows to several
workgroups of a dot product.  The tolerances are those of the Newton parity test
over as many steps: 1e-8 of max|R| for sums that differ in order."""
import numpy as np
import pytest

import oracle
import solfec
from scenes import lattice

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [8, 216, 1000])
@pytest.mark.parametrize("linmaxiter,epsilon", [(1, 0.25), (3, 1e-3), (20, 1e-12), (23, 1e-12)])
def test_cycles_match_oracle(n, linmaxiter, epsilon):
    print(f"[newton] cycles n={n} linmaxiter={linmaxiter}", flush=True)
    s = lattice(n, seed=3)
    b, c = s.bodies(), s.contacts()
    O = oracle.assemble(oracle.bodies_from(b), oracle.contacts_from(c), 1e-3)
    R0 = np.random.default_rng(n).normal(scale=1e-2, size=3 * O["n"])
    kw = dict(linver="GMRES", maxiter=2, meritval=1e-30, gsflag="OFF", linmaxiter=linmaxiter, epsilon=epsilon)
    dev = solfec.Device(0)
    try:
        dev.system(O["rowptr"], O["col"], O["W"], O["Wd"], O["A"], O["B"], O["V"], O["rho"], O["mu"], O["rest"],
                   O["coh"], O["gap"], O["free_energy"], O["step"], R0, np.zeros(3 * O["n"]))
        rep, mer, mv = dev.newton(solfec.newton_param(**kw))
        R, _ = dev.get_RU()
    finally:
        dev.close()
    orep, Ro, _, omer, omv = oracle.newton_solve(oracle.System(O), oracle.nt_param(**kw), R0)
    assert rep.iters == orep.iters == 2 and np.array_equal(mv, omv)
    assert np.abs(R - Ro).max() <= 1e-8 * np.abs(Ro).max()
    np.testing.assert_allclose(mer, omer, rtol=1e-5)
