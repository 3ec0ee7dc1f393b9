"""The semismooth Newton solve of single rows against the oracle in every state
it distinguishes: open, sticking, sliding with and without the reaction against
the slip (alfa < 0), no friction, cohesion and a restitution shift, rows whose
3x3 system needs pivot exchanges, and iteration bounds on either side of the
rho schedule's start (10).  Rows are decoupled, one sweep is one local solve; it
stops at a relative change of 1e-10 after a quadratically convergent step, so
converged reactions agree to well within 1e-9 of the largest (1e-4 in the FP32
sweeps of a mixed solve, which stop at 1e-6 and round to 6e-8).  Bounded solves
compare the iterate itself: two differently rounded solvers are within 1e-9."""
import numpy as np
import pytest

import oracle
import solfec

pytestmark = pytest.mark.gpu


def _rows(kind, n, seed):
    rng = np.random.default_rng(seed)
    Wd = np.zeros((n, 3, 3))
    for i in range(n):
        q = np.linalg.qr(rng.normal(size=(3, 3)))[0] if kind == "pivot" else np.eye(3)
        d = np.array([3.5e-3, 3.5e-3, 1e-3]) if kind != "pivot" else 1e-3 * np.array([1.0, 0.2, 0.04])
        p = rng.normal(scale=2e-4, size=(3, 3))
        Wd[i] = q @ np.diag(d * rng.uniform(0.5, 1.5, 3)) @ q.T + 0.05 * (p @ p.T)
        Wd[i] = 0.5 * (Wd[i] + Wd[i].T)
    mu = rng.uniform(0.1, 0.8, n) if kind != "frictionless" else np.zeros(n)
    B = rng.normal(scale=1e-2, size=(n, 3))
    B[:, 2] = -np.abs(B[:, 2]) if kind != "open" else np.abs(B[:, 2])
    if kind == "stick":
        B[:, :2] *= 1e-2
    if kind in ("slide", "against"):
        B[:, :2] *= 5.0
    R0 = np.zeros((n, 3))
    R0[:, 2] = rng.uniform(0.5, 10.0, n)
    ang = np.arctan2(-B[:, 1], -B[:, 0]) + (np.pi if kind == "against" else 0.0)
    R0[:, 0], R0[:, 1] = 0.9 * mu * R0[:, 2] * np.cos(ang), 0.9 * mu * R0[:, 2] * np.sin(ang)
    U0 = B + np.einsum("nij,nj->ni", Wd, R0)
    coh = np.full(n, 2.0) if kind == "cohesion" else np.zeros(n)
    rest = np.full(n, 0.5) if kind == "restitution" else np.zeros(n)
    V = np.zeros((n, 3))
    V[:, 2] = -rng.uniform(0, 1e-2, n)
    return dict(n=n, rowptr=np.zeros(n + 1, np.int32), col=np.zeros(0, np.int32), W=np.zeros(0),
                Wd=np.swapaxes(Wd, 1, 2).ravel().copy(), A=np.swapaxes(np.linalg.inv(Wd), 1, 2).ravel().copy(),
                B=B.ravel(), V=V.ravel(), rho=1.0 / np.linalg.eigvalsh(Wd)[:, -1], mu=mu, rest=rest, coh=coh,
                gap=np.full(n, -1e-6), free_energy=1.0, step=1e-3), R0.ravel(), U0.ravel()


@pytest.mark.parametrize("kind", ["stick", "slide", "against", "open", "frictionless", "cohesion", "restitution", "pivot"])
@pytest.mark.parametrize("diagmax", [2, 9, 100])
def test_rows_match_oracle(kind, diagmax):
    print(f"[newton rows] {kind} diagmaxiter={diagmax}", flush=True)
    O, R0, U0 = _rows(kind, 190, 7)
    dev = solfec.Device(0)
    for precision in (0, 1) if diagmax == 100 else (0,):
        dev.system(O["rowptr"], O["col"], O["W"], O["Wd"], O["A"], O["B"], O["V"], O["rho"], O["mu"], O["rest"],
                   O["coh"], O["gap"], O["free_energy"], O["step"], R0, U0)
        # one sweep; failed rows (the bound reached) keep the iterate only without the fallback chain
        kw = dict(diagepsilon=1e-10, diagmaxiter=diagmax, failure=2 if diagmax < 100 else 0)
        dev.solve(solfec.make_param(1e-14, 2 if precision else 1, precision=precision, refine=0, **kw))
        R, U = dev.get_RU()
        _, _, Ro, Uo, _, _ = oracle.gs_solve(oracle.System(O), oracle.gs_param(1e-14, 2 if precision else 1, **kw),
                                             np.arange(O["n"], dtype=np.int32), R0, U0)
        tol = 1e-4 if precision else 1e-9
        assert np.abs(R.ravel() - Ro.ravel()).max() <= tol * max(np.abs(Ro).max(), 1.0)
        assert np.abs(U.ravel() - Uo.ravel()).max() <= tol * max(np.abs(Uo).max(), 1e-2)
    dev.close()
