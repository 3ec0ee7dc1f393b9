"""The merit of states that are not finite: every contact's term is not a number,
infinite or finite where the reference's residual makes it so (mrf.c:35-184, which
forms 0.5 (|l| + l) of the two spectral values), and finite terms agree.  Rows are
decoupled and U is given (update_U = 0), so a bad reaction does not reach the
residual through U.  The finite terms are a few hundred FP64 operations apart at
most, 1e-16 each, on values of one sign: 1e-9 covers the cancellation in S - F."""
import numpy as np
import pytest

import oracle
import solfec

pytestmark = pytest.mark.gpu

NAN, INF = float("nan"), float("inf")


def _system(n, fri, coh):
    rng = np.random.default_rng(11)
    Wd = np.zeros((n, 3, 3))
    for i in range(n):
        q = rng.normal(scale=2e-4, size=(3, 3))
        Wd[i] = np.diag(np.array([3.5e-3, 3.5e-3, 1e-3]) * rng.uniform(0.5, 1.5, 3)) + q @ q.T
    return dict(n=n, rowptr=np.zeros(n + 1, np.int32), col=np.zeros(0, np.int32), W=np.zeros(0),
                Wd=np.swapaxes(Wd, 1, 2).ravel().copy(), A=np.swapaxes(np.linalg.inv(Wd), 1, 2).ravel().copy(),
                B=rng.normal(scale=1e-2, size=3 * n), V=np.zeros(3 * n), rho=1.0 / np.linalg.eigvalsh(Wd)[:, -1],
                mu=np.full(n, fri), rest=np.zeros(n), coh=np.full(n, coh), gap=np.full(n, -1e-6), free_energy=1.0,
                step=1e-3)


def _kind(v):
    return np.where(np.isnan(v), 2, np.where(np.isinf(v), 1, 0))


@pytest.mark.parametrize("fri,coh", [(0.3, 0.0), (0.0, 0.0), (0.6, 2.0)])
def test_merit_of_states_not_finite(fri, coh):
    # each special value alone in each of the six places, on rows that press, slide and
    # have no tangential part at all, and finite rows between them
    base = [((0.1, -0.2, 3.0), (1e-3, 2e-3, 0.0)), ((0.9, 0.3, 1.0), (-3e-3, 1e-3, -1e-4)),
            ((0.0, 0.0, 2.0), (0.0, 0.0, 1e-3)), ((0.0, 0.0, -1.0), (0.0, 0.0, 0.0))]
    R, U = [], []
    for r, u in base:
        R.append(r)
        U.append(u)
        for place in range(6):
            for v in (NAN, INF, -INF):
                rr, uu = list(r), list(u)
                (rr if place < 3 else uu)[place % 3] = v
                R.append(rr)
                U.append(uu)
    R, U = np.array(R).ravel(), np.array(U).ravel()
    n = len(R) // 3
    O = _system(n, fri, coh)
    print(f"[merit] states not finite: n={n} friction={fri} cohesion={coh}", flush=True)
    dev = solfec.Device(0)
    try:
        dev.system(O["rowptr"], O["col"], O["W"], O["Wd"], O["A"], O["B"], O["V"], O["rho"], O["mu"], O["rest"],
                   O["coh"], O["gap"], O["free_energy"], O["step"], R, U)
        m, cm = dev.merit(0, conmerit=True)
    finally:
        dev.close()
    mo, _, co = oracle.merit(oracle.System(O), R, U, 0)
    assert np.isnan(mo) and np.isnan(m)
    assert (_kind(co) == 2).sum() > n // 2 and (_kind(co) == 0).sum() >= len(base)
    wrong = np.flatnonzero(_kind(cm) != _kind(co))
    assert not len(wrong), [(R.reshape(-1, 3)[i].tolist(), U.reshape(-1, 3)[i].tolist(), cm[i], co[i]) for i in wrong[:8]]
    ok = _kind(co) == 0
    assert np.abs(cm[ok] - co[ok]).max() <= 1e-9 * np.abs(co[ok]).max()
