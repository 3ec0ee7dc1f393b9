"""The packed slices of the sweep layout at their edges: rows without blocks,
rows of one to a few dozen blocks, a row longer than one round of the gather
(256 blocks in FP64, 384 in FP32), slices whose blocks end on and beside a slot
boundary, and a last slice of one row; 1 to 8 lanes per row, with and without
the merit's second product.  The system is an uploaded one with blocks small
against the diagonal, so that three sweeps stay within the rounding of the sums
(at most 700 products of relative error 1e-16 each, hence 1e-12) of the oracle."""
import numpy as np
import pytest

import oracle
import solfec

pytestmark = pytest.mark.gpu


def _system(n, hub, seed):
    rng = np.random.default_rng(seed)
    edges = set()
    for i in range(1, n):
        for j in rng.integers(1, n, rng.choice([0, 0, 1, 2, 4, 9])):
            if i != j:
                edges.add((min(i, j), max(i, j)))
    for j in rng.choice(np.arange(1, n), hub, replace=False):
        edges.add((0, int(j)))
    nb = [[] for _ in range(n)]
    for i, j in sorted(edges):
        w = 1e-5 * rng.normal(size=(3, 3))
        nb[i].append((j, w))
        nb[j].append((i, w.T))
    rowptr = np.concatenate([[0], np.cumsum([len(x) for x in nb])]).astype(np.int32)
    col = np.array([j for x in nb for j, _ in x], np.int32)
    W = np.concatenate([w.T.ravel() for x in nb for _, w in x]) if len(col) else np.zeros(0)
    Wd = np.zeros((n, 3, 3))
    for i in range(n):
        q = rng.normal(scale=1e-4, size=(3, 3))
        Wd[i] = np.diag([3.5e-3, 3.5e-3, 1e-3]) * (1 + 0.05 * len(nb[i])) + q @ q.T
    B = rng.normal(scale=1e-2, size=(n, 3))
    B[:, 2] -= 1e-2
    return dict(n=n, rowptr=rowptr, col=col, W=W, Wd=np.swapaxes(Wd, 1, 2).ravel().copy(),
                A=np.swapaxes(np.linalg.inv(Wd), 1, 2).ravel().copy(), B=B.ravel(), V=np.zeros(3 * n),
                rho=1.0 / np.linalg.eigvalsh(Wd)[:, -1], mu=np.full(n, 0.4), rest=np.zeros(n), coh=np.zeros(n),
                gap=np.full(n, -1e-6), free_energy=1.0, step=1e-3)


@pytest.mark.parametrize("lanes", [1, 2, 4, 8])
@pytest.mark.parametrize("n,hub", [(2, 1), (97, 40), (129, 0), (900, 257), (901, 700)])
def test_slices_match_oracle(lanes, n, hub):
    print(f"[slices] n={n} hub={hub} lanes={lanes}", flush=True)
    O = _system(n, hub, n + hub)
    rng = np.random.default_rng(5)
    R0 = np.abs(rng.normal(scale=3.0, size=(n, 3)))
    R0[:, :2] *= 0.1
    R0, U0 = R0.ravel(), rng.normal(scale=1e-3, size=3 * n)
    dev = solfec.Device(0)
    dev.set_layout(lanes)
    try:
        for kw in (dict(meritval=1.0), dict(meritval=1e-14), dict(meritval=1e-14, reverse=1),
                   dict(meritval=1e-14, precision=1, refine=1)):
            dev.system(O["rowptr"], O["col"], O["W"], O["Wd"], O["A"], O["B"], O["V"], O["rho"], O["mu"], O["rest"],
                       O["coh"], O["gap"], O["free_energy"], O["step"], R0, U0)
            L = dev.locdyn()
            assert np.array_equal(L["W"], O["W"]) and np.array_equal(L["Wd"], O["Wd"])
            rep, _, _ = dev.solve(solfec.make_param(1e-14, 3, diagepsilon=1e-10, diagmaxiter=100, **kw))
            R, U = dev.get_RU()
            order, _ = oracle.colour_order(L["colour"], int(L["colour"].max()) + 1)
            p = oracle.gs_param(1e-14, 3, meritval=kw["meritval"], reverse=kw.get("reverse", 0), diagepsilon=1e-10,
                                diagmaxiter=100)
            _, orep, Ro, Uo, _, _ = oracle.gs_solve(oracle.System(O), p, order, R0, U0)
            # MIXED: two sweeps in FP32 (6e-8 a product), one in FP64
            tol = 1e-12 if "precision" not in kw else 1e-4
            assert rep.iters == orep.iters
            assert np.abs(R.ravel() - Ro.ravel()).max() <= tol * np.abs(Ro).max(), kw
            assert np.abs(U.ravel() - Uo.ravel()).max() <= tol * max(np.abs(Uo).max(), 1e-2), kw
            # the standalone product (merit with the update of U) on the returned R
            dev.merit(1)
            U1 = dev.get_RU()[1]
            want = O["B"].reshape(n, 3) + np.einsum("nji,nj->ni", O["Wd"].reshape(n, 3, 3), R)
            rows = np.repeat(np.arange(n), np.diff(O["rowptr"]))
            np.add.at(want, rows, np.einsum("nji,nj->ni", O["W"].reshape(-1, 3, 3), R[O["col"]]))
            assert np.abs(U1 - want).max() <= 1e-12 * max(np.abs(want).max(), 1e-2)
    finally:
        dev.close()
