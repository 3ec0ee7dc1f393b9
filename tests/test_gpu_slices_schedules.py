"""Slices whose blocks go round the gather several times, in the launches that hold a
whole solve or a whole batch.  The persistent schedules take a system with a row of
700 blocks, past the eight blocks a lane that the dataflow schedule waits for at once
(512 a slice), and follow the per-colour schedule to the bit, as they do on short rows
(alternating sweeps under the dataflow schedule are per-colour ones as well).
The batch takes scenes of bodies with 24 contacts each, 32 or 64 rows of 23 blocks in a
slice: its two schedules agree to the bit and follow the oracle's serial solve of every
scene.  There a local solve ends within 1e-10 of its solution and a row's coupling
|W_ii^-1 W_ij| is at most one a block, so that three sweeps of 24 colours stay within
1e-6 of the largest reaction."""
import numpy as np
import pytest

import oracle
import solfec
from solfec import batch
from test_gpu_slices import _system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [dict(meritval=1.0), dict(meritval=1e-14), dict(meritval=1e-14, reverse=1),
                                dict(meritval=1e-14, precision=1, refine=1)])
@pytest.mark.parametrize("lanes", [1, 2])
@pytest.mark.parametrize("sched", [1, 3])
def test_persistent_schedules_with_long_rows(sched, lanes, kw):
    n, hub = 901, 700
    print(f"[slices] schedule {sched} n={n} hub={hub} lanes={lanes} {kw}", flush=True)
    O = _system(n, hub, n + hub)
    assert np.diff(O["rowptr"]).max() > 512
    rng = np.random.default_rng(5)
    R0 = np.abs(rng.normal(scale=3.0, size=(n, 3)))
    R0[:, :2] *= 0.1
    R0, U0 = R0.ravel(), rng.normal(scale=1e-3, size=3 * n)
    dev = solfec.Device(0)
    dev.set_layout(lanes)
    out = []
    try:
        for sc in (0, sched):
            dev.set_schedule(sc)
            dev.system(O["rowptr"], O["col"], O["W"], O["Wd"], O["A"], O["B"], O["V"], O["rho"], O["mu"], O["rest"],
                       O["coh"], O["gap"], O["free_energy"], O["step"], R0, U0)
            rep, _, _ = dev.solve(solfec.make_param(1e-14, 6, diagepsilon=1e-10, diagmaxiter=100, **kw))
            out.append((rep, dev.get_RU()))
    finally:
        dev.close()
    (r0, (Ra, Ua)), (r1, (Rb, Ub)) = out
    assert r0.iters == r1.iters == 6 and r0.error == r1.error
    assert np.array_equal(Ra, Rb) and np.array_equal(Ua, Ub)


def _scene(nb, m, seed):
    """nb bodies apart from each other, each with m contacts of its own under it."""
    rng = np.random.default_rng(seed)
    eye = np.eye(3).ravel()
    velo = np.zeros((nb, 6))
    velo[:, 3:] = rng.normal(scale=0.05, size=(nb, 3)) + [0.0, 0.0, -1.0]
    x0 = rng.uniform(0.0, 10.0, (nb, 3))
    bodies = dict(kind=np.zeros(nb, np.int32), rot=np.tile(eye, nb), x0=x0.ravel(), jinv=np.tile(eye / 0.4, nb),
                  minv=np.ones(nb), velo=velo.ravel(), velo0=velo.ravel())
    n = nb*m
    master = np.repeat(np.arange(nb, dtype=np.int32), m)
    off = rng.uniform(-0.3, 0.3, (n, 3))
    off[:, 2] = -0.5
    pt = (x0[master] + off).ravel()
    z = np.zeros(n)
    R = np.abs(rng.normal(scale=3.0, size=(n, 3)))
    R[:, :2] *= 0.1
    contacts = dict(master=master, slave=np.full(n, -1, np.int32), mpnt=pt, spnt=pt, base=np.tile(eye, n), gap=z - 1e-6,
                    friction=z + 0.3, restitution=z, cohesion=z, R=R.ravel(), U=np.zeros(3*n))
    return bodies, contacts


@pytest.mark.parametrize("lanes", [1, 2])
@pytest.mark.parametrize("reverse", [0, 1])
def test_batch_slices_of_many_rounds(lanes, reverse):
    print(f"[slices] batch lanes={lanes} reverse={reverse}", flush=True)
    scenes = [_scene(70, 24, 1), _scene(3, 24, 2), _scene(129, 24, 3), _scene(1, 1, 4)]
    B, Cn, bs, cs = batch.concat(scenes)
    kw = dict(meritval=1e-14, diagepsilon=1e-10, diagmaxiter=100, reverse=reverse)
    dev = solfec.Device(0)
    dev.set_layout(lanes)
    out = []
    try:
        for sched in (0, 1):
            ns = batch.upload(dev, B, Cn, bs, 1e-3)
            reps, _ = dev.batch_solve(solfec.make_param(1e-14, 3, **kw), ns, tune=(lanes, 4, 0, sched))
            out.append((reps, dev.get_RU()))
        colours = dev.locdyn()["colour"]
    finally:
        dev.close()
    (r0, (Ra, Ua)), (r1, (Rb, Ub)) = out
    assert np.array_equal(r0["iters"], r1["iters"])
    assert np.array_equal(Ra, Rb) and np.array_equal(Ua, Ub)
    Rs, Us, Cols = batch.split(Ra, cs, 3), batch.split(Ua, cs, 3), batch.split(colours, cs, 1)
    for k, (b, c) in enumerate(scenes):
        O = oracle.assemble(oracle.bodies_from(b), oracle.contacts_from(c), 1e-3)
        col = Cols[k].ravel()
        order, _ = oracle.colour_order(col, int(col.max()) + 1)
        _, orep, Ro, Uo, _, _ = oracle.gs_solve(oracle.System(O), oracle.gs_param(1e-14, 3, **kw), order, c["R"], c["U"])
        assert int(r0["iters"][k]) == orep.iters
        assert np.abs(Rs[k] - Ro).max() <= 1e-6 * np.abs(Ro).max()
        assert np.abs(Us[k] - Uo).max() <= 1e-6 * max(np.abs(Uo).max(), 1e-2)
