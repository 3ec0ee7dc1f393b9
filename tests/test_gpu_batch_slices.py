"""Slices of half the rows serve the colour launches only: the persistent batch launch,
whose few wavefronts take all slices of a scene in turn, has 64 / lanes rows in every
slice but a colour's last.  With one wavefront per workgroup and a workgroup for every
row asked for, a scene gets as many workgroups as it has slices, which counts them.
Switching between the schedules moves the blocks and nothing else: the system stays the
same to the bit, and so do the solves, from the uploaded reactions or from those a solve
of the other schedule left, against contexts that never switched."""
import numpy as np
import pytest

import solfec
from solfec import batch
from scenes import lattice

pytestmark = pytest.mark.gpu

SIZES = (27, 1000, 343, 3375)


def _store():
    return batch.concat([(s.bodies(), s.contacts()) for s in (lattice(n, seed=k + 1) for k, n in enumerate(SIZES))])


def _system(dev):
    L = dev.locdyn()
    return {k: np.array(L[k]) for k in ("rowptr", "col", "W", "Wd", "B", "colour")}


@pytest.mark.parametrize("lanes", [1, 2])
def test_persistent_launch_has_full_slices(lanes):
    print(f"[batch slices] lanes={lanes}", flush=True)
    B, Cn, bs, cs = _store()
    dev = solfec.Device(0)
    dev.set_layout(lanes)
    try:
        ns = batch.upload(dev, B, Cn, bs, 1e-3)
        reps, _ = dev.batch_solve(solfec.make_param(1e-6, 3), ns, tune=(lanes, 1, 1, 0))
        cols = batch.split(dev.locdyn()["colour"], cs, 1)
    finally:
        dev.close()
    for k in range(ns):
        count = np.bincount(cols[k].ravel())
        assert reps["groups"][k] == int(np.sum(-(-count // (64 // lanes))))


@pytest.mark.parametrize("lanes", [1, 2])
def test_switching_schedules(lanes):
    print(f"[batch slices] switching, lanes={lanes}", flush=True)
    B, Cn, bs, cs = _store()
    fp64 = solfec.make_param(1e-14, 20, meritval=1e-14, diagepsilon=1e-10, diagmaxiter=100)
    mixed = solfec.make_param(1e-14, 20, meritval=1e-14, diagepsilon=1e-10, diagmaxiter=100, precision=1, refine=3)
    steps = [(fp64, 0), (fp64, 1), (mixed, 1), (fp64, 0), (mixed, 0), (fp64, 0)]
    a = solfec.Device(0)
    other = [solfec.Device(0), solfec.Device(0)]
    try:
        for d in (a, *other):
            d.set_layout(lanes)
        R, U = Cn["R"], Cn["U"]
        ns = batch.upload(a, B, Cn, bs, 1e-3)
        want = _system(a)
        for par, sched in steps:
            rep, _ = a.batch_solve(par, ns, tune=(lanes, 2, 256, sched))
            Ra, Ua = a.get_RU()
            L = _system(a)
            assert all(np.array_equal(L[k], want[k]) for k in want)
            # the same step in a context that has run solves of this layout only
            d = other[0 if sched == 0 and par is fp64 else 1]
            batch.upload(d, B, Cn, bs, 1e-3, R=R, U=U)
            repd, _ = d.batch_solve(par, ns, tune=(lanes, 2, 256, sched))
            Rd, Ud = d.get_RU()
            assert np.array_equal(rep["iters"], repd["iters"]) and np.array_equal(rep["merit"], repd["merit"])
            assert np.array_equal(Ra, Rd) and np.array_equal(Ua, Ud)
            R, U = Ra.ravel(), Ua.ravel()
    finally:
        for d in (a, *other):
            d.close()


def test_single_system_after_a_persistent_launch():
    s = lattice(1000, seed=2)
    b, c = s.bodies(), s.contacts()
    par = solfec.make_param(1e-14, 20, meritval=1e-14, diagepsilon=1e-10, diagmaxiter=100)
    out = []
    for first in (0, 1):
        dev = solfec.Device(0)
        try:
            dev.bodies(b["kind"], b["rot"], b["x0"], b["jinv"], b["minv"], b["velo"], b["velo0"])
            dev.contacts(c["master"], c["slave"], c["mpnt"], c["spnt"], c["base"], c["gap"], c["friction"],
                         c["restitution"], c["cohesion"], c["R"], c["U"])
            dev.assemble(1e-3)
            if first:
                dev.batch_solve(par, 1, tune=(2, 4, 1024, 0))
                dev.contacts(c["master"], c["slave"], c["mpnt"], c["spnt"], c["base"], c["gap"], c["friction"],
                             c["restitution"], c["cohesion"], c["R"], c["U"])
                dev.assemble(1e-3)
            rep, rer, mer = dev.solve(par)
            out.append((rep.iters, rer, mer, *dev.get_RU()))
        finally:
            dev.close()
    assert out[0][0] == out[1][0]
    assert all(np.array_equal(x, y) for x, y in zip(out[0][1:], out[1][1:]))
