"""The dataflow schedule of a few hundred to a few thousand slices keeps near the
per-colour launches: its launch must not hold more wavefronts than the slices need,
each of which polls and adds to every sweep's counter.  On 41k rows with two lanes a
row it takes 60 us a sweep with one wavefront per CU, and 144 with six, against 58 by
colours; the bound lies between, at 1.6.  Also the same iterates, with several slices
per wavefront."""
import numpy as np
import pytest

import solfec
from scenes import lattice

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("lanes", [1, 2])
def test_flow_near_colour_launches(lanes, precision):
    s = lattice(27000, seed=3)
    b, c = s.bodies(), s.contacts()
    par = solfec.make_param(1e-14, 100, meritval=1e-14, diagepsilon=1e-8, precision=precision)
    dev = solfec.Device(0)
    ms, out = {}, {}
    try:
        dev.set_layout(lanes)
        dev.bodies(b["kind"], b["rot"], b["x0"], b["jinv"], b["minv"], b["velo"], b["velo0"])
        for _ in range(4):
            for sched in (0, 1):
                dev.set_schedule(sched)
                dev.contacts(c["master"], c["slave"], c["mpnt"], c["spnt"], c["base"], c["gap"], c["friction"],
                             c["restitution"], c["cohesion"], c["R"], c["U"])
                dev.assemble(1e-3)
                rep, _, _ = dev.solve(par, history=False)
                ms[sched] = min(ms.get(sched, np.inf), rep.solve_ms / rep.iters)
                out[sched] = (rep.iters, dev.get_RU())
    finally:
        dev.close()
    print(f"[flow] lanes {lanes} precision {precision}: us a sweep by colours {1e3 * ms[0]:.1f}, dataflow {1e3 * ms[1]:.1f}",
          flush=True)
    assert out[0][0] == out[1][0] == 100
    assert np.array_equal(out[0][1][0], out[1][1][0]) and np.array_equal(out[0][1][1], out[1][1][1])
    assert ms[1] <= 1.6 * ms[0]
