"""The diagonal Newton loop, which tests itself on the device and is enqueued in
batches of 4, 8, 16, 32, 32, ... iterations: ends on, beside and far from a batch's
end by the iteration bound and by the merit, with and without the assembled
blocks.  The iterations do not depend on where the loop ends, so every history is
the start of the longest one and the state the one that many iterations leave, both
to the bit."""
import numpy as np
import pytest

import solfec
from scenes import lattice

pytestmark = pytest.mark.gpu

LONG = 150


@pytest.fixture(scope="module")
def dev():
    d = solfec.Device(0)
    yield d
    d.close()


def _run(dev, maxiter, meritval=1e-300, bodyspace=0):
    s = lattice(125, seed=4)
    b, c = s.bodies(), s.contacts()
    dev.bodies(b["kind"], b["rot"], b["x0"], b["jinv"], b["minv"], b["velo"], b["velo0"])
    dev.contacts(c["master"], c["slave"], c["mpnt"], c["spnt"], c["base"], c["gap"], c["friction"],
                 c["restitution"], c["cohesion"], c["R"], c["U"])
    dev.assemble(1e-3)
    par = solfec.newton_param(linver="DIAG", maxiter=maxiter, meritval=meritval, gsflag="OFF")
    par.bodyspace = bodyspace
    rep, mer, mv = dev.newton(par)
    R, U = dev.get_RU()
    return rep, mer, mv, R, U


@pytest.mark.parametrize("bodyspace", [0, 1])
def test_ends_of_batches(dev, bodyspace):
    print(f"[newton] batches bodyspace={bodyspace}", flush=True)
    rep, mer, mv, _, _ = _run(dev, LONG, bodyspace=bodyspace)
    assert rep.iters == LONG == len(mer) and not rep.converged and not mv.any()
    assert np.isfinite(mer).all() and rep.merit == mer[-1]
    for k in (1, 2, 3, 4, 5, 11, 12, 13, 28, 59, 60, 61, 64, 65, 123, 124, 125):
        one, m1, _, R1, U1 = _run(dev, k, bodyspace=bodyspace)
        assert one.iters == k and one.singular == 0 and one.merit == mer[k - 1]
        assert np.array_equal(m1, mer[:k])
        # the merit ends the loop at its first value not above the bound
        first = int(np.flatnonzero(mer <= mer[k - 1])[0]) + 1
        two, m2, _, R2, U2 = _run(dev, LONG, meritval=mer[k - 1], bodyspace=bodyspace)
        assert two.iters == first and two.converged == 1 and np.array_equal(m2, mer[:first])
        if first == k:
            assert np.array_equal(R1, R2) and np.array_equal(U1, U2)
