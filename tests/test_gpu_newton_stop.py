"""A body-space diagonal Newton loop that ends early does not form the body products
of the iterations that are enqueued past its end: one body with thousands of
contacts, so that a product (one thread adds the body's contacts) takes far longer
than a launch, and a loop whose merit ends it one iteration into a batch of 32.  Its
29 products take what 29 take under the iteration bound (which enqueues no more); 60,
the whole batch, would take twice that.  The bound lies between, at 1.5."""
import time

import numpy as np
import pytest

import solfec

pytestmark = pytest.mark.gpu


def _upload(dev, n):
    rng = np.random.default_rng(2)
    eye = np.eye(3).ravel()
    velo = np.array([0.0, 0.0, 0.0, 0.1, 0.05, -1.0])
    dev.bodies(np.zeros(1, np.int32), eye, np.zeros(3), eye / 0.4, np.ones(1), velo, velo)
    ang = rng.uniform(0.0, 2.0 * np.pi, n)
    pt = np.stack([0.3 * np.cos(ang), 0.3 * np.sin(ang), np.full(n, -0.5)], 1).ravel()
    z = np.zeros(n)
    dev.contacts(np.zeros(n, np.int32), np.full(n, -1, np.int32), pt, pt, np.tile(eye, n), z - 1e-6, z + 0.3, z, z,
                 np.zeros(3 * n), np.zeros(3 * n))
    dev.assemble(1e-3, diagonal_only=True)


def _run(dev, n, maxiter, meritval):
    _upload(dev, n)
    par = solfec.newton_param(linver="DIAG", maxiter=maxiter, meritval=meritval, theta=0.002 / n, gsflag="OFF")
    par.bodyspace = 1
    t = time.perf_counter()
    rep, mer, _ = dev.newton(par)
    t = time.perf_counter() - t
    return t, rep, mer, dev.get_RU()


def test_no_products_past_the_end():
    n, k = 4000, 29
    dev = solfec.Device(0)
    try:
        _, _, mer, _ = _run(dev, n, 200, 1e-300)
        assert np.isfinite(mer).all() and (np.diff(mer[:k + 1]) < 0.0).all()
        bound, early = [], []
        for _ in range(5):
            tb, rb, mb, (Rb, Ub) = _run(dev, n, k, 1e-300)
            te, re, me, (Re, Ue) = _run(dev, n, 200, mer[k - 1])
            assert rb.iters == re.iters == k and not rb.converged and re.converged
            assert np.array_equal(mb, me) and np.array_equal(Rb, Re) and np.array_equal(Ub, Ue)
            bound.append(tb)
            early.append(te)
    finally:
        dev.close()
    print(f"[newton] {k} body-space iterations: {1e3 * min(bound):.2f} ms by the bound, {1e3 * min(early):.2f} ms by the merit",
          flush=True)
    assert min(early) <= 1.5 * min(bound)
