"""The in-place colouring of an assembled contact graph against the oracle's
greedy first-fit (exact): cliques, whose vertices depend on each other in one
chain, from one vertex over the eight neighbours taken together, a wavefront, one
word of the colour mask and the looks of one launch up to the last colour there
is, the first one past it, random graphs with contacts that share both bodies,
and a graph of many workgroups."""
import numpy as np
import pytest

import oracle
import solfec

pytestmark = pytest.mark.gpu


def _assemble(dev, nb, master, slave, kind=None):
    n = len(master)
    rng = np.random.default_rng(n)
    eye = np.tile(np.eye(3).ravel(), nb)
    x0 = rng.uniform(0.0, 1.0, (nb, 3))
    dev.bodies(np.zeros(nb, np.int32) if kind is None else kind, eye, x0.ravel(), 1e3 * eye, np.full(nb, 2.0),
               np.zeros(6 * nb), np.zeros(6 * nb))
    pt = (x0[master] + rng.normal(scale=0.05, size=(n, 3))).ravel()
    base = np.stack([np.linalg.qr(q)[0] for q in rng.normal(size=(n, 3, 3))]).ravel()
    z = np.zeros(n)
    dev.contacts(master, slave, pt, pt, base, z, z + 0.3, z, z, np.zeros(3 * n), np.zeros(3 * n))
    dev.assemble(1e-3)
    return dev.locdyn()


def _check(G):
    nc, want = oracle.colour(G["rowptr"], G["col"])
    assert np.array_equal(G["colour"], want)
    return nc


@pytest.fixture(scope="module")
def dev():
    d = solfec.Device(0)
    yield d
    d.close()


@pytest.mark.parametrize("n", [1, 2, 8, 9, 10, 64, 65, 66, 200, 256])
def test_clique(dev, n):
    print(f"[colour] clique {n}", flush=True)
    G = _assemble(dev, 2, np.zeros(n, np.int32), np.full(n, -1, np.int32))
    assert _check(G) == n


def test_clique_of_too_many_colours(dev):
    print("[colour] clique 257", flush=True)
    with pytest.raises(solfec.SfgsError):
        _assemble(dev, 2, np.zeros(257, np.int32), np.full(257, -1, np.int32))
    assert _check(_assemble(dev, 2, np.zeros(3, np.int32), np.full(3, -1, np.int32))) == 3


@pytest.mark.parametrize("n,nb", [(63, 5), (257, 300), (5000, 1200), (150001, 60000)])
def test_random_graph(dev, n, nb):
    print(f"[colour] random {n} contacts {nb} bodies", flush=True)
    rng = np.random.default_rng(n)
    kind = (rng.uniform(size=nb) < 0.05).astype(np.int32)   # obstacles couple nothing
    kind[0] = 0
    master = rng.integers(0, nb, n).astype(np.int32)
    master[kind[master] != 0] = 0 if n < 300 else 1 + np.flatnonzero(kind[1:] == 0)[0]
    hub = np.bincount(master, minlength=nb).argmax()
    # the bodies that took the obstacles' contacts keep few enough for 256 colours
    extra = np.flatnonzero(master == hub)[100:]
    free = np.flatnonzero(kind == 0)
    master[extra] = free[rng.integers(0, len(free), len(extra))]
    slave = rng.integers(-1, nb, n).astype(np.int32)
    slave[slave == master] = -1
    _check(_assemble(dev, nb, master, slave, kind))
