"""Body state to the host in blocks of 8192 bodies through up to eight pinned
slots, one thread each (LSParticle::finalize): every body's values in its row,
for one block, its edges, two blocks, and more blocks than slots: as added, and
against the oracle's rows after steps in which nearly every body has a force
and a torque of its own."""
import dataclasses

import numpy as np
import pytest

import pyoracle as po
from fundem_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("n", [1, 2, 8191, 8192, 8193, 65536, 73729])
def test_every_value_in_its_place(n, precision):
    from fundem_amd import Solver
    scn = W.cluster(n=n, seed=3, templates=W.superellipsoid_family(2, 5, n_grid=8, n_nodes=20))
    c = scn.x.mean(0)
    scn = dataclasses.replace(scn, x=c + 0.65 * (scn.x - c))  # in contact with the neighbours
    real = np.float32 if precision == "fp32" else np.float64
    g = Solver(precision=precision)
    W.apply(scn, g)
    a = g.state()
    assert np.array_equal(a["x"], scn.x)
    for key in ("v", "w"):
        assert np.array_equal(a[key], getattr(scn, key).astype(real).astype(float)), key
    # (orientations are normalised first: a few roundings of components up to 1)
    assert np.abs(a["q"] - scn.q).max() <= 4 * np.finfo(real).eps
    g.step(3)
    o = po.OracleSim(precision == "fp32", True)
    W.apply(scn, o)
    o.step(3)
    b, want = g.state(), o.state()
    for key in b:
        assert np.array_equal(b[key], want[key]), key
    if n > 2:
        # rows that could not be told apart would not show a misplaced one
        for key in ("F", "T"):
            rows = np.unique(want[key][np.abs(want[key]).sum(1) > 0], axis=0)
            assert len(rows) > 0.95 * n, (key, len(rows))
        assert not np.array_equal(want["F"], want["T"])
    g.close()


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_state_before_initialize_is_the_bodies_as_added(precision):
    """The added bodies come back from the host (no step, nothing rounded to
    the storage precision yet); after initialize() the device's state does."""
    from fundem_amd import Solver

    class Unstarted(Exception):
        pass

    class Probe(Solver):
        def initialize(self, *a):
            raise Unstarted

    scn = W.cluster(n=30, seed=3, templates=W.superellipsoid_family(2, 5, n_grid=8, n_nodes=20))
    g = Probe(precision=precision)
    with pytest.raises(Unstarted):
        W.apply(scn, g)
    a = g.state()
    for key in ("x", "v", "w"):
        assert np.array_equal(a[key], getattr(scn, key)), key
    assert np.abs(a["q"] - scn.q).max() <= 4 * np.finfo(float).eps
    assert not a["F"].any() and not a["T"].any()
    g.close()
    empty = Solver(precision=precision)
    assert empty.state()["x"].shape == (0, 3)
    empty.close()


def test_reads_by_several_threads_and_of_several_sizes():
    """The pinned blocks of the reads are kept by the process and taken by
    whichever read comes: threads with solvers of one block, two and nine, each
    reading its own bodies again and again; then solvers created and closed."""
    import threading
    from fundem_amd import Solver
    tm = W.superellipsoid_family(2, 5, n_grid=8, n_nodes=20)
    scns = {n: W.cluster(n=n, seed=n, templates=tm) for n in (3, 9000, 73729, 500)}
    wrong = []

    def read(n, count):
        g = Solver()
        W.apply(scns[n], g)
        for _ in range(count):
            if not np.array_equal(g.state()["x"], scns[n].x):
                wrong.append(n)
        g.close()

    threads = [threading.Thread(target=read, args=(n, 12)) for n in scns]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for n in (9000, 3, 73729, 500, 3):
        read(n, 1)
    assert not wrong
