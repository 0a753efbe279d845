"""The fold of a step joined with the next step's first half (kReduceStep), and
the list decision by the last workgroup to arrive (decideLast).

Steps queued in one call are chained that way; a call of a single step ends
with the fold kernel and begins with the step-begin kernel. Both have to give
the same bits, at the sizes where the decision changes hands: one workgroup of
256 bodies, two, and 64 and more (a second level of arrival counters)."""
import dataclasses

import numpy as np
import pytest

from fundem_amd import workloads as W

pytestmark = pytest.mark.gpu


def run(scn, calls, graph, precision, lookahead=None):
    from fundem_amd import Solver
    g = Solver(precision=precision)
    g.use_graph(graph)
    if lookahead is not None:
        g.set_lookahead(lookahead)
    W.apply(scn, g)
    for n in calls:
        g.step(n)
    assert g.status() == 0
    out = (g.state(), [g.contacts(k) for k in range(5)], g.pair_totals())
    g.close()
    return out


def assert_same(a, b):
    for key in ("x", "v", "w", "q", "F", "T"):
        assert np.array_equal(a[0][key], b[0][key]), key
    for u, v in zip(a[1], b[1]):
        for key in ("A", "B", "k", "spring"):
            assert np.array_equal(u[key], v[key]), key


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("counts", [(1, 1, 1), (5, 3, 17), (16, 4, 4), (1, 1, 257), (32, 32, 16), (32, 32, 17)])
def test_chained_steps_equal_single_steps(counts, precision):
    scn = W.pour(counts, seed=7, dt=1e-6, templates=W.superellipsoid_family(2, 21, n_grid=12, n_nodes=60))
    scn.v[:, 2] = -0.05 - (scn.x[:, 2] - scn.x[:, 2].min()) / 1e-3
    scn.w[:] = np.random.default_rng(3).normal(0., 200., scn.w.shape)
    ref = run(scn, [1] * 90, False, precision, 0)
    print(f"{counts}: pairs {ref[2]}, contacts {[c['A'].size for c in ref[1]]}", flush=True)
    for graph in (False, True):
        assert_same(run(scn, [90], graph, precision), ref)
    assert_same(run(scn, [1, 2, 40, 3, 44], True, precision), ref)


def test_chained_periodic_and_bonded_steps_equal_single_steps():
    """Ghost visibility, wraps (a list build in the next step) and bond
    records in the fold."""
    for scn, steps in ((W.cluster(n=10, seed=5, speed=2.0, spin=50.0, spacing=2.4, periodic=(True, True)), 200),
                       (W.bonded_beam(counts=(12, 3, 3)), 60)):
        ref = run(scn, [1] * steps, False, "fp32", 0)
        assert_same(run(scn, [steps], True, "fp32"), ref)
        assert_same(run(scn, [steps // 2, steps - steps // 2], False, "fp32", 3), ref)


def test_a_system_that_is_no_number_leaves_the_others_their_lists():
    """A batch in which one system of several workgroups has lost its numbers
    (a run that blew up): the other system's lists are built again as it moves,
    and its states and contacts are those of the run alone."""
    from fundem_amd import Solver
    tm = W.superellipsoid_family(2, 5, n_grid=12, n_nodes=100)
    lost = W.cluster(n=700, seed=1, templates=tm, walls=False)
    lost = dataclasses.replace(lost, v=np.full_like(lost.v, np.nan))
    moving = W.cluster(n=64, seed=2, templates=tm, speed=0.2)
    moving = dataclasses.replace(moving, v=moving.v - (moving.x - moving.x.mean(0)) / 1e-3)
    alone = Solver()
    W.apply(moving, alone)
    both = Solver()
    W.apply_batch([lost, moving], both)
    seen = 0
    for i in range(8):
        alone.step(40)
        both.step(40)
        a, b = alone.state(), both.state()
        for key in ("x", "v", "w", "q", "F", "T"):
            assert np.array_equal(a[key], b[key][700:]), (i, key)
        u, v = alone.contacts(0), both.contacts(0)
        assert np.array_equal(u["A"], v["A"][v["A"] >= 700] - 700), i
        seen += u["A"].size
    assert seen > 0 and alone.list_builds()[0] > 1
    assert np.isnan(both.state()["x"][:700]).all()
