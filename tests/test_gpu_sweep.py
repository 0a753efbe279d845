"""The sweep of candidate pairs in runs (contact.hip, sweepRun): groups of 16
nodes and SDF cell codes cull, the exact predicate decides.

* sizes around the culls' units against the oracle, bit for bit: nodes per
  template (one, a group and its neighbours, a unit of sixteen groups and its
  neighbours, the largest count), SDF grids, both storage precisions, a curved
  (not affine) wall, and small particles on a finer grid than their partners';
* run lengths of one to eight pairs: a compressed lattice of thousands of
  pairs on a small sweep grid equals the kernel that culls by 64-node chunk
  (law mode 2), which shares none of the culls, in every bit."""
import dataclasses

import numpy as np
import pytest

import pyoracle as po
from fundem_amd import generators as gen
from fundem_amd import workloads as W
from test_gpu_parity import assert_contacts_equal, assert_states_equal

pytestmark = pytest.mark.gpu


def squeezed(n=8, seed=3, templates=None, **kw):
    """A cluster driven towards its centre, so that it collides at once."""
    scn = W.cluster(n=n, seed=seed, speed=0.2, spin=50.0, spacing=2.4, periodic=(True, True),
                    templates=templates, **kw)
    return dataclasses.replace(scn, v=scn.v - (scn.x - scn.x.mean(0)) / 1e-3)


def against_oracle(scn, steps, every, precision="fp32"):
    from fundem_amd import Solver
    g = Solver(precision=precision)
    W.apply(scn, g)
    o = po.OracleSim(precision == "fp32", True)
    W.apply(scn, o)
    seen = 0
    for i in range(every, steps + 1, every):
        g.step(every)
        o.step(every)
        assert_states_equal(g.state(), o.state(), f"step {i}")
        assert_contacts_equal(g, o, f"step {i}")
        seen += sum(o.contacts(s)["A"].size for s in (po.SET_PP, po.SET_PW, po.SET_GX, po.SET_GY))
    assert g.status() == 0
    g.close()
    return seen


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("nodes,grid", [(15, 16), (16, 7), (17, 16), (255, 16), (257, 24), (1000, 12)])
def test_node_and_grid_sizes_bitexact(nodes, grid, precision):
    tm = W.superellipsoid_family(2, 11, n_grid=grid, n_nodes=nodes, axes=(0.8e-3, 1.2e-3))
    assert against_oracle(squeezed(templates=tm), 320, 40, precision) > 0


def test_one_node_and_the_largest_count_bitexact():
    tm = W.superellipsoid_family(2, 12, n_grid=16, n_nodes=4096, axes=(0.8e-3, 1.2e-3))
    one = dataclasses.replace(tm[1], nodes=tm[1].nodes[:1], tris=None)
    assert against_oracle(squeezed(templates=[tm[0], one]), 240, 40) > 0


def test_fine_and_coarse_partners_bitexact():
    """A partner's spacing fifteen times smaller than the other's."""
    coarse = gen.superellipsoid_template(1.2e-3, 1.0e-3, 1.1e-3, 3.0, 5.0, n_grid=9, n_nodes=300)
    fine = gen.superellipsoid_template(4e-4, 3e-4, 4e-4, 2.5, 4.0, n_grid=40, n_nodes=200)
    scn = squeezed(n=12, templates=[coarse, fine])
    assert against_oracle(dataclasses.replace(scn, cell_size=0.0), 320, 40) > 0


def test_curved_wall_bitexact():
    """A sphere as a wall: its level set is not affine, so its pairs are
    culled by cell codes and without a bounding sphere."""
    scn = squeezed(n=8)
    ball = gen.sphere_template(1.5e-3, n_grid=20, n_nodes=200)
    c = scn.x.mean(0)
    scn = dataclasses.replace(
        scn, wall_templates=list(scn.wall_templates) + [ball], cell_size=0.0,
        walls=list(scn.walls) + [(c, np.zeros(3), np.zeros(3), W.IDENT, 0, len(scn.wall_templates))])
    assert against_oracle(scn, 320, 40) > 0


@pytest.mark.parametrize("counts", [(14, 14, 5), (20, 20, 8), (22, 22, 22)])
def test_run_lengths_equal_the_chunk_sweep(counts):
    from fundem_amd import Solver
    scn = W.pour(counts, seed=5, dt=1e-6, templates=W.superellipsoid_family(4, 21, n_nodes=300))
    scn.v[:, 2] = -(scn.x[:, 2] - scn.x[:, 2].min()) / 3e-3
    runs = []
    for shape in (dict(law_mode=2), dict(law_mode=1, sweep_waves_per_cu=4)):
        g = Solver()
        g.set_capacity(12, 64)
        g.set_launch_tuning(**shape)
        W.apply(scn, g)
        g.step(760)
        assert g.status() == 0
        runs.append((g.state(), [g.contacts(k) for k in range(5)], g.pair_totals()))
        g.close()
    (a, ca, pa), (b, cb, pb) = runs
    print(f"{counts}: candidate pairs {pb}, contacts {[c['A'].size for c in cb]}", flush=True)
    assert ca[0]["A"].size > 0
    for key in ("x", "v", "w", "q", "F", "T"):
        assert np.array_equal(a[key], b[key]), key
    for u, v in zip(ca, cb):
        for key in ("A", "B", "k", "spring"):
            assert np.array_equal(u[key], v[key]), key


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("n,nodes,steps", [(2, 1500, 60), (2, 4000, 60), (12, 900, 60), (40, 1500, 40)])
def test_contacts_of_a_run_around_one_wave_bitexact(n, nodes, steps, precision):
    """Blunt bodies pressed into each other and the floor: contacts of a run
    from a few (one per lane) to several batches of 64 staged in memory, pairs
    that cross a batch's edge, new and kept springs."""
    from fundem_amd import Solver
    tm = [gen.superellipsoid_template(1e-3, 0.9e-3, 1.1e-3, 8.0, 8.0, n_grid=16, n_nodes=nodes)]
    scn = squeezed(n=n, templates=tm, kn=20.0)
    scn = dataclasses.replace(scn, x=scn.x.mean(0) + 0.76 * (scn.x - scn.x.mean(0)), v=0.02 * scn.v)
    g = Solver(precision=precision)
    g.set_capacity(24, 400)
    W.apply(scn, g)
    o = po.OracleSim(precision == "fp32", True)
    W.apply(scn, o)
    most = []
    for i in range(1, steps + 1, 4):
        g.step(4)
        o.step(4)
        assert_states_equal(g.state(), o.state(), f"step {i}")
        assert_contacts_equal(g, o, f"step {i}")
        c = o.contacts(po.SET_PP)
        most.append(int(np.unique(np.stack([c["A"], c["B"]]), axis=1, return_counts=True)[1].max()) if c["A"].size else 0)
    print(f"{n} {nodes}: contacts of the fullest pair {min(most)}..{max(most)}", flush=True)
    assert g.status() == 0 and max(most) > 0
    g.close()
